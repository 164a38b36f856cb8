"""GPU parity of the Gated DeltaNet kernels against the oracle (oracle/gdn.py): od_gdn_prep and od_gdn_norm_quant
bit-exact (every open-order sum is exact on both sides), od_gdn_recurrence against the float64 recurrence within
one bf16 step per output (plus 2e-3 relative in norm) and its fp32 final state within 1e-5 relative."""
import pytest
import torch

from oracle import gdn as og
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _bf(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16)


def _proj(g, M, n_k, n_v, dk, dv, pad=8):
    C = 2 * n_k * dk + n_v * dv
    P = C + n_v * dv + 2 * n_v
    pad += (-(P + pad)) % 8  # rows of 16-byte multiples, as the kernel requires
    p = _bf(g, M, P + pad)
    p[:, C + n_v * dv:] = _bf(g, M, 2 * n_v + pad, scale=3.0)  # b and a over a wider range
    return p


@pytest.mark.parametrize("S,L,n_k,n_v,with_state", [(2, 5, 2, 4, False), (3, 33, 2, 4, True), (4, 1, 2, 4, True),
                                                    (2, 2, 1, 2, True), (1, 70, 16, 32, False), (2, 24, 16, 32, True)])
def test_gdn_prep_bit_exact(gpu_lib, S, L, n_k, n_v, with_state):
    from opendecider_amd import kernels
    dk = dv = 128
    g = torch.Generator().manual_seed(S * 100 + L + n_k)
    C = 2 * n_k * dk + n_v * dv
    proj = _proj(g, S * L, n_k, n_v, dk, dv)
    conv_w = _bf(g, C, 4, scale=0.3)
    A_log = torch.log(torch.rand(n_v, generator=g) * 15.5 + 0.5).to(torch.bfloat16)
    dt = (1 + 0.1 * torch.randn(n_v, generator=g)).to(torch.bfloat16)
    n_states = 3
    conv_in = _bf(g, n_states, 3, C) if with_state else None
    seq = torch.randint(0, n_states, (S,), generator=g, dtype=torch.int32) if with_state else None
    if with_state and S > 1:
        seq[-1] = 7  # outside [0, n_states): reads zeros
    print(f"gdn_prep S={S} L={L} n_k={n_k} n_v={n_v} state={with_state}", flush=True)
    qk, v, gg, beta, co = kernels.gdn_prep(proj.to(DEV), conv_w.to(DEV), A_log.to(DEV), dt.to(DEV), S, L, n_k, n_v,
                                           dk, dv, None if conv_in is None else conv_in.to(DEV),
                                           None if seq is None else seq.to(DEV), conv_out=True)
    qkv_r, z_r, b_r, a_r = og.split_proj(proj[:, :C + n_v * dv + 2 * n_v], og.GDNConfig(n_k_heads=n_k, n_v_heads=n_v))
    cs = None
    if with_state:
        cs = torch.zeros(S, 3, C, dtype=torch.bfloat16)
        for i in range(S):
            if 0 <= int(seq[i]) < n_states:
                cs[i] = conv_in[int(seq[i])]
    y, new = og.conv_silu(qkv_r.reshape(S, L, C), conv_w, cs)
    y = y.reshape(S * L, C)
    kd = n_k * dk
    q_r = og.l2norm_bf16(y[:, :kd].reshape(-1, n_k, dk)).reshape(-1, kd)
    k_r = og.l2norm_bf16(y[:, kd:2 * kd].reshape(-1, n_k, dk)).reshape(-1, kd)
    g_r, beta_r = og.gates(a_r, b_r, A_log, dt)
    assert torch.equal(qk.cpu(), torch.cat([q_r, k_r], 1))
    assert torch.equal(v.cpu(), y[:, 2 * kd:])
    assert torch.equal(gg.cpu(), g_r) and torch.equal(beta.cpu(), beta_r)
    assert torch.equal(co.cpu(), new)


@pytest.mark.parametrize("S,L,n_k,n_v,dk,dv", [(2, 15, 2, 4, 16, 32), (1, 16, 1, 2, 64, 128), (2, 17, 1, 1, 256, 64),
                                               (1, 33, 1, 2, 512, 16), (1, 18, 1, 1, 1024, 16), (3, 32, 16, 32, 128, 128)])
def test_gdn_prep_tiles_and_special_values(gpu_lib, S, L, n_k, n_v, dk, dv):
    """od_gdn_prep at the edges of its 16-token tiles and over its head dims (2 to 64 lanes per head, 16 channels per
    thread at 1024), inputs of every magnitude (zero rows, 2^-130 .. 2^120, sums at bf16 midpoints, infinities, NaN):
    the oracle's bits, NaN for NaN."""
    from opendecider_amd import kernels
    g = torch.Generator().manual_seed(S * 100 + L + dk)
    C = 2 * n_k * dk + n_v * dv
    proj = _proj(g, S * L, n_k, n_v, dk, dv)
    conv_w = _bf(g, C, 4, scale=0.3)
    conv_w[::7] = 1.0                                             # exact sums: many ties
    proj[L // 3, :C] = 0
    scale = 2.0 ** torch.randint(-130, 121, (C,), generator=g).float()
    proj[L // 2, :C] = (proj[L // 2, :C].float() * scale).to(torch.bfloat16)
    proj[L - 1, 3] = float("inf")
    proj[L - 1, 5] = float("-inf")
    proj[L - 1, C - 2] = float("nan")
    A_log = torch.log(torch.rand(n_v, generator=g) * 15.5 + 0.5).to(torch.bfloat16)
    dt = (1 + 0.1 * torch.randn(n_v, generator=g)).to(torch.bfloat16)
    conv_in = _bf(g, S, 3, C)
    lens = torch.tensor([min(L, 16), L, 0][:S], dtype=torch.int32)
    print(f"gdn_prep special S={S} L={L} dk={dk} dv={dv}", flush=True)
    qk, v, _, _, co = kernels.gdn_prep(proj.to(DEV), conv_w.to(DEV), A_log.to(DEV), dt.to(DEV), S, L, n_k, n_v, dk, dv,
                                       conv_in.to(DEV), conv_out=True, seq_len=lens.to(DEV))
    cfg = og.GDNConfig(n_k_heads=n_k, n_v_heads=n_v, dk=dk, dv=dv)
    y, new = og.conv_silu(og.split_proj(proj[:, :C + n_v * dv + 2 * n_v], cfg)[0].reshape(S, L, C), conv_w, conv_in, lens)
    y = y.reshape(S * L, C)
    kd = n_k * dk
    want = torch.cat([og.l2norm_bf16(y[:, :kd].reshape(-1, n_k, dk)).reshape(-1, kd),
                      og.l2norm_bf16(y[:, kd:2 * kd].reshape(-1, n_k, dk)).reshape(-1, kd)], 1)
    for got, ref in ((qk.cpu(), want), (v.cpu(), y[:, 2 * kd:]), (co.cpu(), new)):  # (a NaN's payload is free)
        assert torch.equal(got.isnan(), ref.isnan())
        assert torch.equal(got.nan_to_num(nan=0.0).view(torch.int16), ref.nan_to_num(nan=0.0).view(torch.int16))


@pytest.mark.parametrize("S,L,n_k,n_v,lens", [(4, 11, 2, 4, [11, 6, 2, 0]), (3, 40, 16, 32, [40, 17, 1]),
                                               (2, 9, 2, 4, [3, 8])])
def test_gdn_prep_padded_sequences_bit_exact(gpu_lib, S, L, n_k, n_v, lens):
    """od_gdn_prep_ex with right-padded sequences (the reference's padded continuation): gates beta = 0, g = -0 at
    every pad (what b = a = -inf give), the conv window ending at each sequence's last real token (the state's own
    window for an empty one), everything at real positions as without padding; bit-exact against the oracle."""
    from opendecider_amd import kernels
    dk = dv = 128
    g = torch.Generator().manual_seed(S * 31 + L)
    C = 2 * n_k * dk + n_v * dv
    proj = _proj(g, S * L, n_k, n_v, dk, dv)
    conv_w = _bf(g, C, 4, scale=0.3)
    A_log = torch.log(torch.rand(n_v, generator=g) * 15.5 + 0.5).to(torch.bfloat16)
    dt = (1 + 0.1 * torch.randn(n_v, generator=g)).to(torch.bfloat16)
    conv_in = _bf(g, S, 3, C)
    seq_len = torch.tensor(lens, dtype=torch.int32)
    print(f"gdn_prep padded S={S} L={L} lens={lens}", flush=True)
    qk, v, gg, beta, co = kernels.gdn_prep(proj.to(DEV), conv_w.to(DEV), A_log.to(DEV), dt.to(DEV), S, L, n_k, n_v,
                                           dk, dv, conv_in.to(DEV), conv_out=True, seq_len=seq_len.to(DEV))
    cfg = og.GDNConfig(n_k_heads=n_k, n_v_heads=n_v)
    qkv_r, z_r, b_r, a_r = og.split_proj(proj[:, :C + n_v * dv + 2 * n_v], cfg)
    keep = (torch.arange(L)[None, :] < seq_len[:, None].long()).reshape(-1, 1)
    ninf = torch.full((), -float("inf"), dtype=torch.bfloat16)
    g_r, beta_r = og.gates(torch.where(keep, a_r, ninf), torch.where(keep, b_r, ninf), A_log, dt)
    y, new = og.conv_silu(qkv_r.reshape(S, L, C), conv_w, conv_in, lens)
    y = y.reshape(S * L, C)
    kd = n_k * dk
    real = keep[:, 0]
    q_r = og.l2norm_bf16(y[:, :kd].reshape(-1, n_k, dk)).reshape(-1, kd)
    k_r = og.l2norm_bf16(y[:, kd:2 * kd].reshape(-1, n_k, dk)).reshape(-1, kd)
    assert torch.equal(qk.cpu()[real], torch.cat([q_r, k_r], 1)[real])
    assert torch.equal(v.cpu()[real], y[real, 2 * kd:])
    assert torch.equal(gg.cpu().view(torch.int32), g_r.view(torch.int32))
    assert torch.equal(beta.cpu(), beta_r)
    assert (beta.cpu()[~real] == 0).all() and (gg.cpu()[~real] == 0).all()
    assert torch.equal(co.cpu(), new)


@pytest.mark.parametrize("L", [1, 2, 3, 4, 5])
def test_gdn_prep_short_sequences(gpu_lib, L):
    """Up to the 4 tokens that the short-sequence kernel takes and one more, with values of every magnitude, states with
    and without an entry, and 0 to L real tokens; heads of 1024 over several of its tiles."""
    test_gdn_prep_tiles_and_special_values(gpu_lib, 3, L, 2, 4, 128, 128)
    test_gdn_prep_tiles_and_special_values(gpu_lib, 2, L, 1, 2, 16, 16)
    test_gdn_prep_tiles_and_special_values(gpu_lib, 3, L + 6, 1, 1, 1024, 32)
    test_gdn_prep_bit_exact(gpu_lib, 5, L, 2, 4, True)
    test_gdn_prep_bit_exact(gpu_lib, 3, L, 16, 32, False)
    test_gdn_prep_padded_sequences_bit_exact(gpu_lib, L + 1, L, 2, 4, list(range(L + 1)))


@pytest.mark.parametrize("chunked", [True, False])
def test_gdn_padded_continuation_keeps_each_state(gpu_lib, chunked):
    """The recurrence over right-padded sequences (gates from od_gdn_prep_ex) leaves each sequence's final state equal
    to that of its unpadded pass at its real length, and a sequence with no real token its initial state bit for
    bit."""
    from opendecider_amd import kernels
    dk = dv = 128
    n_k, n_v, S, L = 2, 4, 3, 37
    lens = [37, 12, 0]
    g = torch.Generator().manual_seed(77)
    C = 2 * n_k * dk + n_v * dv
    proj = _proj(g, S * L, n_k, n_v, dk, dv).to(DEV)
    conv_w = _bf(g, C, 4, scale=0.3).to(DEV)
    A_log = torch.log(torch.rand(n_v, generator=g) * 15.5 + 0.5).to(torch.bfloat16).to(DEV)
    dt = (1 + 0.1 * torch.randn(n_v, generator=g)).to(torch.bfloat16).to(DEV)
    conv_in = _bf(g, S, 3, C).to(DEV)
    init = (torch.randn(S, n_v, dk, dv, generator=g) * 0.05).to(DEV)
    print(f"gdn padded continuation chunked={chunked}", flush=True)
    qk, v, gg, beta, _ = kernels.gdn_prep(proj, conv_w, A_log, dt, S, L, n_k, n_v, dk, dv, conv_in,
                                          seq_len=torch.tensor(lens, dtype=torch.int32, device=DEV))
    _, fin = kernels.gdn_recurrence(qk, v, gg, beta, S, L, n_k, n_v, dk, dv, init=init, final=True, chunked=chunked)
    assert torch.equal(fin[2], init[2])
    for s_, n in enumerate(lens[:2]):
        rows = slice(s_ * L, s_ * L + n)
        qk1, v1, g1, b1, _ = kernels.gdn_prep(proj[rows].contiguous(), conv_w, A_log, dt, 1, n, n_k, n_v, dk, dv,
                                              conv_in[s_:s_ + 1])
        _, fin1 = kernels.gdn_recurrence(qk1, v1, g1, b1, 1, n, n_k, n_v, dk, dv, init=init[s_:s_ + 1].contiguous(),
                                         final=True, chunked=chunked)
        d = (fin[s_] - fin1[0]).abs().max().item()
        assert d <= 1e-5 * fin1.abs().max().item() + 1e-7, (s_, d)


def _rec_inputs(g, S, L, n_k, n_v, dk=128, dv=128):
    M = S * L
    q = og.l2norm_bf16(_bf(g, M, n_k, dk))
    k = og.l2norm_bf16(_bf(g, M, n_k, dk))
    v = _bf(g, M, n_v, dv)
    a, b = _bf(g, M, n_v, scale=2.0), _bf(g, M, n_v, scale=2.0)
    A_log = torch.log(torch.rand(n_v, generator=g) * 15.5 + 0.5).to(torch.bfloat16)
    dt = (1 + 0.1 * torch.randn(n_v, generator=g)).to(torch.bfloat16)
    gg, beta = og.gates(a, b, A_log, dt)
    return q, k, v, gg, beta


@pytest.mark.parametrize("chunked", [True, False])
@pytest.mark.parametrize("S,L,n_k,n_v,init,gmul", [(2, 1, 2, 4, False, 1), (2, 16, 2, 4, True, 1),
                                                   (3, 70, 2, 4, True, 1), (1, 33, 16, 32, False, 1),
                                                   (4, 24, 16, 32, True, 1), (2, 300, 2, 4, True, 1),
                                                   (2, 64, 2, 4, True, 40), (2, 96, 2, 4, True, 0.01)])
def test_gdn_recurrence_matches_float64(gpu_lib, S, L, n_k, n_v, init, gmul, chunked):
    """Both forms (the chunked one on bf16 MFMA, and token by token) against the float64 recurrence; gmul scales the
    log-decays (x40: most of the state vanishes within a token; x0.01: almost no decay over the sequence)."""
    from opendecider_amd import kernels
    dk = dv = 128
    g = torch.Generator().manual_seed(S * 1000 + L + n_v)
    q, k, v, gg, beta = _rec_inputs(g, S, L, n_k, n_v)
    gg = gg * gmul
    n_states = 3
    st0 = torch.randn(n_states, n_v, dk, dv, generator=g) * 0.5 if init else None
    seq = torch.randint(0, n_states, (S,), generator=g, dtype=torch.int32) if init else None
    print(f"gdn_recurrence S={S} L={L} n_k={n_k} n_v={n_v} init={init} gmul={gmul} chunked={chunked}", flush=True)
    qk = torch.cat([q.reshape(S * L, -1), k.reshape(S * L, -1)], 1)
    o, fs = kernels.gdn_recurrence(qk.to(DEV), v.reshape(S * L, -1).to(DEV), gg.to(DEV), beta.to(DEV), S, L, n_k,
                                   n_v, dk, dv, None if st0 is None else st0.to(DEV),
                                   None if seq is None else seq.to(DEV), final=True, chunked=chunked)
    rep = n_v // n_k
    init_r = None if st0 is None else st0[seq.long()]
    o_r, st_r = og.recurrence(q.repeat_interleave(rep, 1).reshape(S, L, n_v, dk),
                              k.repeat_interleave(rep, 1).reshape(S, L, n_v, dk), v.reshape(S, L, n_v, dv),
                              gg.reshape(S, L, n_v), beta.reshape(S, L, n_v), init_r, torch.float64)
    o_r = o_r.reshape(S * L, n_v * dv).float()
    got = o.cpu().float()
    d = (got - o_r).abs()
    assert (d <= o_r.abs() * 2.0 ** -7 + 1e-6).all(), d.max().item()
    assert (d.norm() / o_r.norm()).item() <= 2e-3
    assert torch.allclose(fs.cpu(), st_r.float(), rtol=1e-5, atol=1e-5 * st_r.abs().max().item())


@pytest.mark.parametrize("S,L,n_k,n_v,dv,gmul", [(2, 33, 2, 4, 128, 1), (3, 64, 1, 2, 64, 1), (1, 65, 2, 2, 128, -5e-4),
                                                 (2, 128, 2, 6, 64, 1), (1, 161, 1, 8, 128, 1), (3, 193, 2, 4, 192, 1)])
def test_gdn_chunk_chain_edges(gpu_lib, S, L, n_k, n_v, dv, gmul):
    """The chunk chain at 2 to 7 chunks, whole and partial last ones, 1 to 3 column blocks per head, block counts that
    are and are not multiples of 8, growing gates (gmul < 0), started from shared states: the bars of
    test_gdn_recurrence_matches_float64. Those hold where the terms of an output are not much larger than the output:
    every product keeps 16 bits, so a growth of e^G over the sequence leaves 2^-16 e^G of the state in an output. The
    gates here sum to about -900 (2000 at the largest A), so gmul = -5e-4 keeps e^G under 3 (at -0.01 the state grows
    by e^9 to e^20 and outputs that cancel to its 2^-16 miss the one-step bar)."""
    from opendecider_amd import kernels
    g = torch.Generator().manual_seed(S * 1000 + L + dv)
    q, k, v, gg, beta = _rec_inputs(g, S, L, n_k, n_v, dv=dv)
    gg = gg * gmul
    st0 = torch.randn(2, n_v, 128, dv, generator=g) * 0.5
    seq = torch.randint(0, 2, (S,), generator=g, dtype=torch.int32)
    print(f"gdn chain S={S} L={L} n_k={n_k} n_v={n_v} dv={dv}", flush=True)
    qk = torch.cat([q.reshape(S * L, -1), k.reshape(S * L, -1)], 1)
    o, fs = kernels.gdn_recurrence(qk.to(DEV), v.reshape(S * L, -1).to(DEV), gg.to(DEV), beta.to(DEV), S, L, n_k, n_v,
                                   128, dv, st0.to(DEV), seq.to(DEV), final=True)
    rep = n_v // n_k
    o_r, st_r = og.recurrence(q.repeat_interleave(rep, 1).reshape(S, L, n_v, 128),
                              k.repeat_interleave(rep, 1).reshape(S, L, n_v, 128), v.reshape(S, L, n_v, dv),
                              gg.reshape(S, L, n_v), beta.reshape(S, L, n_v), st0[seq.long()], torch.float64)
    o_r = o_r.reshape(S * L, n_v * dv).float()
    d = (o.cpu().float() - o_r).abs()
    assert (d <= o_r.abs() * 2.0 ** -7 + 1e-6).all(), d.max().item()
    assert (d.norm() / o_r.norm()).item() <= 2e-3
    assert torch.allclose(fs.cpu(), st_r.float(), rtol=1e-5, atol=1e-5 * st_r.abs().max().item())


@pytest.mark.parametrize("S,L,final", [(16, 33, True), (16, 64, False), (17, 33, False), (17, 64, True)])
def test_gdn_two_chunks_over_many_sequences(gpu_lib, S, L, final):
    """Two chunks on both sides of the line between the two kernels that take them (four blocks of 64 columns
    per CU: 16 sequences of 32 heads of 128). The first, a middle and the last sequence against float64, with the bars of
    test_gdn_recurrence_matches_float64, but an absolute floor of 2^-16 of the largest output (a product keeps 16 bits
    of terms of that size, and among this many outputs some cancel); all of them against the token-by-token kernel, which
    may be as far off the other way."""
    from opendecider_amd import kernels
    n_k, n_v, dv = 16, 32, 128
    g = torch.Generator().manual_seed(S * 1000 + L)
    q, k, v, gg, beta = _rec_inputs(g, S, L, n_k, n_v, dv=dv)
    st0 = torch.randn(2, n_v, 128, dv, generator=g) * 0.5
    seq = torch.randint(0, 3, (S,), generator=g, dtype=torch.int32)  # 2: outside the states, zeros
    print(f"gdn two chunks S={S} L={L} final={final}", flush=True)
    qk = torch.cat([q.reshape(S * L, -1), k.reshape(S * L, -1)], 1)
    args = [x.to(DEV) for x in (qk, v.reshape(S * L, -1), gg, beta)]
    kw = dict(init=st0.to(DEV), seq_state=seq.to(DEV), final=final)
    o, fs = kernels.gdn_recurrence(*args, S, L, n_k, n_v, 128, dv, **kw)
    o1, fs1 = kernels.gdn_recurrence(*args, S, L, n_k, n_v, 128, dv, chunked=False, **kw)
    o, o1 = o.cpu().float(), o1.cpu().float()
    floor = 2.0 ** -16 * o1.abs().max().item()
    assert ((o - o1).abs() <= o1.abs() * 2.0 ** -6 * 1.01 + 2 * floor).all()
    rep, pick = n_v // n_k, [0, S // 2, S - 1]

    def rows(x, *shape):
        return x.reshape(S, L, *shape)[pick]

    init = torch.cat([st0, torch.zeros(1, n_v, 128, dv)])[seq.long()[pick]]
    o_r, st_r = og.recurrence(rows(q.repeat_interleave(rep, 1), n_v, 128), rows(k.repeat_interleave(rep, 1), n_v, 128),
                              rows(v, n_v, dv), rows(gg, n_v), rows(beta, n_v), init, torch.float64)
    o_r = o_r.reshape(len(pick), L, -1).float()
    d = (rows(o, n_v * dv) - o_r).abs()
    assert (d <= o_r.abs() * 2.0 ** -7 + floor).all(), d.max().item()
    assert (d.norm() / o_r.norm()).item() <= 2e-3
    assert final == (fs is not None)
    if final:
        assert torch.allclose(fs.cpu()[pick], st_r.float(), rtol=1e-5, atol=1e-5 * st_r.abs().max().item())
        assert torch.allclose(fs, fs1, rtol=2e-5, atol=2e-5 * fs1.abs().max().item())


@pytest.mark.parametrize("S,L,n_k,n_v,dv,states", [(1, 1, 2, 4, 128, 1), (3, 32, 1, 2, 128, 0), (200, 5, 2, 4, 128, 3),
                                                   (130, 31, 1, 8, 128, 2), (70, 9, 2, 4, 256, 3), (5, 24, 2, 4, 64, 2)])
def test_gdn_one_chunk_rows(gpu_lib, S, L, n_k, n_v, dv, states):
    """Sequences of at most 32 tokens that keep no final state (option rows): runs of one and several sequences per
    workgroup, a last run that is shorter, states in any order with one index outside the states (zeros), no states at
    all, two column blocks, and the other kernel's dv = 64: the bars of test_gdn_recurrence_matches_float64."""
    from opendecider_amd import kernels
    g = torch.Generator().manual_seed(S * 1000 + L + dv)
    q, k, v, gg, beta = _rec_inputs(g, S, L, n_k, n_v, dv=dv)
    st0 = torch.randn(states, n_v, 128, dv, generator=g) * 0.5 if states else None
    seq = torch.randint(0, states, (S,), generator=g, dtype=torch.int32) if states else None
    if states > 1:
        seq[S // 2] = states
    print(f"gdn rows S={S} L={L} n_v={n_v} dv={dv} states={states}", flush=True)
    qk = torch.cat([q.reshape(S * L, -1), k.reshape(S * L, -1)], 1)
    o, fs = kernels.gdn_recurrence(qk.to(DEV), v.reshape(S * L, -1).to(DEV), gg.to(DEV), beta.to(DEV), S, L, n_k, n_v,
                                   128, dv, None if st0 is None else st0.to(DEV), None if seq is None else seq.to(DEV))
    assert fs is None
    rep = n_v // n_k
    init = None
    if states:
        init = torch.cat([st0, torch.zeros(1, n_v, 128, dv)])[seq.long()]
    o_r, _ = og.recurrence(q.repeat_interleave(rep, 1).reshape(S, L, n_v, 128),
                           k.repeat_interleave(rep, 1).reshape(S, L, n_v, 128), v.reshape(S, L, n_v, dv),
                           gg.reshape(S, L, n_v), beta.reshape(S, L, n_v), init, torch.float64)
    o_r = o_r.reshape(S * L, n_v * dv).float()
    d = (o.cpu().float() - o_r).abs()
    assert (d <= o_r.abs() * 2.0 ** -7 + 1e-6).all(), d.max().item()
    assert (d.norm() / o_r.norm()).item() <= 2e-3


@pytest.mark.parametrize("S,L,n_k,n_v", [(9, 3, 16, 32), (15, 2, 16, 32), (4097, 1, 2, 4)])
def test_gdn_row_runs_are_one_round(gpu_lib, S, L, n_k, n_v):
    """Row counts that do not fill a round of one workgroup per CU: runs of two with a shorter last one, and more rows
    than a round of the longest runs takes (two rounds of equal runs)."""
    test_gdn_one_chunk_rows(gpu_lib, S, L, n_k, n_v, 128, 3)


@pytest.mark.parametrize("S,L,n_k,n_v", [(1, 1, 1, 1), (2, 15, 1, 2), (1, 16, 2, 6), (1, 17, 2, 4), (3, 31, 1, 3),
                                         (1, 32, 2, 4), (2, 33, 2, 2), (2, 48, 1, 2)])
@pytest.mark.parametrize("same_key", [False, True])
def test_gdn_chunk_t_matches_float64(gpu_lib, S, L, n_k, n_v, same_key):
    """T = (I + A)^{-1} diag(beta), as the chunk workspace holds it (bf16 hi + lo), against a float64 triangular solve:
    chunks that end in either 16-token block, one to three value heads per key head, and one key for all tokens with
    beta = 0.999. Bound: the split's 2^-16 |T|, 32u |X| |I + A| |T| of a forward substitution (u = 2^-24, X = (I + A)^{-1};
    the factor 4 covers the block form's three products), and |X| dA |T| with dA from the 128-term product of
    the keys, the 32-term sum of the gates and the exponential (4 ulp and 2u per unit of its argument)."""
    from opendecider_amd import kernels
    from opendecider_amd._lib import check, lib, ptr, stream_of
    g = torch.Generator().manual_seed(S * 1000 + L + n_v)
    q, k, v, gg, beta = _rec_inputs(g, S, L, n_k, n_v)
    if same_key:
        k = k.reshape(S * L, n_k, 128)[:1].expand(S * L, -1, -1).reshape(k.shape).contiguous()
        beta = torch.full_like(beta, 0.999)
        gg = gg * 0.01
    print(f"gdn T S={S} L={L} n_k={n_k} n_v={n_v} same_key={same_key}", flush=True)
    qk = torch.cat([q.reshape(S * L, -1), k.reshape(S * L, -1)], 1).to(DEV)
    o = torch.empty(S * L, n_v * 128, dtype=torch.bfloat16, device=DEV)
    ws = torch.zeros(kernels.gdn_chunk_workspace_floats(S, L, n_v), device=DEV)
    vd, gd, bd = v.reshape(S * L, -1).to(DEV), gg.to(DEV), beta.to(DEV)
    check(lib().od_gdn_recurrence_chunked(ptr(qk), ptr(vd), ptr(gd), ptr(bd), ptr(None), ptr(None), 0, S, L, n_k, n_v,
                                          128, 128, ptr(o), ptr(None), ptr(ws), ws.numel(), stream_of(qk)),
          "od_gdn_recurrence_chunked")
    nc, rep = (L + 31) // 32, n_v // n_k
    hl = ws.cpu()[:S * nc * n_v * 1136].reshape(S, nc, n_v, 1136)[..., :1024].contiguous().view(torch.bfloat16)
    hl = hl.reshape(S, nc, n_v, 2, 32, 32).double()

    def chunks(x, heads):  # [S L, heads, ...] -> [S, nc, heads, 32, ...]
        x = x.reshape(S, L, heads, -1).double()
        return torch.nn.functional.pad(x, (0, 0, 0, 0, 0, nc * 32 - L)).reshape(S, nc, 32, heads, -1).transpose(2, 3)
    kc = chunks(k, n_k).repeat_interleave(rep, 2)
    gc, bc = chunks(gg, n_v)[..., 0], chunks(beta, n_v)[..., 0]
    gam = gc.cumsum(-1)
    e = bc[..., :, None] * torch.exp(gam[..., :, None] - gam[..., None, :]).tril(-1)
    kk = kc @ kc.transpose(-1, -2)
    eye = torch.eye(32, dtype=torch.float64)
    IA = eye + (e * kk).tril(-1)
    T = torch.linalg.solve_triangular(IA, torch.diag_embed(bc), upper=False)
    X = torch.linalg.solve_triangular(IA, eye.expand_as(IA), upper=False)
    u = 2.0 ** -24
    n2 = kc.norm(dim=-1)
    span = gc.abs().sum(-1)[..., None, None]
    dA = e * (128 * u * n2[..., :, None] * n2[..., None, :] + kk.abs() * u * (10 + 66 * span))
    bound = 2.0 ** -16 * T.abs() + 4 * 32 * u * X.abs() @ IA.abs() @ T.abs() + X.abs() @ dA @ T.abs()
    err = (hl[..., 0, :, :] + hl[..., 1, :, :] - T).abs()
    assert (err <= bound + 1e-30).all(), (err - bound).max().item()


@pytest.mark.parametrize("chunked", [True, False])
def test_gdn_recurrence_in_place_state_and_continuation(gpu_lib, chunked):
    """Running L1 tokens, then L2 more continuing the written state in place, equals one run over L1 + L2 tokens up
    to rounding: the split moves the chunk boundaries (and the token-by-token form's scalar decay factor is
    multiplied into the state there), so the states agree to 1e-5 and the outputs to one bf16 step."""
    from opendecider_amd import kernels
    S, n_k, n_v, L1, L2 = 2, 2, 4, 45, 50
    g = torch.Generator().manual_seed(5)
    q, k, v, gg, beta = _rec_inputs(g, S, L1 + L2, n_k, n_v)

    def part(lo, hi):
        sel = lambda x: x.reshape(S, L1 + L2, *x.shape[1:])[:, lo:hi].reshape(S * (hi - lo), *x.shape[1:])
        qk = torch.cat([sel(q).reshape(S * (hi - lo), -1), sel(k).reshape(S * (hi - lo), -1)], 1)
        return qk.to(DEV), sel(v).reshape(S * (hi - lo), -1).to(DEV), sel(gg).to(DEV), sel(beta).to(DEV)

    whole, fs_whole = kernels.gdn_recurrence(*part(0, L1 + L2), S, L1 + L2, n_k, n_v, 128, 128, final=True,
                                             chunked=chunked)
    o1, st = kernels.gdn_recurrence(*part(0, L1), S, L1, n_k, n_v, 128, 128, final=True, chunked=chunked)
    o2, st2 = kernels.gdn_recurrence(*part(L1, L1 + L2), S, L2, n_k, n_v, 128, 128, init=st, final=st,
                                     chunked=chunked)
    assert st2.data_ptr() == st.data_ptr()
    both = torch.cat([o1.reshape(S, L1, -1), o2.reshape(S, L2, -1)], 1).reshape(S * (L1 + L2), -1).float()
    whole = whole.float()
    assert ((both - whole).abs() <= whole.abs() * 2.0 ** -7 + 1e-6).all()
    assert (both != whole).float().mean().item() < 0.01
    assert torch.allclose(st2, fs_whole, rtol=1e-5, atol=1e-5 * fs_whole.abs().max().item())


def test_gdn_norm_quant_every_gate_value(gpu_lib):
    """The gate z takes every finite bf16 value (the fast fp32 SiLU product and its float64 fallback both run) under
    random o and weights: bytes and scales equal the oracle's."""
    from opendecider_amd import kernels
    M, n_v, dv = 16, 32, 128
    g = torch.Generator().manual_seed(17)
    bits = torch.arange(65536, dtype=torch.int32).to(torch.int16)
    zv = bits.view(torch.bfloat16)
    zv = zv[torch.isfinite(zv.float())]
    z = torch.cat([zv, zv[: M * n_v * dv - zv.numel()]]).reshape(M, n_v * dv)
    o = _bf(g, M, n_v * dv, scale=0.3)
    w = (1 + 0.1 * torch.randn(dv, generator=g)).to(torch.bfloat16)
    inv = (1.0 / (torch.rand(n_v * dv, generator=g) * 1.5 + 0.5)).to(torch.bfloat16)
    for smooth in (None, inv):
        xq, sx = kernels.gdn_norm_quant(o.to(DEV), z.to(DEV), w.to(DEV), 1e-6, n_v, dv,
                                        None if smooth is None else smooth.to(DEV))
        y = og.gated_norm(o.reshape(M, n_v, dv), z.reshape(M, n_v, dv), w, 1e-6).reshape(M, n_v * dv)
        rq, rs = oq.act_quant(y, smooth)
        assert torch.equal(sx.cpu(), rs) and torch.equal(xq.cpu(), rq)


@pytest.mark.parametrize("M,n_v,smooth", [(5, 4, False), (33, 4, True), (64, 32, True), (3, 2, False),
                                          (512, 32, True)])
def test_gdn_norm_quant_bit_exact(gpu_lib, M, n_v, smooth):
    from opendecider_amd import kernels
    dv = 128
    g = torch.Generator().manual_seed(M + n_v)
    o = _bf(g, M, n_v * dv, scale=0.3)
    if M > 2:
        o[1] = 0                                               # a zero row: r = 1 / sqrt(eps)
    zz = _bf(g, M, n_v * dv + 40, scale=2.0)[:, 24:24 + n_v * dv]   # a strided column slice, as from proj
    w = (1 + 0.1 * torch.randn(dv, generator=g)).to(torch.bfloat16)
    inv = (1.0 / (torch.rand(n_v * dv, generator=g) * 1.5 + 0.5)).to(torch.bfloat16) if smooth else None
    print(f"gdn_norm_quant M={M} n_v={n_v} smooth={smooth}", flush=True)
    zd = zz.to(DEV)
    xq, sx = kernels.gdn_norm_quant(o.to(DEV), zd, w.to(DEV), 1e-6, n_v, dv, None if inv is None else inv.to(DEV))
    y = og.gated_norm(o.reshape(M, n_v, dv), zz.reshape(M, n_v, dv), w, 1e-6).reshape(M, n_v * dv)
    rq, rs = oq.act_quant(y, inv)
    assert torch.equal(sx.cpu(), rs) and torch.equal(xq.cpu(), rq)
