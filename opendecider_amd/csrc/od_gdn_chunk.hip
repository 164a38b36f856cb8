// Chunked gated delta rule on bf16 MFMA (gfx950), the fast form of od_gdn_recurrence's arithmetic.
//
// The recurrence of a value head (state S in R^{dk x dv}, token i: S_i = e^{g_i} S_{i-1} + k_i delta_i^T,
// delta_i = beta_i (v_i - (e^{g_i} S_{i-1})^T k_i), o_i = S_i^T q~_i with q~ = q / sqrt(dk); transformers'
// torch_recurrent_gated_delta_rule, which the reference runs for Qwen3.5's linear-attention layers) is unrolled over
// chunks of C = 32 tokens. With gamma_i = g_1 + ... + g_i inside the chunk and S_0 the state at its start:
//   A_ij = beta_i e^{gamma_i - gamma_j} (k_i . k_j)  (j < i),   T = (I + A)^{-1} diag(beta)
//   delta = T V - T diag(e^gamma) K S_0
//   O     = diag(e^gamma) Q~ S_0 + (Q~ K^T o D) delta,            D_ij = e^{gamma_i - gamma_j} (j <= i), else 0
//   S_C   = e^{gamma_C} S_0 + K^T diag(e^{gamma_C - gamma}) delta
// (the WY form of the chunked delta rule, as transformers' torch_chunk_gated_delta_rule evaluates it). Every
// exponent is of a non-positive number, so nothing overflows whatever the decay.
//
// gdn_chunk_t, per (sequence, chunk, key head): K K^T on MFMA and T in fp32, by forward substitution in two blocks,
// for each value head of that key head, written as bf16 hi / lo in the layout the second kernel copies straight into
// LDS, with the vectors gamma, e^gamma, e^{gamma_C - gamma} and e^{gamma_C}. Then, chunk after chunk (the only
// sequential part), one of three kernels with 16 state columns per wave (see the dispatch): gdn_chunk_roles<false>, a
// role per wave, per (sequence, value head, 64 columns); gdn_chunk_roles<true>, the same over one-chunk sequences that
// keep no state, per (run of sequences, value head, 128 columns); gdn_chunk_state, one or two chunks with every wave
// doing all of it, per (sequence, value head, 64 columns). gdn_chunk_state takes P from
// K Q~^T on MFMA, then the products above. The state lives in the MFMA accumulators
// (V_MFMA_F32_16X16X32_BF16, lane l: column l % 16, rows 4 (l / 16) + i of each 16 x 16 tile) and feeds the next
// products straight from there: an accumulator tile's rows become a B operand's k-values in the order
// (4h .. 4h+3, 16+4h .. 16+4h+3) for lane group h, and the A operand reads its k-index in the same order, so no
// transpose goes through LDS; T diag(e^gamma) X is taken as T (diag(e^gamma) X), the scaling on X's rows. Products
// whose operands are both exact in bf16 (K K^T, K Q^T) take one MFMA; an fp32 operand is split into bf16 hi + lo
// (16 significant bits; residual 2^-17 relative) and a product of two fp32 operands takes hi.hi + hi.lo + lo.hi, so
// every product carries ~16 bits against fp32's 24, accumulated in fp32.
#include "od_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kC = 32;                // tokens per chunk
constexpr int kDk = 128;
constexpr int kCols = 64;             // state columns per workgroup of gdn_chunk_state (16 per wave)
// workspace per (sequence, chunk, value head): T as two bf16 [32][32] matrices (hi, lo), then 112 floats: gamma [32],
// e^gamma [32], e^{gamma_C - gamma} [32], e^{gamma_C}, padding
constexpr int kMat = kC * kC;                      // bf16 per matrix
constexpr int kVecOff = 2 * kMat / 2;              // float offset of the vectors
constexpr int kVecN = 112;
constexpr int kTWs = kVecOff + kVecN;              // floats per block (4544 bytes, a multiple of 16)

__device__ __forceinline__ v4f mfma16(bf16x8 a, bf16x8 b, v4f c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ __bf16 bfr(float x) { return __builtin_bit_cast(__bf16, od_f32_to_bf16(x)); }
__device__ __forceinline__ float bff(__bf16 x) { return __uint_as_float((uint32_t)__builtin_bit_cast(uint16_t, x) << 16); }
// x = hi + lo + O(2^-17 |x|), hi and lo bf16
__device__ __forceinline__ void split(float x, __bf16& hi, __bf16& lo) {
  hi = bfr(x);
  lo = bfr(x - bff(hi));
}
// 8 bf16 of an LDS row in the permuted k-order of an accumulator used as a B operand: elements
// base + 4h .. base + 4h + 3, then base + 16 + 4h .. base + 16 + 4h + 3
__device__ __forceinline__ bf16x8 lds_perm(const uint16_t* row, int base, int h) {
  const uint2 a = *reinterpret_cast<const uint2*>(row + base + 4 * h);
  const uint2 b = *reinterpret_cast<const uint2*>(row + base + 16 + 4 * h);
  const uint4 w = make_uint4(a.x, a.y, b.x, b.y);
  return __builtin_bit_cast(bf16x8, w);
}
__device__ __forceinline__ bf16x8 lds8(const uint16_t* p) {
  return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(p));
}
// two fp32 values -> their bf16 hi and lo parts, each pair packed in one word (a in the low half)
__device__ __forceinline__ void split2(float a, float b, uint32_t& hi, uint32_t& lo) {
  hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((od_f32x2){a, b}, od_bf16x2));
  const float ra = a - __uint_as_float(hi << 16), rb = b - __uint_as_float(hi & 0xffff0000u);
  lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((od_f32x2){ra, rb}, od_bf16x2));
}
// the B operand, split, of accumulator tiles a (rows 0..15) and b (rows 16..31): values 4h .. 4h + 3 of a, then of b
__device__ __forceinline__ void acc_to_b(const v4f& a, const v4f& b, bf16x8& hi, bf16x8& lo) {
  uint32_t h[4], l[4];
  split2(a[0], a[1], h[0], l[0]);
  split2(a[2], a[3], h[1], l[1]);
  split2(b[0], b[1], h[2], l[2]);
  split2(b[2], b[3], h[3], l[3]);
  hi = __builtin_bit_cast(bf16x8, make_uint4(h[0], h[1], h[2], h[3]));
  lo = __builtin_bit_cast(bf16x8, make_uint4(l[0], l[1], l[2], l[3]));
}
// 8 bf16 in natural order from an 8-byte aligned row
__device__ __forceinline__ bf16x8 lds_nat(const uint16_t* p) {
  const uint2 a = *reinterpret_cast<const uint2*>(p);
  const uint2 b = *reinterpret_cast<const uint2*>(p + 4);
  return __builtin_bit_cast(bf16x8, make_uint4(a.x, a.y, b.x, b.y));
}
__device__ __forceinline__ uint16_t bf_bits(float x) { return od_f32_to_bf16(x); }

// ------------------------------------------------------------------------------------------------ gdn_chunk_t
struct TArgs {
  const uint16_t* qk;
  const float* g;
  const float* beta;
  float* ws;
  int64_t L, nchunk;
  int n_k, n_v;
};

// One wave per (sequence, chunk, key head), two of its value heads at a time. With I + A in 16 x 16 blocks
//   (I + A)^{-1} = [X11, 0; -X22 A21 X11, X22],   X11 = (I + A11)^{-1},   X22 = (I + A22)^{-1}
// the four diagonal blocks of the two heads are inverted at once, a lane per (block, column), and the corner takes two
// fp32 MFMA products. Bound by a wave's chain of LDS reads and fmas; the blocks make that 120 dependent fmas
// on 36 row reads in place of 496 on 140 (one substitution over the 32 rows): 52 -> 36 us at 4 x 4096 tokens, 16 / 32
// heads, 29 -> 17 us at 256 x 24.
constexpr int kTRow = 20;                   // floats per row of a 16 x 16 block
constexpr int kTBlk = 16 * kTRow + 16;      // and per block: the blocks of one read start 16 banks apart

__global__ __launch_bounds__(64) void gdn_chunk_t_kernel(TArgs p) {
  // per head the blocks (1,1), (2,1), (2,2): A by rows, then X, then T by columns
  __shared__ __attribute__((aligned(16))) float blk[2][3][kTBlk];
  __shared__ __attribute__((aligned(16))) float gam[2][kC], bet[2][kC], gsum[2][kC];
  const int64_t bid = blockIdx.x;
  const int hk = (int)(bid % p.n_k);
  const int64_t c = (bid / p.n_k) % p.nchunk;
  const int64_t s = bid / ((int64_t)p.n_k * p.nchunk);
  const int l = threadIdx.x, h4 = l >> 4, lc = l & 15;
  const int64_t t0 = c * kC, m0 = s * p.L;
  const int64_t kd = (int64_t)p.n_k * kDk;
  const int rep = p.n_v / p.n_k;

  // K K^T, tiles (0,0), (1,0), (1,1): both operands are rows (token 16 t + lc, dk 32 m + 8 h4 .. + 7)
  bf16x8 kf[2][4];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t tok = t0 + 16 * t + lc;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      uint4 wk = make_uint4(0, 0, 0, 0);
      if (tok < p.L) wk = *reinterpret_cast<const uint4*>(p.qk + (m0 + tok) * 2 * kd + kd + (int64_t)hk * kDk + 32 * m +
                                                          8 * h4);
      kf[t][m] = __builtin_bit_cast(bf16x8, wk);
    }
  }
  v4f kk[3] = {};
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    kk[0] = mfma16(kf[0][m], kf[0][m], kk[0]);
    kk[1] = mfma16(kf[1][m], kf[0][m], kk[1]);
    kk[2] = mfma16(kf[1][m], kf[1][m], kk[2]);
  }

  const int half = l >> 5, j = l & 31;
  for (int pp = 0; pp < rep; pp += 2) {
    const bool valid = pp + half < rep;
    const int hv = hk * rep + pp + half;
    const int64_t tok = t0 + j;
    float gj = 0.0f, bj = 0.0f;
    if (valid && tok < p.L) {
      gj = p.g[(m0 + tok) * p.n_v + hv];
      bj = p.beta[(m0 + tok) * p.n_v + hv];
    }
    gam[half][j] = gj;
    bet[half][j] = bj;
    __syncthreads();
    float cum = 0.0f;
#pragma unroll
    for (int u4 = 0; u4 < kC; u4 += 4) {
      const float4 gv = *reinterpret_cast<const float4*>(&gam[half][u4]);
      const float ge[4] = {gv.x, gv.y, gv.z, gv.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) cum += u4 + e <= j ? ge[e] : 0.0f;
    }
    gsum[half][j] = cum;
    __syncthreads();
    // A_ij = beta_i e^{gamma_i - gamma_j} kk_ij below the diagonal, from the accumulators: rows 4 h4 + r, column lc
    // (what a diagonal block holds on and above its diagonal is not read)
#pragma unroll
    for (int hd = 0; hd < 2; ++hd)
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const int ib = q ? 16 : 0, jb = q == 2 ? 16 : 0;
        const float4 gi = *reinterpret_cast<const float4*>(&gsum[hd][ib + 4 * h4]);
        const float4 bi = *reinterpret_cast<const float4*>(&bet[hd][ib + 4 * h4]);
        const float gc = gsum[hd][jb + lc];
        const float ga[4] = {gi.x, gi.y, gi.z, gi.w}, ba[4] = {bi.x, bi.y, bi.z, bi.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
          blk[hd][q][(4 * h4 + r) * kTRow + lc] = ba[r] * __expf(ga[r] - gc) * kk[q][r];
      }
    __syncthreads();
    // column lc of the diagonal block (head half, block h4 & 1): forward substitution
    float* const own = blk[half][2 * (h4 & 1)];
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float acc = i == lc ? 1.0f : 0.0f;
      const float4* row = reinterpret_cast<const float4*>(own + i * kTRow);
#pragma unroll
      for (int m4 = 0; m4 < (i + 3) / 4; ++m4) {
        const float4 a = row[m4];
        const float av[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (4 * m4 + e < i) acc = fmaf(-av[e], x[4 * m4 + e], acc);
      }
      x[i] = acc;
    }
    __syncthreads();  // every lane is done reading its block
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
      *reinterpret_cast<float4*>(own + lc * kTRow + 4 * i4) =
          make_float4(x[4 * i4], x[4 * i4 + 1], x[4 * i4 + 2], x[4 * i4 + 3]);
    __syncthreads();
    // the corner X21 = -X22 (A21 X11), k in the order 4 h4 + m: the first product's accumulator is the second's operand
    v4f x21[2];
#pragma unroll
    for (int hd = 0; hd < 2; ++hd) {
      const float4 a4 = *reinterpret_cast<const float4*>(&blk[hd][1][lc * kTRow + 4 * h4]);
      const float4 b4 = *reinterpret_cast<const float4*>(&blk[hd][0][lc * kTRow + 4 * h4]);
      const float av[4] = {a4.x, a4.y, a4.z, a4.w}, bv[4] = {b4.x, b4.y, b4.z, b4.w};
      v4f w = {0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < 4; ++m) w = __builtin_amdgcn_mfma_f32_16x16x4f32(av[m], bv[m], w, 0, 0, 0);
      v4f y = {0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < 4; ++m)
        y = __builtin_amdgcn_mfma_f32_16x16x4f32(blk[hd][2][(4 * h4 + m) * kTRow + lc], w[m], y, 0, 0, 0);
      x21[hd] = y;
    }
    __syncthreads();
    // T = (I + A)^{-1} diag(beta), by columns
    const float bc = bet[half][16 * (h4 & 1) + lc];
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
      *reinterpret_cast<float4*>(own + lc * kTRow + 4 * i4) =
          make_float4(x[4 * i4] * bc, x[4 * i4 + 1] * bc, x[4 * i4 + 2] * bc, x[4 * i4 + 3] * bc);
#pragma unroll
    for (int hd = 0; hd < 2; ++hd) {
      const float b0 = -bet[hd][lc];
      *reinterpret_cast<float4*>(&blk[hd][1][lc * kTRow + 4 * h4]) =
          make_float4(x21[hd][0] * b0, x21[hd][1] * b0, x21[hd][2] * b0, x21[hd][3] * b0);
    }
    __syncthreads();
    // rows of T as bf16 hi / lo: lane (row l / 4 of a half, columns 8 (l % 4) .. + 7), 1 KB per store
#pragma unroll
    for (int hd = 0; hd < 2; ++hd) {
      if (pp + hd >= rep) break;
      uint4* out = reinterpret_cast<uint4*>(p.ws + ((s * p.nchunk + c) * p.n_v + hk * rep + pp + hd) * (int64_t)kTWs);
#pragma unroll
      for (int ih = 0; ih < 2; ++ih) {
        const int i = l >> 2, u = l & 3;
        const float* col = &blk[hd][ih + (ih & (u >> 1))][8 * (u & 1) * kTRow + i];
        uint32_t th[4], tl[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) split2(col[2 * e * kTRow], col[(2 * e + 1) * kTRow], th[e], tl[e]);
        if (ih == 0 && u >= 2)
#pragma unroll
          for (int e = 0; e < 4; ++e) th[e] = tl[e] = 0;
        out[64 * ih + l] = make_uint4(th[0], th[1], th[2], th[3]);
        out[kMat / 8 + 64 * ih + l] = make_uint4(tl[0], tl[1], tl[2], tl[3]);
      }
    }
    if (valid) {
      const float glast = gsum[half][kC - 1];
      float* vec = p.ws + ((s * p.nchunk + c) * p.n_v + hv) * (int64_t)kTWs + kVecOff;
      vec[j] = cum;
      vec[kC + j] = __expf(cum);
      vec[2 * kC + j] = __expf(glast - cum);
      if (j == 0) vec[3 * kC] = __expf(glast);
    }
    __syncthreads();
  }
}

// ------------------------------------------------------------------------------------------------ gdn_chunk_state
struct CArgs {
  const uint16_t* qk;
  const uint16_t* v;
  const float* init;
  const int32_t* seq_state;
  const float* ws;
  uint16_t* o;
  float* final_state;
  int64_t L, nchunk, n_states;
  int n_k, n_v, dv;
  int64_t S;
  int run;  // gdn_chunk_roles<true>: sequences per workgroup
};

constexpr int kRowK = kDk + 8;    // K, Q rows (272 bytes: conflict-free 8-byte reads per half-wave)
constexpr int kRowT = kC + 4;     // K^T, V^T rows (72 bytes: conflict-free paired-token 4-byte writes)
constexpr int kRowM = kC + 8;     // the six matrices (80 bytes, 16-byte aligned rows)

struct CStage {
  uint16_t k[kC][kRowK];          // K (tokens x dk)
  uint16_t q[kC][kRowK];          // Q (tokens x dk)
  uint16_t kt[kDk][kRowT];        // K^T (dk x tokens)
  uint16_t vt[kCols][kRowT];      // V^T of the workgroup's 64 columns (columns x tokens)
  uint16_t m4[4][kC][kRowM];      // T hi, lo; P hi, lo
  float vec[kVecN];               // gamma [32], e^gamma [32], e^{gamma_C - gamma} [32], e^{gamma_C}
};

__device__ __forceinline__ uint32_t lo_pair(uint32_t a, uint32_t b) { return (a & 0xffffu) | (b << 16); }
__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }

__global__ __launch_bounds__(256) void gdn_chunk_state_kernel(CArgs p) {
  __shared__ __attribute__((aligned(16))) CStage st;
  __shared__ __attribute__((aligned(16))) uint16_t ob[kC][kCols + 8];
  const int nblk = p.dv / kCols;
  const int64_t bid = blockIdx.x;
  const int cb = (int)(bid % nblk);
  const int h = (int)((bid / nblk) % p.n_v);
  const int64_t s = bid / ((int64_t)nblk * p.n_v);
  const int hk = h / (p.n_v / p.n_k);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, h4 = lane >> 4, lc = lane & 15;
  const int64_t kd = (int64_t)p.n_k * kDk, ldv = (int64_t)p.n_v * p.dv;
  const int64_t m0 = s * p.L;
  const int col = cb * kCols + 16 * w + lc;  // this lane's state column
  const float qscale = (float)0.08838834764831845;  // fp32(1 / sqrt(128)), the reference's query scale

  // the state: tile r holds dk rows 16 r + 4 h4 + i of column `col`
  v4f S[8];
  const int64_t sidx = p.seq_state ? (int64_t)p.seq_state[s] : s;
  const bool has_init = p.init && sidx >= 0 && sidx < p.n_states;
#pragma unroll
  for (int r = 0; r < 8; ++r)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      S[r][i] = has_init ? p.init[((sidx * p.n_v + h) * kDk + 16 * r + 4 * h4 + i) * p.dv + col] : 0.0f;

  // chunk inputs, loaded into registers first. K and V: thread (tp, part) takes tokens 2 tp and
  // 2 tp + 1 of one 8-wide part, so that the transposed copies are written as token pairs
  const int tp = tid & 15, kp = tid >> 4, vp = (tid >> 4) & 7;
  struct Pre {
    uint4 k0, k1, q0, q1, v0, v1, w0, vec;
  };
  auto gload = [&](int64_t c) -> Pre {
    const int64_t t0 = c * kC;
    const uint4 z = make_uint4(0, 0, 0, 0);
    Pre r;
    {
      const int64_t ta = t0 + 2 * tp, tb = ta + 1;
      const uint16_t* src = p.qk + kd + (int64_t)hk * kDk + 8 * kp;
      r.k0 = ta < p.L ? *reinterpret_cast<const uint4*>(src + (m0 + ta) * 2 * kd) : z;
      r.k1 = tb < p.L ? *reinterpret_cast<const uint4*>(src + (m0 + tb) * 2 * kd) : z;
    }
    {
      const int64_t ta = t0 + (tid >> 4), tb = ta + 16;
      const uint16_t* src = p.qk + (int64_t)hk * kDk + 8 * (tid & 15);
      r.q0 = ta < p.L ? *reinterpret_cast<const uint4*>(src + (m0 + ta) * 2 * kd) : z;
      r.q1 = tb < p.L ? *reinterpret_cast<const uint4*>(src + (m0 + tb) * 2 * kd) : z;
    }
    {
      const int64_t ta = t0 + 2 * tp, tb = ta + 1;
      const uint16_t* src = p.v + (int64_t)h * p.dv + cb * kCols + 8 * vp;
      r.v0 = tid < 128 && ta < p.L ? *reinterpret_cast<const uint4*>(src + (m0 + ta) * ldv) : z;
      r.v1 = tid < 128 && tb < p.L ? *reinterpret_cast<const uint4*>(src + (m0 + tb) * ldv) : z;
    }
    const uint4* blk = reinterpret_cast<const uint4*>(p.ws + ((s * p.nchunk + c) * p.n_v + h) * (int64_t)kTWs);
    r.w0 = blk[tid];                                              // T hi, lo: 256 pieces
    r.vec = tid < kVecN / 4 ? blk[2 * kMat / 8 + tid] : z;        // the vectors: 28 pieces
    return r;
  };
  auto swrite = [&](const Pre& r) {
    *reinterpret_cast<uint4*>(&st.k[2 * tp][8 * kp]) = r.k0;
    *reinterpret_cast<uint4*>(&st.k[2 * tp + 1][8 * kp]) = r.k1;
    {
      const uint32_t a[4] = {r.k0.x, r.k0.y, r.k0.z, r.k0.w}, b[4] = {r.k1.x, r.k1.y, r.k1.z, r.k1.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        *reinterpret_cast<uint32_t*>(&st.kt[8 * kp + 2 * e][2 * tp]) = lo_pair(a[e], b[e]);
        *reinterpret_cast<uint32_t*>(&st.kt[8 * kp + 2 * e + 1][2 * tp]) = hi_pair(a[e], b[e]);
      }
    }
    *reinterpret_cast<uint4*>(&st.q[tid >> 4][8 * (tid & 15)]) = r.q0;
    *reinterpret_cast<uint4*>(&st.q[16 + (tid >> 4)][8 * (tid & 15)]) = r.q1;
    if (tid < 128) {
      const uint32_t a[4] = {r.v0.x, r.v0.y, r.v0.z, r.v0.w}, b[4] = {r.v1.x, r.v1.y, r.v1.z, r.v1.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        *reinterpret_cast<uint32_t*>(&st.vt[8 * vp + 2 * e][2 * tp]) = lo_pair(a[e], b[e]);
        *reinterpret_cast<uint32_t*>(&st.vt[8 * vp + 2 * e + 1][2 * tp]) = hi_pair(a[e], b[e]);
      }
    }
    *reinterpret_cast<uint4*>(&st.m4[tid >> 7][(tid & 127) >> 2][8 * (tid & 3)]) = r.w0;
    if (tid < kVecN / 4) *reinterpret_cast<uint4*>(&st.vec[4 * tid]) = r.vec;
  };

  // one chunk on the staged inputs: the outputs go to `ob`, the state advances
  const float* gam = st.vec;
  const float* eg = st.vec + kC;
  const float* ec = st.vec + 2 * kC;
  auto compute = [&]() {
    // P^T = K Q~^T o D^T on MFMA, tiles (key tile, query tile) = (0,0), (0,1), (1,1) on waves 0..2; lane: query i,
    // keys 4 h4 .. 4 h4 + 3 of the tile, written as P[i][j] hi / lo 8 bytes at a time. Wave 3 clears the upper tile.
    if (w < 3) {
      const int tj = w == 2 ? 1 : 0, ti = w == 0 ? 0 : 1;
      v4f a = {0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < 4; ++m)
        a = mfma16(lds8(&st.k[16 * tj + lc][32 * m + 8 * h4]), lds8(&st.q[16 * ti + lc][32 * m + 8 * h4]), a);
      const int i = 16 * ti + lc, j0 = 16 * tj + 4 * h4;
      float pv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        pv[r] = j0 + r <= i ? a[r] * qscale * __expf(gam[i] - gam[j0 + r]) : 0.0f;
      uint32_t h0, l0, h1, l1;
      split2(pv[0], pv[1], h0, l0);
      split2(pv[2], pv[3], h1, l1);
      *reinterpret_cast<uint2*>(&st.m4[2][i][j0]) = make_uint2(h0, h1);
      *reinterpret_cast<uint2*>(&st.m4[3][i][j0]) = make_uint2(l0, l1);
    } else {
      *reinterpret_cast<uint2*>(&st.m4[2][lc][16 + 4 * h4]) = make_uint2(0, 0);
      *reinterpret_cast<uint2*>(&st.m4[3][lc][16 + 4 * h4]) = make_uint2(0, 0);
    }
    __syncthreads();
    // X = K S_0 and Y = Q S_0 (tokens x this wave's 16 columns), S_0 split from the accumulators
    bf16x8 sh[4], sl[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) acc_to_b(S[2 * m], S[2 * m + 1], sh[m], sl[m]);
    v4f X[2], Y[2], U[2], D[2], O[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      X[t] = v4f{0, 0, 0, 0};
      Y[t] = v4f{0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const bf16x8 ak = lds_perm(&st.k[16 * t + lc][0], 32 * m, h4);
        const bf16x8 aq = lds_perm(&st.q[16 * t + lc][0], 32 * m, h4);
        X[t] = mfma16(ak, sh[m], X[t]);
        Y[t] = mfma16(aq, sh[m], Y[t]);
        X[t] = mfma16(ak, sl[m], X[t]);
        Y[t] = mfma16(aq, sl[m], Y[t]);
      }
    }
    // U = T V (natural token order)
    const bf16x8 bv = lds_nat(&st.vt[16 * w + lc][8 * h4]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      U[t] = mfma16(lds8(&st.m4[0][16 * t + lc][8 * h4]), bv, v4f{0, 0, 0, 0});
      U[t] = mfma16(lds8(&st.m4[1][16 * t + lc][8 * h4]), bv, U[t]);
    }
    // delta = U - T (diag(e^gamma) X)
    v4f x0, x1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      x0[e] = -eg[4 * h4 + e] * X[0][e];
      x1[e] = -eg[16 + 4 * h4 + e] * X[1][e];
    }
    bf16x8 xh, xl;
    acc_to_b(x0, x1, xh, xl);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const bf16x8 ath = lds_perm(&st.m4[0][16 * t + lc][0], 0, h4), atl = lds_perm(&st.m4[1][16 * t + lc][0], 0, h4);
      D[t] = mfma16(ath, xh, U[t]);
      D[t] = mfma16(ath, xl, D[t]);
      D[t] = mfma16(atl, xh, D[t]);
    }
    // O = diag(e^gamma / sqrt(dk)) Y + P delta
    bf16x8 dh, dl;
    acc_to_b(D[0], D[1], dh, dl);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int r = 0; r < 4; ++r) O[t][r] = eg[16 * t + 4 * h4 + r] * qscale * Y[t][r];
      const bf16x8 aph = lds_perm(&st.m4[2][16 * t + lc][0], 0, h4), apl = lds_perm(&st.m4[3][16 * t + lc][0], 0, h4);
      O[t] = mfma16(aph, dh, O[t]);
      O[t] = mfma16(aph, dl, O[t]);
      O[t] = mfma16(apl, dh, O[t]);
#pragma unroll
      for (int r = 0; r < 4; ++r) ob[16 * t + 4 * h4 + r][16 * w + lc] = bf_bits(O[t][r]);
    }
    // S = e^{gamma_C} S_0 + K^T diag(e^{gamma_C - gamma}) delta
    v4f d0, d1;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      d0[e] = ec[4 * h4 + e] * D[0][e];
      d1[e] = ec[16 + 4 * h4 + e] * D[1][e];
    }
    bf16x8 eh, el;
    acc_to_b(d0, d1, eh, el);
    const float elast = st.vec[3 * kC];
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      S[r] *= elast;
      const bf16x8 akt = lds_perm(&st.kt[16 * r + lc][0], 0, h4);
      S[r] = mfma16(akt, eh, S[r]);
      S[r] = mfma16(akt, el, S[r]);
    }
  };
  auto finish = [&](int64_t c) {
    __syncthreads();  // every wave is done with the stage and has written its outputs
    const int64_t tt = c * kC + (tid >> 3);
    if (tt < p.L)
      *reinterpret_cast<uint4*>(p.o + (m0 + tt) * ldv + (int64_t)h * p.dv + cb * kCols + 8 * (tid & 7)) =
          *reinterpret_cast<const uint4*>(&ob[tid >> 3][8 * (tid & 7)]);
  };

  // one or two chunks (see the dispatch), the second one's inputs loaded while the first is computed
  Pre pre = gload(0);
  swrite(pre);
  __syncthreads();
  if (p.nchunk > 1) pre = gload(1);
  compute();
  finish(0);
  if (p.nchunk > 1) {
    swrite(pre);
    __syncthreads();
    compute();
    finish(1);
  }
  if (p.final_state) {
#pragma unroll
    for (int r = 0; r < 8; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        p.final_state[((s * p.n_v + h) * kDk + 16 * r + 4 * h4 + i) * p.dv + col] = S[r][i];
  }
}


// ------------------------------------------------------------------------------------------------ gdn_chunk_roles
// The chunk chain of a (sequence, value head, 64 columns) with a role per wave, so that the sequential part is only
// the chunk's products:
//   chain waves 0..3    16 state columns each: U = T V, X = K S_0 and Y = Q S_0 from one split of S_0,
//                       delta = U - T (e^gamma X), the state update, O = e^gamma Y + P delta
//   staging waves 4..7  chunk c + 2 from registers to LDS and the loads of chunk c + 4, P of chunk c + 1, the output
//                       stores of chunk c - 1
// Each role is a loop of its own (the registers of one role are not live in the other) with one barrier per chunk
// over three stage buffers. Bound: the chain wave's own chunk, ~210 vector instructions, 64 MFMAs and ~45 LDS reads in
// sequence, about 2500 cycles, with the staging waves just below it (4 x 4096 tokens, 32 heads: 2900 cycles a chunk
// against 6500 with every wave doing all of it, 476 -> 175 us; one workgroup per CU, LDS 110 KB).
// Rows of K, Q, V, T and P are staged in the order row(j) = 16 ((j >> 2) & 1) + 4 (j >> 3) + (j & 3) and the state's dk
// rows alike within each 32, which makes accumulator tiles 0 and 1 of a lane group h hold tokens (dk) 8 h .. 8 h + 7 in
// order: every operand is then one 16-byte LDS read in natural order, K^T and V^T two transposing reads. Y and O are
// taken transposed (the state as the A operand), so a lane holds four neighbouring columns of a token and the outputs
// leave as 8-byte LDS writes.
// Row strides of 32 bytes past a multiple of 64: a fragment read (row lane % 16, 16 bytes at lane / 16) is then free
// of bank conflicts (ds_read_b128 serves lanes 0-3, 12-15, 20-27 together, and so on: strides of 80 and 272 bytes
// took two cycles for one, measured)
constexpr int kRowK2 = kDk + 16;
constexpr int kRowC = kC + 16;
constexpr int kChain = 4, kRowChain = 8;  // chain waves of a workgroup, 16 columns each
constexpr int kMaxRun = 64;               // sequences of a row workgroup (their state indices sit one per lane)

template <int NC>
struct RoleLds {
  static constexpr int kV = 16 * NC + (NC == 8 ? 16 : 8);  // row strides of V (conflict-free transposing reads) and O
  static constexpr int kO = 16 * NC + 4;
  struct Stage {
    uint16_t k[kC][kRowK2];
    uint16_t q[kC][kRowK2];
    uint16_t v[kC][kV];
    uint16_t tm[2][kC][kRowC];    // T hi, lo
    float vec[kVecN];
  } st[3];
  uint16_t pm[2][2][kC][kRowC];   // P hi, lo of two chunks
  uint16_t ob[2][kC][kO];         // outputs of two chunks
};

__device__ __forceinline__ int perm_row(int j) { return (j & ~31) + 16 * ((j >> 2) & 1) + 4 * ((j & 31) >> 3) + (j & 3); }
// A barrier over LDS only: __syncthreads would also wait for the chunk loads in flight and for the output stores
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef __amdgpu_buffer_rsrc_t rsrc_t;
// rows t0 .. of a [L, stride] bf16 matrix at `base` (its first row), at most one chunk of them: reads past the
// sequence give zeros and writes past it are dropped
__device__ __forceinline__ rsrc_t chunk_rsrc(const uint16_t* base, int64_t stride, int64_t t0, int64_t L) {
  const int64_t rows = t0 < 0 || t0 >= L ? 0 : L - t0 < kC ? L - t0 : kC;
  return __builtin_amdgcn_make_buffer_rsrc((void*)(base + t0 * stride), (short)0, (int)(rows * stride * 2), 0x00020000);
}
__device__ __forceinline__ uint4 bload(rsrc_t r, int off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}

// ROWS false: step c is chunk c of one sequence. ROWS true: one-chunk sequences that keep no final state (option rows),
// step c is sequence s0 + c of a run that shares the head; S_0 is read and split only where the state index changes,
// there is no update, and eight chain waves cover 128 columns.
template <bool ROWS>
__global__ __launch_bounds__(64 * (ROWS ? kRowChain + 4 : kChain + 4), ROWS ? 3 : 2) void gdn_chunk_roles_kernel(CArgs p) {
  constexpr int NC = ROWS ? kRowChain : kChain, COLS = 16 * NC;
  typedef RoleLds<NC> Lds;
  typedef typename Lds::Stage Stage;
  __shared__ __attribute__((aligned(16))) Lds sm;
  const int nblk = p.dv / COLS;
  // consecutive blocks of the (sequence or run, head, column block) order on one XCD: both column blocks and the value
  // heads of a key head read the same K and Q
  const unsigned nb = gridDim.x;
  const int64_t bid = nb % 8 == 0 ? (int64_t)(blockIdx.x % 8) * (nb / 8) + blockIdx.x / 8 : blockIdx.x;
  const int cb = (int)(bid % nblk);
  const int h = (int)((bid / nblk) % p.n_v);
  const int64_t s = bid / ((int64_t)nblk * p.n_v) * (ROWS ? p.run : 1);  // the (first) sequence
  const int hk = h / (p.n_v / p.n_k);
  const int lane = threadIdx.x & 63, h4 = lane >> 4, lc = lane & 15;
  const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int64_t kd = (int64_t)p.n_k * kDk, ldv = (int64_t)p.n_v * p.dv;
  const int n = ROWS ? (int)min((int64_t)p.run, p.S - s) : (int)p.nchunk;
  const int64_t m0 = s * p.L;
  const float qscale = (float)0.08838834764831845;  // fp32(1 / sqrt(128)), the reference's query scale
  const int otok = 8 * (lc >> 2) + (lc & 3);  // the token of row lc of tile 0 (of tile 1: + 4)

  if (w < NC) {
    // ---- chain: element i of state tile 2 m + u is dk row 32 m + 8 h4 + 4 u + i of column `col`
    const int col = cb * COLS + 16 * w + lc;
    v4f S[8];
    const int64_t row0 = 8 * h4;
    auto load_state = [&](int64_t sidx) {
#pragma unroll
      for (int r = 0; r < 8; ++r) S[r] = v4f{0, 0, 0, 0};
      if (p.init && sidx >= 0 && sidx < p.n_states) {
        const float* src = p.init + ((sidx * p.n_v + h) * kDk + row0) * p.dv + col;
#pragma unroll
        for (int r = 0; r < 8; ++r)
#pragma unroll
          for (int i = 0; i < 4; ++i) S[r][i] = src[(int64_t)(32 * (r >> 1) + 4 * (r & 1) + i) * p.dv];
      }
    };
    bf16x8 sh[4], sl[4];
    int states = 0, held = -1;  // ROWS: lane l holds the state index of sequence s + l (-1: none); the index in sh, sl
    if constexpr (ROWS) {
      if (lane < n) {
        const int64_t x = p.seq_state ? (int64_t)p.seq_state[s + lane] : s + lane;
        states = p.init && x >= 0 && x < p.n_states ? (int)x : -1;
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) sh[m] = sl[m] = __builtin_bit_cast(bf16x8, make_uint4(0, 0, 0, 0));
    } else {
      load_state(p.seq_state ? (int64_t)p.seq_state[s] : s);
    }
    bf16x8 th[2], tl[2], bv, kf[4][2], qf[4][2];
    // K^T and V^T operands through transposing reads of the row-major stage: lane 4 e + c of a 16-lane group points at
    // the 8-byte piece c of row e (token 8 h4 + e; the second read: + 4, 16 staged rows on) and lane j receives column
    // j % 4 of piece j / 4 in the four rows
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    typedef __attribute__((address_space(3))) const char lds_char;
    auto tr8 = [&](const void* at, int next) {
      lds_char* src = (lds_char*)at;
      const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)src);
      const s4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(src + next));
      return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
    };
    const int trow = 4 * h4 + (lc >> 2);
    auto frags_kq = [&](const Stage& st) {
      bv = tr8(&st.v[trow][16 * w + 4 * (lc & 3)], 16 * 2 * Lds::kV);  // 16 contiguous columns
#pragma unroll
      for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          kf[m][t] = lds8(&st.k[16 * t + lc][32 * m + 8 * h4]);
          qf[m][t] = lds8(&st.q[16 * t + lc][32 * m + 8 * h4]);
        }
    };
    auto frags_t = [&](const Stage& st) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        th[t] = lds8(&st.tm[0][16 * t + lc][8 * h4]);
        tl[t] = lds8(&st.tm[1][16 * t + lc][8 * h4]);
      }
    };
    lds_barrier();
    if constexpr (!ROWS) {
      frags_kq(sm.st[0]);
      frags_t(sm.st[0]);
    }
    lds_barrier();
    int cur = 0;
    for (int c = 0; c < n; ++c) {
      const Stage& st = sm.st[cur];
      cur = cur == 2 ? 0 : cur + 1;
      const Stage& sn = sm.st[cur];  // chunk c + 1, whole since the last barrier (past the end: stale, unused)
      if constexpr (ROWS) {  // two chain waves per SIMD hide each other's reads: no operands held across a barrier
        frags_kq(st);
        frags_t(st);
        const int want = __builtin_amdgcn_readlane(states, c);
        if (want != held) {
          held = want;
          load_state(want);
#pragma unroll
          for (int m = 0; m < 4; ++m) acc_to_b(S[2 * m], S[2 * m + 1], sh[m], sl[m]);
        }
      }
      const float elast = st.vec[3 * kC];
      const float4 e0 = *reinterpret_cast<const float4*>(&st.vec[kC + 8 * h4]);
      const float4 e1 = *reinterpret_cast<const float4*>(&st.vec[kC + 8 * h4 + 4]);
      const float4 c0 = *reinterpret_cast<const float4*>(&st.vec[2 * kC + 8 * h4]);
      const float4 c1 = *reinterpret_cast<const float4*>(&st.vec[2 * kC + 8 * h4 + 4]);
      const float eq[2] = {st.vec[kC + otok] * qscale, st.vec[kC + otok + 4] * qscale};
      v4f X[2], Y[2], D[2];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        X[t] = v4f{0, 0, 0, 0};
        Y[t] = v4f{0, 0, 0, 0};
        D[t] = mfma16(th[t], bv, v4f{0, 0, 0, 0});  // U = T V
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) D[t] = mfma16(tl[t], bv, D[t]);
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        bf16x8 ah, al;
        if constexpr (ROWS) {
          ah = sh[m];
          al = sl[m];
        } else {
          acc_to_b(S[2 * m], S[2 * m + 1], ah, al);
        }
        X[0] = mfma16(kf[m][0], ah, X[0]);
        X[1] = mfma16(kf[m][1], ah, X[1]);
        Y[0] = mfma16(ah, qf[m][0], Y[0]);
        Y[1] = mfma16(ah, qf[m][1], Y[1]);
        X[0] = mfma16(kf[m][0], al, X[0]);
        X[1] = mfma16(kf[m][1], al, X[1]);
        Y[0] = mfma16(al, qf[m][0], Y[0]);
        Y[1] = mfma16(al, qf[m][1], Y[1]);
        if constexpr (!ROWS) {
          S[2 * m] *= elast;
          S[2 * m + 1] *= elast;
        }
      }
      bf16x8 kt[8], ph[2], pl[2];
#pragma unroll
      for (int r = 0; r < (ROWS ? 0 : 8); ++r)
        kt[r] = tr8(&st.k[trow][32 * (r >> 1) + 8 * (lc & 3) + 4 * (r & 1)], 16 * 2 * kRowK2);
      // delta = U - T (diag(e^gamma) X)
      bf16x8 xh, xl;
      acc_to_b(v4f{-e0.x, -e0.y, -e0.z, -e0.w} * X[0], v4f{-e1.x, -e1.y, -e1.z, -e1.w} * X[1], xh, xl);
      D[0] = mfma16(th[0], xh, D[0]);
      D[1] = mfma16(th[1], xh, D[1]);
      D[0] = mfma16(th[0], xl, D[0]);
      D[1] = mfma16(th[1], xl, D[1]);
      D[0] = mfma16(tl[0], xh, D[0]);
      D[1] = mfma16(tl[1], xh, D[1]);
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        ph[t] = lds8(&sm.pm[c & 1][0][16 * t + lc][8 * h4]);
        pl[t] = lds8(&sm.pm[c & 1][1][16 * t + lc][8 * h4]);
      }
      bf16x8 eh, el, dh, dl;
      if constexpr (!ROWS) {
        frags_kq(sn);
        frags_t(sn);
        // S = e^{gamma_C} S_0 + K^T diag(e^{gamma_C - gamma}) delta
        acc_to_b(v4f{c0.x, c0.y, c0.z, c0.w} * D[0], v4f{c1.x, c1.y, c1.z, c1.w} * D[1], eh, el);
#pragma unroll
        for (int r = 0; r < 8; ++r) S[r] = mfma16(kt[r], eh, S[r]);
#pragma unroll
        for (int r = 0; r < 8; ++r) S[r] = mfma16(kt[r], el, S[r]);
      }
      // O^T = Y^T diag(e^gamma / sqrt(dk)) + delta^T P^T
      acc_to_b(D[0], D[1], dh, dl);
      v4f O[2] = {Y[0] * eq[0], Y[1] * eq[1]};
#pragma unroll
      for (int t = 0; t < 2; ++t) O[t] = mfma16(dh, ph[t], O[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t) O[t] = mfma16(dl, ph[t], O[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t) O[t] = mfma16(dh, pl[t], O[t]);
#pragma unroll
      for (int t = 0; t < 2; ++t)
        *reinterpret_cast<uint2*>(&sm.ob[c & 1][16 * t + lc][16 * w + 4 * h4]) =
            make_uint2(od_pack_bf16x2(O[t][0], O[t][1]), od_pack_bf16x2(O[t][2], O[t][3]));
      lds_barrier();
    }
    if (!ROWS && p.final_state) {
      float* dst = p.final_state + ((s * p.n_v + h) * kDk + row0) * p.dv + col;
#pragma unroll
      for (int r = 0; r < 8; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) dst[(int64_t)(32 * (r >> 1) + 4 * (r & 1) + i) * p.dv] = S[r][i];
    }
  } else {
    // ---- staging: rows of K, Q and V (16 lanes of 16 bytes, or 8, per row), T and the vectors through registers, two
    // sets: a chunk is loaded two steps before it is written to LDS
    const uint16_t* qk0 = p.qk + m0 * 2 * kd + (int64_t)hk * kDk;
    const int tid = threadIdx.x - 64 * NC, ws = w - NC;  // thread and wave of the four
    const uint16_t* v0 = p.v + m0 * ldv + (int64_t)h * p.dv + cb * COLS;
    uint16_t* o0 = p.o + m0 * ldv + (int64_t)h * p.dv + cb * COLS;
    const uint4* tw0 = reinterpret_cast<const uint4*>(p.ws + (s * p.nchunk * p.n_v + h) * (int64_t)kTWs);
    const int tj = ((tid >> 3) & 1) | ((tid >> 2) & 1) << 1 | ((tid >> 4) & 7) << 2, tq = tid & 3;  // row, part of T
    const int rb = (int)(4 * kd), qo = (tid >> 4) * rb + 16 * (tid & 15), ko = qo + (int)(2 * kd);
    constexpr int kParts = COLS / 8, kVRows = 256 / kParts;  // 16-byte parts of a V or O row, rows per pass of 256 threads
    const int vr = tid / kParts, vp = tid % kParts, vo = vr * (int)(2 * ldv) + 16 * vp;
    // step c: chunk c of the sequence, or the one chunk of sequence s + c
    auto rows_of = [&](const uint16_t* base, int64_t stride, int c) {
      if constexpr (ROWS) return chunk_rsrc(base + (int64_t)c * p.L * stride, stride, c >= 0 && c < n ? 0 : -1, p.L);
      return chunk_rsrc(base, stride, (int64_t)c * kC, p.L);
    };
    // Every load is unconditional (chunks past the end: no rows, the last T block again), so that the compiler knows
    // how many are in flight and each use waits for its own loads only
    struct Pre {
      uint4 k0, k1, q0, q1, v0, v1, w0, vec;
    };
    auto gload = [&](int c, Pre& r) {
      const rsrc_t rq = rows_of(qk0, 2 * kd, c), rv = rows_of(v0, ldv, c);
      r.k0 = bload(rq, ko);
      r.k1 = bload(rq, ko + 16 * rb);
      r.q0 = bload(rq, qo);
      r.q1 = bload(rq, qo + 16 * rb);
      r.v0 = bload(rv, vo);
      r.v1 = ROWS ? bload(rv, vo + kVRows * (int)(2 * ldv)) : r.v0;
      const uint4* blk = tw0 + (int64_t)(c < n ? c : n - 1) * p.n_v * (kTWs / 4);
      r.w0 = blk[(tid >> 7) * (kMat / 8) + 4 * tj + tq];                       // T hi, lo: 256 pieces
      r.vec = blk[2 * kMat / 8 + (tid < kVecN / 4 ? tid : kVecN / 4 - 1)];     // the vectors: 28 pieces
    };
    auto swrite = [&](Stage& st, const Pre& r) {
      const int r0 = perm_row(tid >> 4);  // row 16 + (tid >> 4): 8 staged rows on
      *reinterpret_cast<uint4*>(&st.k[r0][8 * (tid & 15)]) = r.k0;
      *reinterpret_cast<uint4*>(&st.k[r0 + 8][8 * (tid & 15)]) = r.k1;
      *reinterpret_cast<uint4*>(&st.q[r0][8 * (tid & 15)]) = r.q0;
      *reinterpret_cast<uint4*>(&st.q[r0 + 8][8 * (tid & 15)]) = r.q1;
      *reinterpret_cast<uint4*>(&st.v[perm_row(vr)][8 * vp]) = r.v0;
      if constexpr (ROWS) *reinterpret_cast<uint4*>(&st.v[perm_row(vr + kVRows)][8 * vp]) = r.v1;
      *reinterpret_cast<uint4*>(&st.tm[tid >> 7][perm_row(tj)][8 * tq]) = r.w0;
      if (tid < kVecN / 4) *reinterpret_cast<uint4*>(&st.vec[4 * tid]) = r.vec;
    };
    // P^T = K Q~^T o D^T, one 16 x 16 tile per wave: keys 8 h4 + 4 tk + r, query i
    auto pmat = [&](const Stage& st, uint16_t (*pm)[kC][kRowC]) {
      const int tk = ws >> 1, ti = ws & 1;
      v4f a = {0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < 4; ++m)
        a = mfma16(lds8(&st.k[16 * tk + lc][32 * m + 8 * h4]), lds8(&st.q[16 * ti + lc][32 * m + 8 * h4]), a);
      const int i = otok + 4 * ti, j0 = 8 * h4 + 4 * tk;
      const float gi = st.vec[i];
      const float4 gj = *reinterpret_cast<const float4*>(&st.vec[j0]);
      const float gv[4] = {gj.x, gj.y, gj.z, gj.w};
      float pv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool seen = j0 + r <= i;
        const float e = a[r] * qscale * __expf(seen ? gi - gv[r] : 0.0f);  // both selects: no branch
        pv[r] = seen ? e : 0.0f;
      }
      uint32_t hi0, lo0, hi1, lo1;
      split2(pv[0], pv[1], hi0, lo0);
      split2(pv[2], pv[3], hi1, lo1);
      *reinterpret_cast<uint2*>(&pm[0][16 * ti + lc][j0]) = make_uint2(hi0, hi1);
      *reinterpret_cast<uint2*>(&pm[1][16 * ti + lc][j0]) = make_uint2(lo0, lo1);
    };
    auto store = [&](int c) {
      const rsrc_t ro = rows_of(o0, ldv, c);
      typedef int v4i __attribute__((ext_vector_type(4)));
#pragma unroll
      for (int r = 0; r < kC; r += kVRows) {
        const uint2* src = reinterpret_cast<const uint2*>(&sm.ob[c & 1][perm_row(vr + r)][8 * vp]);
        const uint2 a = src[0], b = src[1];
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4i, make_uint4(a.x, a.y, b.x, b.y)), ro,
                                               vo + r * (int)(2 * ldv), 0, 0);
      }
    };
    Pre pa, pb;
    gload(0, pa);
    gload(1, pb);
    swrite(sm.st[0], pa);
    gload(2, pa);
    swrite(sm.st[1], pb);
    gload(3, pb);
    lds_barrier();
    pmat(sm.st[0], sm.pm[0]);
    lds_barrier();
    int nxt = 1;  // stage of chunk c + 1
    // (past the last chunk the stages and P written here are not read)
    auto step = [&](int c, Pre& r) {
      const int two = nxt == 2 ? 0 : nxt + 1;
      swrite(sm.st[two], r);
      gload(c + 4, r);
      store(c - 1);
      pmat(sm.st[nxt], sm.pm[(c + 1) & 1]);
      nxt = two;
      lds_barrier();
    };
    for (int c = 0;; c += 2) {
      step(c, pa);
      if (c + 1 >= n) break;
      step(c + 1, pb);
      if (c + 2 >= n) break;
    }
    store(n - 1);
  }
}

}  // namespace

extern "C" int od_gdn_chunk_ws_size(int64_t S, int64_t L, int64_t n_v, int64_t* ws_floats) {
  if (!ws_floats) return OD_ERR_NULL;
  if (S < 0 || L < 0 || n_v < 1) return OD_ERR_SHAPE;
  *ws_floats = S * ((L + kC - 1) / kC) * n_v * kTWs;
  return OD_OK;
}

extern "C" int od_gdn_recurrence_chunked(const uint16_t* qk, const uint16_t* v, const float* g, const float* beta,
                                         const float* init, const int32_t* seq_state, int64_t n_states, int64_t S,
                                         int64_t L, int64_t n_k, int64_t n_v, int64_t dk, int64_t dv, uint16_t* o,
                                         float* final_state, float* ws, int64_t ws_floats, od_stream_t stream) {
  if (S < 0 || L < 0 || n_k < 1 || n_v < 1 || n_states < 0) return OD_ERR_SHAPE;
  if (S == 0 || L == 0) return (S > 0 && final_state) ? OD_ERR_SHAPE : OD_OK;
  if (!qk || !v || !g || !beta || !o || !ws) return OD_ERR_NULL;
  if (dk != kDk || dv % kCols || n_v % n_k) return OD_ERR_UNSUPPORTED;
  if (!od_aligned16(qk) || !od_aligned16(v) || !od_aligned16(o) || !od_aligned16(ws)) return OD_ERR_ALIGN;
  const int64_t nchunk = (L + kC - 1) / kC;
  if (ws_floats < S * nchunk * n_v * kTWs) return OD_ERR_SHAPE;
  const int64_t tblocks = S * nchunk * n_k, cblocks = S * n_v * (dv / kCols);
  if (tblocks > 0x7fffffffll || cblocks > 0x7fffffffll || S * L > 0x7fffffffll) return OD_ERR_SHAPE;
  TArgs tp{qk, g, beta, ws, L, nchunk, (int)n_k, (int)n_v};
  gdn_chunk_t_kernel<<<dim3((unsigned)tblocks), dim3(64), 0, (hipStream_t)stream>>>(tp);
  CArgs cp{qk, v, init, seq_state, ws, o, final_state, L, nchunk, n_states, (int)n_k, (int)n_v, (int)dv, S, 1};
  // One chunk and no state kept (option rows): runs of sequences that share S_0 in registers, as few rounds of one
  // workgroup per CU as kMaxRun allows, of equal runs (rounded down, 15 x 24 tokens of 32 heads took two rounds, 19.8
  // us, and 300 x 24 141, in place of 15.6 and 95). 256 x 24 tokens, with T: over 4 states 227 us on gdn_chunk_state,
  // 82 here, over 4 in turn (a state read at every step) 227 and 118, over 256 of their own 256 and 166; 6 x 24: 17.4
  // and 12.3. Its eight chain waves take 128 columns; other widths, and a state that has to be written per sequence
  // (2 MB each, which is what such a call then takes its time for), stay on gdn_chunk_state.
  if (nchunk == 1 && !final_state && dv % (16 * kRowChain) == 0) {
    const int64_t heads = n_v * (dv / (16 * kRowChain));
    const int64_t per = (S * heads + od_cu_count() - 1) / od_cu_count(), rounds = (per + kMaxRun - 1) / kMaxRun;
    cp.run = (int)((per + rounds - 1) / rounds);
    const int64_t blocks = (S + cp.run - 1) / cp.run * heads;
    gdn_chunk_roles_kernel<true><<<dim3((unsigned)blocks), dim3(64 * (kRowChain + 4)), 0, (hipStream_t)stream>>>(cp);
    return od_launch_status();
  }
  // Two or more chunks: a role per wave (4 x 4096 tokens, 32 heads, both kernels: 508 -> 220 us; 1 x 8192: 887 -> 322;
  // 2 chunks of 4 sequences: 15.8 on gdn_chunk_state, 12.4 here). Its one workgroup per CU loses to three of the other
  // where two chunks come with more than four workgroups per CU (32 heads, 64 tokens, S = 8: 20.4 and 19.0; 16: 30.8
  // and 31.9; 32: 50 and 56; 256: 319 and 401).
  if (nchunk > 2 || (nchunk == 2 && cblocks <= 4 * od_cu_count()))
    gdn_chunk_roles_kernel<false><<<dim3((unsigned)cblocks), dim3(64 * (kChain + 4)), 0, (hipStream_t)stream>>>(cp);
  else
    gdn_chunk_state_kernel<<<dim3((unsigned)cblocks), dim3(256), 0, (hipStream_t)stream>>>(cp);
  return od_launch_status();
}
