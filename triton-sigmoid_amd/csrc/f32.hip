// fp32 inputs on the matrix cores, at the precision of the reference's fp32
// dots (tl.dot with allow_tf32=False, sigmoid_triton_dense.py:123,149,272,
// 289,299,426,443,446,456; sigmoid_triton_padded.py:138,166,297,321,331,461,
// 485,488,498).  Same semantics as the 16-bit MFMA kernels and the portable
// ones: masks are causal (key <= query, top-left) and seq_lens bounds, padded
// rows are written as zeros, packed layouts write each sequence's rows only.
//
// Products are taken on the bf16 matrix instruction, sixteen times the fp32
// one's rate, with every fp32 operand split into three bf16 parts (a = a0 + a1
// + a2, each the rounded rest of the ones before: 8 bits of significand and a
// sign each, so 24 bits are kept exactly) and the six largest of the nine
// partial products added in fp32: a0b0, a0b1, a1b0, a0b2, a1b1, a2b0.  The
// three left out are below 2^-25 of |ab|.  Against 64 bits the sum of 64
// products of N(0,1) values is 4.6e-8 off in the 2-norm with the small terms
// first, where v_mfma_f32_32x32x2_f32 is 1.4e-7 off (128 products: 1.3e-7
// against 2.0e-7; 2048: 6.9e-7 against 8.2e-7), because sixteen products join
// the accumulator with one rounding instead of two.  A 32x32 block of one
// product takes 6·D/16 instructions of 32 cycles for the fp32 instruction's
// D/2 of 64: 2.7 times fewer matrix cycles.
//
// Values that have no such split (infinities, NaN, magnitudes above bf16's
// largest) become NaN there, and magnitudes below 2^-110 lose lower bits:
// bf16's denormals, which the matrix instruction keeps, end at 2^-133, so a
// value is off by up to 2^-134 and a product by that times the other factor.
// A workgroup whose results may show it computes its rows again with
// v_mfma_f32_32x32x2_f32 (the *_full functions) and stores those.  With every
// input at most M in magnitude, S is off by 2^-126·M at most (nothing, for the
// sigmoid, unless scale or M is huge), dP as much, and a result by 2^-112·M²
// for each of its terms and roundings of its own: the rows are computed again
// where a result is NaN or below 2^-88·(M / 2^7)² (M at least 2^7), or where
// M >= 2^60 or the scale >= 2^32.  A zero is taken for one, unless M > 2^24:
// it may stand for less than 2^-110 a term.  Finding M costs one instruction
// for two split values: forward, dQ, dK/dV, us, B=2 T=1999 H=8 D=64 causal
// 73.7, 90.1, 133.7 -> 75.0, 91.4, 133.0, B=2 T=4096 H=16 D=128 causal 857,
// 1079, 1614 -> 841, 1123, 1668.
#include <type_traits>

#include "common.h"
#include "launch.h"

namespace sigattn {
namespace {

constexpr int FB = 32;        // streamed rows per wave and step, rows of an LDS tile
constexpr int FW = 4;         // waves per workgroup

// One workgroup's work: (batch, head), its first stationary row, and the end
// of its rows (not past a block of 32 rows per row group of the workgroup).
struct Item {
  int b, h, row0, row_end;
};


// ---------------------------------------------------------------------------
// v_mfma_f32_32x32x2_f32: C[i][j] += A[i][0] B[0][j] + A[i][1] B[1][j]; lane l
// gives A[l % 32][l / 32] and B[l / 32][l % 32], one float each, and holds
// C[8g + 4(l / 32) + r][l % 32] in accumulator element 4g + r.  Products over
// the head dim (S, dP) reduce d = s (lanes 0-31) and d = D/2 + s (lanes 32-63)
// in step s, so four consecutive steps take one 16-byte piece of the lane's
// row.  Products over the streamed rows (O, dQ, dK, dV) reduce rows 8g + r
// (lanes 0-31) and 8g + 4 + r (lanes 32-63) in step (g, r) -- the rows whose S
// (or dS) value the lane holds in accumulator element 4g + r -- so P and dS
// feed them as B operands where they were computed, with no data movement.
// ---------------------------------------------------------------------------
__device__ __forceinline__ f32x16 mma(float a, float b, const f32x16 &c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// The lane's stationary row, head-dim halves by lane half: v[s] = row[hi * D/2 + s]
// (zeros when !ok; for head_dim 16 in the D = 32 kernels the upper half is zero).
template <int D>
__device__ __forceinline__ void load_half_row(float (&v)[D / 2], const float *row, int hi, bool ok) {
#pragma unroll
  for (int t = 0; t < D / 8; ++t) {
    const f32x4 x = ok ? *(const f32x4 *)(row + hi * (D / 2) + 4 * t) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    v[4 * t] = x.x, v[4 * t + 1] = x.y, v[4 * t + 2] = x.z, v[4 * t + 3] = x.w;
  }
}

// acc += (rows l % 32 of tile t) · v over the head dim (S or dP).
template <int D>
__device__ __forceinline__ void head_product(f32x16 &acc, const float *t, const float (&v)[D / 2], int l32,
                                             int hi) {
#pragma unroll
  for (int c = 0; c < D / 8; ++c) {
    const f32x4 a = *(const f32x4 *)(t + F32Tile<D>::piece(l32, hi * (D / 8) + c));
    acc = mma(a.x, v[4 * c], acc);
    acc = mma(a.y, v[4 * c + 1], acc);
    acc = mma(a.z, v[4 * c + 2], acc);
    acc = mma(a.w, v[4 * c + 3], acc);
  }
}

// accᵀ[d][j] += sum over the tile's rows i of t[i][d] · w[i][j], where the
// lane holds w[8g + 4hi + r][l % 32] in element 4g + r (O, dQ, dK, dV).
template <int D>
__device__ __forceinline__ void row_product(f32x16 (&acc)[D / 32], const float *t, const float (&w)[16],
                                            const F32RowReads<D> &rr) {
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int db = 0; db < D / 32; ++db) acc[db] = mma(t[rr.at(g, r, db)], w[4 * g + r], acc[db]);
}

// Stores row `row` of an output from accᵀ (columns 32db + 8g + 4hi + r in
// element 4g + r of block db), times `mul`; zeros when !valid.
template <int D>
__device__ __forceinline__ void store_row(float *row, const f32x16 (&acc)[D / 32], float mul, bool valid, int hi,
                                          bool half) {
#pragma unroll
  for (int db = 0; db < D / 32; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      if (half && g >= 2) break;  // columns 16..31: not in the tensor
      f32x4 o = {acc[db][4 * g] * mul, acc[db][4 * g + 1] * mul, acc[db][4 * g + 2] * mul,
                 acc[db][4 * g + 3] * mul};
      if (!valid) o = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      *(f32x4 *)(row + 32 * db + 8 * g + 4 * hi) = o;
    }
}

// The workgroup's rows on the fp32 instruction: four waves of 32 stationary
// rows, the streamed rows in two stages of 32-row fp32 tiles.  `lds` holds
// 4 * FB * D floats, then (forward and dQ with score_mod) 2 * FB more.
template <int D, bool CAUSAL, bool SCOREMOD>
__device__ __forceinline__ void fwd_full(const KParams &p, const Item &w_, float *lds) {
  constexpr int NDB = D / 32;
  const int b = w_.b, h = w_.h, q0 = w_.row0;
  const int Lk = p.len_k(b), Lq = p.len_q(b), rows = min(Lq, w_.row_end);
  const bool half = p.half_head(D);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int qw = q0 + 32 * w, myq = qw + l32;
  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);
  const float *Kb = (const float *)p.k + koff, *Vb = (const float *)p.v + koff;

  const int nend = CAUSAL ? min(Lk, rows) : Lk;
  const int ntiles = (nend + FB - 1) / FB;
  // This wave's keys: causal waves stop after their own diagonal block.
  const int wend = qw >= rows ? 0 : (CAUSAL ? min(nend, qw + 32) : nend);
  const float scale = *p.scale, bias = p.bias[b];
  const float nsl = -scale * kLog2e;

  float qv[D / 2];
  load_half_row<D>(qv, (const float *)p.q + qoff + (int64_t)myq * p.sq_t, hi, myq < rows && !(half && hi));
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = zero16();
  DmaPlan<FB, 2 * D, FW> dma;
  dma.init(w, lane, half);
  F32RowReads<D> rr;
  rr.init(l32, hi);
  const int stride_bytes = (int)(p.sk_t * 4);
  for (int t = 0; t < ntiles; ++t) {
    float *tK = lds + (t & 1) * 2 * FB * D, *tV = tK + FB * D, *tC = lds + 4 * FB * D + (t & 1) * FB;
    // Stage t & 1 was last read for tile t - 2, before the barrier of tile t - 1.
    dma.issue((uint16_t *)tK, (const uint16_t *)Kb, stride_bytes, t * FB, Lk);
    dma.issue((uint16_t *)tV, (const uint16_t *)Vb, stride_bytes, t * FB, Lk);
    if (SCOREMOD && tid < FB) {
      const int key = min(t * FB + tid, Lk - 1);
      tC[tid] = -(bias + p.score_mod[p.mod_base(b) + key]) * kLog2e;
    }
    wait_dma();
    __syncthreads();
    const int k0 = t * FB;
    if (k0 >= wend) continue;
    f32x16 s = zero16();
    head_product<D>(s, tK, qv, l32, hi);
    float pr[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int kr = 8 * (i / 4) + 4 * hi + i % 4;
      const float c = SCOREMOD ? tC[kr] : -bias * kLog2e;
      pr[i] = sigmoid_from_neg_log2(__builtin_fmaf(s[i], nsl, c));
      if (k0 + kr >= Lk || (CAUSAL && k0 + kr > myq)) pr[i] = 0.0f;
    }
    row_product<D>(acc, tV, pr, rr);
  }
  if (myq < min(w_.row_end, p.q_rows_out(Lq)))
    store_row<D>((float *)p.out + qoff + (int64_t)myq * p.sq_t, acc, 1.0f, myq < Lq, hi, half);
}

template <int D, bool CAUSAL, bool SCOREMOD>
__device__ __forceinline__ void dq_full(const KParams &p, const Item &w_, float *lds) {
  constexpr int NDB = D / 32;
  const int b = w_.b, h = w_.h, q0 = w_.row0;
  const int Lk = p.len_k(b), Lq = p.len_q(b), rows = min(Lq, w_.row_end);
  const bool half = p.half_head(D);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int qw = q0 + 32 * w, myq = qw + l32;
  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);
  const float *Kb = (const float *)p.k + koff, *Vb = (const float *)p.v + koff;

  const int nend = CAUSAL ? min(Lk, rows) : Lk;
  const int ntiles = (nend + FB - 1) / FB;
  const int wend = qw >= rows ? 0 : (CAUSAL ? min(nend, qw + 32) : nend);
  const float scale = *p.scale, bias = p.bias[b];
  const float nsl = -scale * kLog2e;

  float qv[D / 2], ov[D / 2];
  const bool ok = myq < rows && !(half && hi);
  load_half_row<D>(qv, (const float *)p.q + qoff + (int64_t)myq * p.sq_t, hi, ok);
  load_half_row<D>(ov, (const float *)p.dout + qoff + (int64_t)myq * p.sq_t, hi, ok);
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = zero16();
  DmaPlan<FB, 2 * D, FW> dma;
  dma.init(w, lane, half);
  F32RowReads<D> rr;
  rr.init(l32, hi);
  const int stride_bytes = (int)(p.sk_t * 4);
  for (int t = 0; t < ntiles; ++t) {
    float *tK = lds + (t & 1) * 2 * FB * D, *tV = tK + FB * D, *tC = lds + 4 * FB * D + (t & 1) * FB;
    dma.issue((uint16_t *)tK, (const uint16_t *)Kb, stride_bytes, t * FB, Lk);
    dma.issue((uint16_t *)tV, (const uint16_t *)Vb, stride_bytes, t * FB, Lk);
    if (SCOREMOD && tid < FB) {
      const int key = min(t * FB + tid, Lk - 1);
      tC[tid] = -(bias + p.score_mod[p.mod_base(b) + key]) * kLog2e;
    }
    wait_dma();
    __syncthreads();
    const int k0 = t * FB;
    if (k0 >= wend) continue;
    f32x16 s = zero16(), dp = zero16();
    head_product<D>(s, tK, qv, l32, hi);
    head_product<D>(dp, tV, ov, l32, hi);
    float ds[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int kr = 8 * (i / 4) + 4 * hi + i % 4;
      const float c = SCOREMOD ? tC[kr] : -bias * kLog2e;
      const float pr = sigmoid_from_neg_log2(__builtin_fmaf(s[i], nsl, c)), u = pr * dp[i];
      ds[i] = __builtin_fmaf(-pr, u, u);
      if (k0 + kr >= Lk || (CAUSAL && k0 + kr > myq)) ds[i] = 0.0f;
    }
    row_product<D>(acc, tK, ds, rr);
  }
  if (myq < min(w_.row_end, p.q_rows_out(Lq)))
    store_row<D>((float *)p.dq + qoff + (int64_t)myq * p.sq_t, acc, scale, myq < Lq, hi, half);
}

template <int D, bool CAUSAL, bool SCOREMOD>
__device__ __forceinline__ void dkdv_full(const KParams &p, const Item &w_, float *lds) {
  constexpr int NDB = D / 32;
  const int b = w_.b, h = w_.h, k0 = w_.row0;
  const int Lk = p.len_k(b), Lq = p.len_q(b), rows = min(Lk, w_.row_end);
  const bool half = p.half_head(D);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int kw = k0 + 32 * w, myk = kw + l32;
  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);

  // Causal: queries before the workgroup's first key see none of its keys.
  const int mstart = CAUSAL ? min(k0, Lq) : 0;
  const int ntiles = k0 < rows ? (Lq - mstart + FB - 1) / FB : 0;
  const float scale = *p.scale, bias = p.bias[b];
  const float nsl = -scale * kLog2e;
  const bool kok = myk < rows;
  float nc = -bias * kLog2e;
  if (SCOREMOD) nc = kok ? -(bias + p.score_mod[p.mod_base(b) + myk]) * kLog2e : 0.0f;

  float kv[D / 2], vv[D / 2];
  const bool ok = kok && !(half && hi);
  load_half_row<D>(kv, (const float *)p.k + koff + (int64_t)myk * p.sk_t, hi, ok);
  load_half_row<D>(vv, (const float *)p.v + koff + (int64_t)myk * p.sk_t, hi, ok);
  f32x16 dka[NDB], dva[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) dka[db] = dva[db] = zero16();
  DmaPlan<FB, 2 * D, FW> dma;
  dma.init(w, lane, half);
  F32RowReads<D> rr;
  rr.init(l32, hi);
  const int stride_bytes = (int)(p.sq_t * 4);
  const float *Qm = (const float *)p.q + qoff + (int64_t)mstart * p.sq_t;
  const float *dOm = (const float *)p.dout + qoff + (int64_t)mstart * p.sq_t;
  for (int t = 0; t < ntiles; ++t) {
    float *tQ = lds + (t & 1) * 2 * FB * D, *tO = tQ + FB * D;
    dma.issue((uint16_t *)tQ, (const uint16_t *)Qm, stride_bytes, t * FB, Lq - mstart);
    dma.issue((uint16_t *)tO, (const uint16_t *)dOm, stride_bytes, t * FB, Lq - mstart);
    wait_dma();
    __syncthreads();
    const int m0 = mstart + t * FB;
    if (kw >= rows || (CAUSAL && m0 + FB <= kw)) continue;
    f32x16 s = zero16(), dp = zero16();
    float pr[16], ds[16];
    head_product<D>(s, tQ, kv, l32, hi);
    head_product<D>(dp, tO, vv, l32, hi);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int q = m0 + 8 * (i / 4) + 4 * hi + i % 4;
      pr[i] = sigmoid_from_neg_log2(__builtin_fmaf(s[i], nsl, nc));
      const float u = pr[i] * dp[i];
      ds[i] = __builtin_fmaf(-pr[i], u, u);
      if (q >= Lq || (CAUSAL && q < myk)) pr[i] = ds[i] = 0.0f;
    }
    row_product<D>(dva, tO, pr, rr);
    row_product<D>(dka, tQ, ds, rr);
  }
  if (myk < min(w_.row_end, p.k_rows_out(Lk))) {
    store_row<D>((float *)p.dk + koff + (int64_t)myk * p.sk_t, dka, scale, myk < Lk, hi, half);
    store_row<D>((float *)p.dv + koff + (int64_t)myk * p.sk_t, dva, 1.0f, myk < Lk, hi, half);
  }
}

// ---------------------------------------------------------------------------
// The split kernels.  Workgroup: four waves, in 4 / WK row groups of 32
// stationary rows; the WK waves of a group hold the same rows and take every
// WK-th 32-row tile of the streamed ones, and their accumulators are added in
// wave order at the end.  WK = 1 reads each streamed tile once per 128
// stationary rows; small grids take WK = 2 or 4, WK times the workgroups of a
// WK-th of the chain.
//   * The 32·WK streamed rows of a step are loaded one step ahead into
//     registers, split there and stored as three bf16 tiles per tensor
//     (swizzled as the 16-bit kernels' tiles), one stage: the other
//     workgroups of the CU run while one stores.
//   * The stationary rows are split once and stay in registers.
//   * P and dS are split where the accumulators left them, which is the B
//     operand layout of the next product (see common.h).
// ---------------------------------------------------------------------------

// Three bf16 parts of eight values, two per word.
__device__ __forceinline__ void split_pair(float x, float y, uint32_t &w0, uint32_t &w1, uint32_t &w2) {
  w0 = Elem<__bf16>::pack(x, y);
  x -= __builtin_bit_cast(float, w0 << 16);
  y -= __builtin_bit_cast(float, w0 & 0xffff0000u);
  w1 = Elem<__bf16>::pack(x, y);
  x -= __builtin_bit_cast(float, w1 << 16);
  y -= __builtin_bit_cast(float, w1 & 0xffff0000u);
  w2 = Elem<__bf16>::pack(x, y);
}
__device__ __forceinline__ void split8(f32x4 x, f32x4 y, u32x4 (&o)[3]) {
  const float v[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    uint32_t w0, w1, w2;
    split_pair(v[2 * e], v[2 * e + 1], w0, w1, w2);
    o[0][e] = w0, o[1][e] = w1, o[2][e] = w2;
  }
}

// The largest magnitude of the inputs that a thread split.
struct SplitRange {
  float top = 0.0f;
  __device__ __forceinline__ void see(f32x4 x) {
    // fmaxf would canonicalise every operand first.
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(x.x), "v"(x.y));
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(top) : "v"(x.z), "v"(x.w));
  }
  // The first parts of a stationary row, after the loop: looked at where they
  // are split, they hold up the first tile's loads (0.8 us of a 16 us kernel).
  template <int N> __device__ __forceinline__ void see(const u32x4 (&part)[N]) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 m = {0, 0};
#pragma unroll
    for (int s = 0; s < N; ++s)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, part[s][e] & 0x7fff7fffu));
    const uint32_t most = m.x > m.y ? m.x : m.y;
    top = fmaxf(top, __builtin_bit_cast(float, most << 16));
  }
  // Results need more than the look at 2^-88.
  __device__ __forceinline__ bool wide(float scale) const {
    return top > 0x1p7f || !(__builtin_fabsf(scale) < 0x1p32f);
  }
};

// The lane's stationary row as B operands of the three parts (k = 16s + 8hi + j);
// zeros when !ok and, for head_dim 16 in the D = 32 kernels, past column 16.
template <int D>
__device__ __forceinline__ void load_split_row(u32x4 (&o)[3][D / 16], const float *row, int hi, bool ok, bool half) {
#pragma unroll
  for (int s = 0; s < D / 16; ++s) {
    const bool in = ok && !(half && s > 0);
    const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
    u32x4 t[3];
    split8(in ? *(const f32x4 *)(row + 16 * s + 8 * hi) : z, in ? *(const f32x4 *)(row + 16 * s + 8 * hi + 4) : z, t);
#pragma unroll
    for (int i = 0; i < 3; ++i) o[i][s] = t[i];
  }
}

// The streamed tiles of two tensors: TR rows a step.
template <int D, int TR> struct SplitTiles {
  static constexpr int PART = TR * D;           // elements of one part of one tensor
  static constexpr int CH = TR * D / 8;         // 8-element chunks per tensor
  static constexpr int NCH = 2 * CH / (64 * FW);  // chunks per thread
  static_assert(2 * CH % (64 * FW) == 0 && CH % 64 == 0, "tile shape");
  f32x4 r[NCH][2];

  static __device__ __forceinline__ uint16_t *part(uint16_t *lds, int tensor, int i) {
    return lds + (3 * tensor + i) * PART;
  }
  // Rows row0 .. of both tensors; rows at or past nvalid are zeros and not read.
  __device__ __forceinline__ void load(const float *a, const float *c, int64_t stride, int row0, int nvalid,
                                       bool half) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const int ch = threadIdx.x + 64 * FW * i;
      const int row = row0 + ch % CH / (D / 8), col = 8 * (ch % (D / 8));
      const float *src = (ch < CH ? a : c) + (int64_t)row * stride + col;
      const bool in = row < nvalid && !(half && col >= 16);
      const f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
      r[i][0] = in ? *(const f32x4 *)src : z;
      r[i][1] = in ? *(const f32x4 *)(src + 4) : z;
    }
  }
  __device__ __forceinline__ void store(uint16_t *lds, SplitRange &rg) const {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      rg.see(r[i][0]), rg.see(r[i][1]);
      const int ch = threadIdx.x + 64 * FW * i;
      const int off = toff<D>(ch % CH / (D / 8), 8 * (ch % (D / 8)));
      u32x4 o[3];
      split8(r[i][0], r[i][1], o);
#pragma unroll
      for (int x = 0; x < 3; ++x) *(u32x4 *)&part(lds, ch < CH ? 0 : 1, x)[off] = o[x];
    }
  }
};

__device__ __forceinline__ f32x16 mb(u32x4 a, u32x4 b, f32x16 c) { return Elem<__bf16>::mfma(a, b, c); }

// (rows row16 + l % 32 of the tile whose parts start at t, PART apart) · b over
// the head dim: the five small partial products first, whose sum is below
// 2^-7 of the whole, then the large one with its D/16 roundings.
template <int D, int PART>
__device__ __forceinline__ f32x16 head3(const uint16_t *t, const TileOffsets<D> &to, int row16,
                                        const u32x4 (&b)[3][D / 16]) {
  f32x16 s = zero16();
#pragma unroll
  for (int k = 0; k < D / 16; ++k) {
    const u32x4 a0 = ld_row<D>(t, to, row16, k), a1 = ld_row<D>(t + PART, to, row16, k),
                a2 = ld_row<D>(t + 2 * PART, to, row16, k);
    s = mb(a2, b[0][k], s);
    s = mb(a1, b[1][k], s);
    s = mb(a0, b[2][k], s);
    s = mb(a1, b[0][k], s);
    s = mb(a0, b[1][k], s);
  }
#pragma unroll
  for (int k = 0; k < D / 16; ++k) s = mb(ld_row<D>(t, to, row16, k), b[0][k], s);
  return s;
}

// accᵀ[d][j] += sum over the tile's 32 rows (16-row steps ks, ks + 1) of
// t[row][d] · w[row][j], w in the accumulator layout.
template <int D, int PART>
__device__ __forceinline__ void row3(f32x16 (&acc)[D / 32], const uint16_t *t, const TileOffsets<D> &to, int ks,
                                     const float (&w)[16]) {
  uint32_t p[3][8];
#pragma unroll
  for (int e = 0; e < 8; ++e) split_pair(w[2 * e], w[2 * e + 1], p[0][e], p[1][e], p[2][e]);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    u32x4 b[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) b[i] = (u32x4){p[i][4 * j], p[i][4 * j + 1], p[i][4 * j + 2], p[i][4 * j + 3]};
#pragma unroll
    for (int db = 0; db < D / 32; ++db) {
      const u32x4 a0 = ld_tr<D>(t, to, ks + j, db), a1 = ld_tr<D>(t + PART, to, ks + j, db),
                  a2 = ld_tr<D>(t + 2 * PART, to, ks + j, db);
      f32x16 &c = acc[db];
      c = mb(a2, b[0], c);
      c = mb(a1, b[1], c);
      c = mb(a0, b[2], c);
      c = mb(a1, b[0], c);
      c = mb(a0, b[1], c);
      c = mb(a0, b[0], c);
    }
  }
}

// True where a result is NaN, or below `least` and not zero (or zero too).
template <int N> __device__ __forceinline__ bool in_doubt(const f32x16 (&acc)[N], float least, bool zeros) {
  bool bad = false;
#pragma unroll
  for (int db = 0; db < N; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float a = __builtin_fabsf(acc[db][i]);
      bad |= !(a >= least || (a == 0.0f && !zeros));
    }
  return bad;
}

// The smallest result that is not in doubt, and whether zeros are, for the
// workgroup's largest input; false where that is out of range.  All threads
// call it; no wave uses `lds` any more once all have arrived here.
__device__ __forceinline__ bool doubt_below(const SplitRange &rg, float *lds, float &least, bool &zeros) {
  uint32_t *most = (uint32_t *)lds;
  if (threadIdx.x == 0) *most = 0;
  __syncthreads();
  atomicMax(most, __builtin_bit_cast(uint32_t, rg.top));
  __syncthreads();
  const float m = __builtin_bit_cast(float, *most);
  const float r = m * 0x1p-7f > 1.0f ? m * 0x1p-7f : 1.0f;
  least = 0x1p-88f * r * r, zeros = m > 0x1p24f;
  return m < 0x1p60f;
}

// Adds the accumulators of a row group's waves into its first wave, in wave
// order, through LDS (the tiles' memory: every read of them is done).
template <int N, int WK>
__device__ __forceinline__ void add_waves(f32x16 (&acc)[N], float *lds, int w, int lane) {
  if constexpr (WK > 1) {
    const int kw = w % WK;
#pragma unroll 1
    for (int x = 1; x < WK; ++x) {
      __syncthreads();
      float *at = lds + (w / WK) * N * 1024 + 4 * lane;
      if (kw == x) {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            *(f32x4 *)(at + (4 * i + g) * 256) =
                (f32x4){acc[i][4 * g], acc[i][4 * g + 1], acc[i][4 * g + 2], acc[i][4 * g + 3]};
      }
      __syncthreads();
      if (kw == 0) {
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 v = *(const f32x4 *)(at + (4 * i + g) * 256);
            acc[i][4 * g] += v.x, acc[i][4 * g + 1] += v.y, acc[i][4 * g + 2] += v.z, acc[i][4 * g + 3] += v.w;
          }
      }
    }
  }
}

// LDS of a kernel in floats: the split tiles, or the full functions' tiles.
template <int D, int WK> constexpr int lds_floats() {
  constexpr int split = 6 * 32 * WK * D / 2, full = 4 * FB * D;
  return split > full ? split : full;
}

// Workgroups per CU that the registers are budgeted for.  They are what runs
// while one stores its tiles; with one wave per SIMD the matrix cores idle
// through its sigmoid and splits.
template <int D, int WK> constexpr int fwd_f32_occupancy() {
  return WK == 1 ? (D == 128 ? 2 : 3) : (WK * D <= 128 ? 2 : 1);
}
template <int D, int WK> constexpr int bwd_f32_occupancy() { return D < 128 && WK * D <= 128 ? 2 : 1; }

// (batch, head) and row block of a workgroup, those with the most work first:
// ragged batches in WorkOrder's order (ROWS_Q: the rows are queries), causal
// dense ones from the last query or first key block.  occ: workgroups per CU.
// Ragged, forward + backward, us, in index order / WorkOrder's: padded B=4
// T=3000 H=8 D=64 1350 / 971, packed causal B=8 T=1500 H=8 D=128 949 / 726.
// WorkOrder's passes over the batch, up to 4 us of every workgroup, need items
// of some length: forward, time of index order over WorkOrder's, lengths T/4..T,
// 0.75 to 2 blocks per CU: T=33 0.57-0.89, 128 0.71-1.05, 200 0.86-1.24, 384
// 0.96-1.30, 512 0.99-1.37.
// (Dense blocks of one head on one XCD, as the 16-bit kernels have them: B=2
// T=1024 H=8 D=64 145 -> 152.)
template <int WK, bool CAUSAL, bool ROWS_Q>
__device__ __forceinline__ Item item_of(const KParams &p, int wg, int occ) {
  constexpr int RB = 32 * FW / WK;
  if (p.ragged() && p.B <= 64 && (ROWS_Q ? p.Tk : p.Tq) > 128) {
    const auto rows = [&](int i) SIGATTN_INLINE { return ROWS_Q ? p.len_q(i) : p.len_k(i); };
    const auto stream = [&](int i) SIGATTN_INLINE { return ROWS_Q ? p.len_k(i) : p.len_q(i); };
    const WorkItem it = CAUSAL ? WorkOrder::by_level(wg, p.B, p.H, rows, RB, p.nblk, ROWS_Q, p.ncu, occ)
                               : WorkOrder::by_stream(wg, p.B, p.H, rows, RB, p.nblk, stream);
    return Item{it.b, it.h, it.blk * RB, it.blk * RB + RB};
  }
  const int BH = p.B * p.H, bh = wg % BH;
  int blk = wg / BH;
  if (CAUSAL && ROWS_Q) blk = p.nblk - 1 - blk;
  return Item{bh / p.H, bh % p.H, blk * RB, blk * RB + RB};
}

// Forward: O = sigmoid(Q·Kᵀ·scale + bias [+ score_mod]) · V, keys streamed.
template <int D, bool CAUSAL, bool SCOREMOD, int WK>
__global__ __launch_bounds__(64 * FW, (fwd_f32_occupancy<D, WK>())) void fwd_f32_kernel(const KParams p) {
  constexpr int NKS = D / 16, NDB = D / 32, TR = FB * WK;
  using Tiles = SplitTiles<D, TR>;
  __shared__ __attribute__((aligned(16))) float lds[lds_floats<D, WK>() + (SCOREMOD ? 2 * TR : 0)];
  uint16_t *tiles = (uint16_t *)lds;
  float *sC = lds + lds_floats<D, WK>();

  const int wg = gap_prologue<4>(p, lds);  // packed layouts: leading gap-zeroing workgroups
  if (wg < 0) return;
  const Item it = item_of<WK, CAUSAL, true>(p, wg, fwd_f32_occupancy<D, WK>());
  const int b = it.b, h = it.h;
  const int Lq = p.len_q(b), Lk = p.len_k(b);
  const bool half = p.half_head(D);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int qw = it.row0 + 32 * (w / WK), myq = qw + l32, wt = w % WK;

  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);
  const float *Kb = (const float *)p.k + koff, *Vb = (const float *)p.v + koff;
  int nend = Lk;
  if (CAUSAL) nend = min(nend, min(it.row_end, Lq));
  if (it.row0 >= Lq) nend = 0;
  const int nsteps = (nend + TR - 1) / TR;
  // This wave's keys: causal waves stop after their own diagonal block.
  const int wend = qw >= Lq ? 0 : (CAUSAL ? min(nend, qw + 32) : nend);
  const float scale = *p.scale, bias = p.bias[b];
  const float nsl = -scale * kLog2e, nbl = -bias * kLog2e;

  SplitRange rg;
  u32x4 qf[3][NKS];
  load_split_row<D>(qf, (const float *)p.q + qoff + (int64_t)myq * p.sq_t, hi, myq < Lq, half);
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = zero16();
  TileOffsets<D> to;
  to.init(lane);
  Tiles st;
  float creg = 0.0f;
  auto load = [&](int t) SIGATTN_INLINE {
    st.load(Kb, Vb, p.sk_t, t * TR, Lk, half);
    if (SCOREMOD && tid < TR)
      creg = t * TR + tid < Lk ? -(bias + p.score_mod[p.mod_base(b) + t * TR + tid]) * kLog2e : 0.0f;
  };
  if (nsteps > 0) load(0);
  for (int t = 0; t < nsteps; ++t) {
    __syncthreads();  // every read of step t - 1 is done
    st.store(tiles, rg);
    if (SCOREMOD && tid < TR) sC[tid] = creg;
    if (t + 1 < nsteps) load(t + 1);
    __syncthreads();
    const int k0 = t * TR + FB * wt;
    if (k0 >= wend) continue;
    const f32x16 s = head3<D, Tiles::PART>(tiles, to, FB * wt, qf);
    const bool mask = k0 + FB > Lk || (CAUSAL && k0 + FB - 1 > qw);
    const int lim = (CAUSAL ? min(Lk, myq + 1) : Lk) - k0 - 4 * hi;  // key k0 + 4hi + e valid iff e < lim
    float pr[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float c = SCOREMOD ? sC[FB * wt + 8 * (i / 4) + 4 * hi + i % 4] : nbl;
      pr[i] = sigmoid_from_neg_log2(__builtin_fmaf(s[i], nsl, c));
    }
    if (mask) {
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (8 * (i / 4) + i % 4 >= lim) pr[i] = 0.0f;
    }
    row3<D, Tiles::PART>(acc, Tiles::part(tiles, 1, 0), to, 2 * wt, pr);
  }
  add_waves<NDB, WK>(acc, lds, w, lane);
  if (wt == 0) rg.see(qf[0]);
  if (__syncthreads_or((wt == 0 && myq < Lq && in_doubt(acc, 0x1p-88f, false)) || rg.wide(scale))) {
    float least;
    bool zeros;
    const bool fits = doubt_below(rg, lds, least, zeros) && __builtin_fabsf(scale) < 0x1p32f;
    if (__syncthreads_or(!fits || (wt == 0 && myq < Lq && in_doubt(acc, least, zeros)))) {
      fwd_full<D, CAUSAL, SCOREMOD>(p, it, lds);
      return;
    }
  }
  if (wt == 0 && myq < p.q_rows_out(Lq))
    store_row<D>((float *)p.out + qoff + (int64_t)myq * p.sq_t, acc, 1.0f, myq < Lq, hi, half);
}

// dQ = (dP ⊙ P ⊙ (1 - P)) · K · scale with dP = dO · Vᵀ; keys streamed.
template <int D, bool CAUSAL, bool SCOREMOD, int WK>
__global__ __launch_bounds__(64 * FW, (bwd_f32_occupancy<D, WK>())) void dq_f32_kernel(const KParams p) {
  constexpr int NKS = D / 16, NDB = D / 32, TR = FB * WK;
  using Tiles = SplitTiles<D, TR>;
  __shared__ __attribute__((aligned(16))) float lds[lds_floats<D, WK>() + (SCOREMOD ? 2 * TR : 0)];
  uint16_t *tiles = (uint16_t *)lds;
  float *sC = lds + lds_floats<D, WK>();

  const int wg = gap_prologue<4>(p, lds);  // packed layouts: leading gap-zeroing workgroups
  if (wg < 0) return;
  const Item it = item_of<WK, CAUSAL, true>(p, wg, bwd_f32_occupancy<D, WK>());
  const int b = it.b, h = it.h;
  const int Lq = p.len_q(b), Lk = p.len_k(b);
  const bool half = p.half_head(D);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int qw = it.row0 + 32 * (w / WK), myq = qw + l32, wt = w % WK;

  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);
  const float *Kb = (const float *)p.k + koff, *Vb = (const float *)p.v + koff;
  int nend = Lk;
  if (CAUSAL) nend = min(nend, min(it.row_end, Lq));
  if (it.row0 >= Lq) nend = 0;
  const int nsteps = (nend + TR - 1) / TR;
  const int wend = qw >= Lq ? 0 : (CAUSAL ? min(nend, qw + 32) : nend);
  const float scale = *p.scale, bias = p.bias[b];
  const float nsl = -scale * kLog2e, nbl = -bias * kLog2e;

  SplitRange rg;
  u32x4 qf[3][NKS], of[3][NKS];
  load_split_row<D>(qf, (const float *)p.q + qoff + (int64_t)myq * p.sq_t, hi, myq < Lq, half);
  load_split_row<D>(of, (const float *)p.dout + qoff + (int64_t)myq * p.sq_t, hi, myq < Lq, half);
  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = zero16();
  TileOffsets<D> to;
  to.init(lane);
  Tiles st;
  float creg = 0.0f;
  auto load = [&](int t) SIGATTN_INLINE {
    st.load(Kb, Vb, p.sk_t, t * TR, Lk, half);
    if (SCOREMOD && tid < TR)
      creg = t * TR + tid < Lk ? -(bias + p.score_mod[p.mod_base(b) + t * TR + tid]) * kLog2e : 0.0f;
  };
  if (nsteps > 0) load(0);
  for (int t = 0; t < nsteps; ++t) {
    __syncthreads();
    st.store(tiles, rg);
    if (SCOREMOD && tid < TR) sC[tid] = creg;
    if (t + 1 < nsteps) load(t + 1);
    __syncthreads();
    const int k0 = t * TR + FB * wt;
    if (k0 >= wend) continue;
    const f32x16 s = head3<D, Tiles::PART>(tiles, to, FB * wt, qf);
    const f32x16 dp = head3<D, Tiles::PART>(Tiles::part(tiles, 1, 0), to, FB * wt, of);
    float ds[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float c = SCOREMOD ? sC[FB * wt + 8 * (i / 4) + 4 * hi + i % 4] : nbl;
      const float pr = sigmoid_from_neg_log2(__builtin_fmaf(s[i], nsl, c)), u = pr * dp[i];
      ds[i] = __builtin_fmaf(-pr, u, u);  // dP·P·(1 - P)
    }
    if (k0 + FB > Lk || (CAUSAL && k0 + FB - 1 > qw)) {
      const int lim = (CAUSAL ? min(Lk, myq + 1) : Lk) - k0 - 4 * hi;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (8 * (i / 4) + i % 4 >= lim) ds[i] = 0.0f;
    }
    row3<D, Tiles::PART>(acc, tiles, to, 2 * wt, ds);
  }
  add_waves<NDB, WK>(acc, lds, w, lane);
  if (wt == 0) rg.see(qf[0]), rg.see(of[0]);
  if (__syncthreads_or((wt == 0 && myq < Lq && in_doubt(acc, 0x1p-88f, false)) || rg.wide(scale))) {
    float least;
    bool zeros;
    const bool fits = doubt_below(rg, lds, least, zeros) && __builtin_fabsf(scale) < 0x1p32f;
    if (__syncthreads_or(!fits || (wt == 0 && myq < Lq && in_doubt(acc, least, zeros)))) {
      dq_full<D, CAUSAL, SCOREMOD>(p, it, lds);
      return;
    }
  }
  if (wt == 0 && myq < p.q_rows_out(Lq))
    store_row<D>((float *)p.dq + qoff + (int64_t)myq * p.sq_t, acc, scale, myq < Lq, hi, half);
}

// dV = Pᵀ · dO and dK = dSᵀ · Q · scale; queries streamed.
template <int D, bool CAUSAL, bool SCOREMOD, int WK>
__global__ __launch_bounds__(64 * FW, (bwd_f32_occupancy<D, WK>())) void dkdv_f32_kernel(const KParams p) {
  constexpr int NKS = D / 16, NDB = D / 32, TR = FB * WK;
  using Tiles = SplitTiles<D, TR>;
  __shared__ __attribute__((aligned(16))) float lds[lds_floats<D, WK>()];
  uint16_t *tiles = (uint16_t *)lds;

  const Item it = item_of<WK, CAUSAL, false>(p, blockIdx.x, bwd_f32_occupancy<D, WK>());
  const int b = it.b, h = it.h;
  const int Lq = p.len_q(b), Lk = p.len_k(b);
  const bool half = p.half_head(D);
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int k0 = it.row0, kw = k0 + 32 * (w / WK), myk = kw + l32, wt = w % WK;

  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);
  const float *Qb = (const float *)p.q + qoff, *dOb = (const float *)p.dout + qoff;
  // Queries of the workgroup: causal ones before its first key see none of its keys.
  const int mstart = CAUSAL ? min(k0, Lq) : 0;
  const int nsteps = k0 < Lk ? (Lq - mstart + TR - 1) / TR : 0;
  const float scale = *p.scale, bias = p.bias[b];
  const float nsl = -scale * kLog2e;
  const bool kok = myk < Lk;
  float nc = -bias * kLog2e;
  if (SCOREMOD) nc = kok ? -(bias + p.score_mod[p.mod_base(b) + myk]) * kLog2e : 0.0f;

  SplitRange rg;
  u32x4 kf[3][NKS], vf[3][NKS];
  load_split_row<D>(kf, (const float *)p.k + koff + (int64_t)myk * p.sk_t, hi, kok, half);
  load_split_row<D>(vf, (const float *)p.v + koff + (int64_t)myk * p.sk_t, hi, kok, half);
  f32x16 dka[NDB], dva[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) dka[db] = dva[db] = zero16();
  TileOffsets<D> to;
  to.init(lane);
  Tiles st;
  auto load = [&](int t) SIGATTN_INLINE { st.load(Qb, dOb, p.sq_t, mstart + t * TR, Lq, half); };
  if (nsteps > 0) load(0);
  for (int t = 0; t < nsteps; ++t) {
    __syncthreads();
    st.store(tiles, rg);
    if (t + 1 < nsteps) load(t + 1);
    __syncthreads();
    const int m0 = mstart + t * TR + FB * wt;
    // Nothing for keys past Lk, queries past Lq, or (causal) queries that all
    // precede the wave's first key.
    if (kw >= Lk || m0 >= Lq || (CAUSAL && m0 + FB <= kw)) continue;
    const uint16_t *tQ = tiles, *tO = Tiles::part(tiles, 1, 0);
    const f32x16 s = head3<D, Tiles::PART>(tQ, to, FB * wt, kf);
    const f32x16 dp = head3<D, Tiles::PART>(tO, to, FB * wt, vf);
    float pr[16], ds[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      pr[i] = sigmoid_from_neg_log2(__builtin_fmaf(s[i], nsl, nc));
      const float u = pr[i] * dp[i];
      ds[i] = __builtin_fmaf(-pr[i], u, u);
    }
    // Queries at or past seq_lens_q, or (causal) before the lane's key.
    if (m0 + FB > Lq || (CAUSAL && m0 < kw + 31)) {
      const int e_end = Lq - m0 - 4 * hi;               // query m0 + 4hi + e valid iff
      const int e_lo = CAUSAL ? myk - m0 - 4 * hi : 0;  // e_lo <= e < e_end
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int e = 8 * (i / 4) + i % 4;
        if (e >= e_end || e < e_lo) pr[i] = ds[i] = 0.0f;
      }
    }
    row3<D, Tiles::PART>(dva, tO, to, 2 * wt, pr);
    row3<D, Tiles::PART>(dka, tQ, to, 2 * wt, ds);
  }
  add_waves<NDB, WK>(dva, lds, w, lane);
  add_waves<NDB, WK>(dka, lds, w, lane);
  if (wt == 0) rg.see(kf[0]), rg.see(vf[0]);
  if (__syncthreads_or(rg.wide(scale) ||
                       (wt == 0 && kok && (in_doubt(dva, 0x1p-88f, false) || in_doubt(dka, 0x1p-88f, false))))) {
    float least;
    bool zeros;
    const bool fits = doubt_below(rg, lds, least, zeros) && __builtin_fabsf(scale) < 0x1p32f;
    if (__syncthreads_or(!fits ||
                         (wt == 0 && kok && (in_doubt(dva, least, zeros) || in_doubt(dka, least, zeros))))) {
      dkdv_full<D, CAUSAL, SCOREMOD>(p, it, lds);
      return;
    }
  }
  if (wt == 0 && myk < p.k_rows_out(Lk)) {
    store_row<D>((float *)p.dk + koff + (int64_t)myk * p.sk_t, dka, scale, kok, hi, half);
    store_row<D>((float *)p.dv + koff + (int64_t)myk * p.sk_t, dva, 1.0f, kok, hi, half);
  }
}

// Waves per row group.  Every workgroup streams its rows' whole range, so a
// grid of few 128-row blocks is as long as its longest one; with WK = 2 (4) the
// chain is a half (a quarter) as long in twice (four times) the workgroups, for
// as many times the tile loads and splits.  Forward + backward, us, WK = 1 / 2 /
// 4 (before, on the fp32 instruction): B=2 T=1024 H=8 D=64, 128 blocks, 218 /
// 145 / 192 (342); causal B=2 T=1999 H=8 D=64, 256 blocks, 407 / 288 / 401
// (650); causal B=1 T=2000 H=8 D=128, 128 blocks, 838 / 464 (1240); causal B=4
// T=2048 H=12 D=64, 768 blocks, 640 / 688 / 1226 (1138); causal B=4 T=4096 H=16
// D=128, 2048 blocks, 7016 / 7780 (10357).  Four waves pay where their blocks of
// 32 rows leave CUs idle (B=2 T=256 H=4 D=64: kernels 25 + 32 + 40 -> 12 + 15 +
// 16 us); 128 rows of three parts of two tensors do not fit at D = 128.
// At D = 128 two waves need the whole CU, so more than half a block per CU of
// them is two rounds: worth it where the items differ and are long.  Time of
// WK = 1 over 2, 0.75 to 1.5 blocks per CU, forward / dQ and dK/dV: T=100 0.69-0.93 /
// 0.76-1.0 (D = 64, from 1.25: 0.77-0.97 / 0.79-0.93), dense non-causal T=200 to
// 512 0.71-1.00 / 0.75-1.08, causal T=512 1.04-1.55 / 0.89-1.27; T=33 0.9-1.2.
template <int D> int f32_waves_per_rows(const KParams &p, int rows, int stream, bool causal) {
  const int64_t bh = (int64_t)p.B * p.H, blocks = bh * ((rows + 127) / 128), cus = p.ncu;
  if (D < 128 && bh * ((rows + 31) / 32) <= cus) return 4;
  if (D == 128 && stream <= 128 && blocks > cus) return 1;
  if (D >= 64 && stream > 64 && (D == 128 ? 2 : 1) * blocks > cus &&
      (stream <= 128 || (D == 128 && !causal && !p.ragged() && (stream <= 256 || blocks <= cus))))
    return 1;
  return blocks < 2 * cus ? 2 : 1;
}

// Calls launch(std::integral_constant<int, WK>, p, workgroups) with p.nblk set.
template <int D, class F> void by_waves(const KParams &kp, int rows, int stream, bool causal, F &&launch) {
  KParams p = kp;
  const auto go = [&](auto wk) {
    constexpr int RB = 32 * FW / decltype(wk)::value;
    p.nblk = (rows + RB - 1) / RB;
    launch(wk, p, (int64_t)p.nblk * p.B * p.H);
  };
  switch (f32_waves_per_rows<D>(p, rows, stream, causal)) {
    case 4:
      if constexpr (D < 128) return go(std::integral_constant<int, 4>{});
      break;
    case 2: return go(std::integral_constant<int, 2>{});
    default: break;
  }
  go(std::integral_constant<int, 1>{});
}

template <int D> void fwd_t(const KParams &kp, bool causal, bool scoremod, hipStream_t st) {
  by_waves<D>(kp, kp.Tq, kp.Tk, causal, [&](auto wk, const KParams &p, int64_t n) {
    constexpr int WK = decltype(wk)::value;
    const dim3 grid((unsigned)(n + p.ngap[0] + p.ngap[1])), block(64 * FW);
    if (causal) {
      if (scoremod) fwd_f32_kernel<D, true, true, WK><<<grid, block, 0, st>>>(p);
      else fwd_f32_kernel<D, true, false, WK><<<grid, block, 0, st>>>(p);
    } else {
      if (scoremod) fwd_f32_kernel<D, false, true, WK><<<grid, block, 0, st>>>(p);
      else fwd_f32_kernel<D, false, false, WK><<<grid, block, 0, st>>>(p);
    }
  });
}

template <int D> void dq_t(const KParams &kp, bool causal, bool scoremod, hipStream_t st) {
  by_waves<D>(kp, kp.Tq, kp.Tk, causal, [&](auto wk, const KParams &p, int64_t n) {
    constexpr int WK = decltype(wk)::value;
    const dim3 grid((unsigned)(n + p.ngap[0] + p.ngap[1])), block(64 * FW);
    if (causal) {
      if (scoremod) dq_f32_kernel<D, true, true, WK><<<grid, block, 0, st>>>(p);
      else dq_f32_kernel<D, true, false, WK><<<grid, block, 0, st>>>(p);
    } else {
      if (scoremod) dq_f32_kernel<D, false, true, WK><<<grid, block, 0, st>>>(p);
      else dq_f32_kernel<D, false, false, WK><<<grid, block, 0, st>>>(p);
    }
  });
}

template <int D> void dkdv_t(const KParams &kp, bool causal, bool scoremod, hipStream_t st) {
  by_waves<D>(kp, kp.Tk, kp.Tq, causal, [&](auto wk, const KParams &p, int64_t n) {
    constexpr int WK = decltype(wk)::value;
    const dim3 grid((unsigned)n), block(64 * FW);  // no gap rows here (the dQ launch's)
    if (causal) {
      if (scoremod) dkdv_f32_kernel<D, true, true, WK><<<grid, block, 0, st>>>(p);
      else dkdv_f32_kernel<D, true, false, WK><<<grid, block, 0, st>>>(p);
    } else {
      if (scoremod) dkdv_f32_kernel<D, false, true, WK><<<grid, block, 0, st>>>(p);
      else dkdv_f32_kernel<D, false, false, WK><<<grid, block, 0, st>>>(p);
    }
  });
}

}  // namespace

void launch_fwd_f32(const KParams &p, int D, bool causal, bool scoremod, hipStream_t st) {
  if (D == 128) fwd_t<128>(p, causal, scoremod, st);
  else if (D == 64) fwd_t<64>(p, causal, scoremod, st);
  else fwd_t<32>(p, causal, scoremod, st);
}

void launch_bwd_dq_f32(const KParams &p, int D, bool causal, bool scoremod, hipStream_t st) {
  if (D == 128) dq_t<128>(p, causal, scoremod, st);
  else if (D == 64) dq_t<64>(p, causal, scoremod, st);
  else dq_t<32>(p, causal, scoremod, st);
}

void launch_bwd_dkdv_f32(const KParams &p, int D, bool causal, bool scoremod, hipStream_t st) {
  if (D == 128) dkdv_t<128>(p, causal, scoremod, st);
  else if (D == 64) dkdv_t<64>(p, causal, scoremod, st);
  else dkdv_t<32>(p, causal, scoremod, st);
}

}  // namespace sigattn
