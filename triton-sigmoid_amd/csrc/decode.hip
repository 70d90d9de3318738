// Split-KV forward for short query blocks (Tq <= 32, non-causal): the decode
// and chunked-prefill shape, where the 256-query tiles of the main forward
// kernel would leave most MFMA rows empty and one workgroup per (batch, head)
// could not fill the GPU.
//
// Semantics are the forward's (src/triton_sigmoid/sigmoid_triton_padded.py:
// 24-171 in the reference, as in fwd.hip): O = sigmoid(Q·Kᵀ·scale + bias +
// score_mod)·V with P rounded to the I/O dtype, fp32 accumulation, padded query
// rows zero.  Sigmoid attention has no row normalisation, so O over a key range
// is the plain sum of O over its parts: the keys of each (batch, head) are cut
// into nsplit chunks, one workgroup per chunk writes an fp32 partial, and a
// second kernel sums the partials in chunk order (deterministic).  With one
// chunk the workgroup writes O itself and no workspace is used.
//
// Workgroup: four waves, 32 queries (the MFMA's 32 columns); the waves share
// one key chunk or take one each (unit_waves below).  Each wave streams its
// own 32-key blocks through a private two-stage LDS ring with direct
// global->LDS copies and waits for them with its own vmcnt, so the key loop has
// no workgroup barriers.  The kernel is HBM-bound (2·D·2 bytes of K and V per
// key against 4·D·32 MFMA FLOPs), so each block is computed as a plain
// sequence: Sᵀ = K·Qᵀ, P = sigmoid(Sᵀ) on packed words, Oᵀ += Vᵀ·Pᵀ.
#include <atomic>
#include <mutex>

#include "common.h"
#include "launch.h"

namespace sigattn {

// Partials of sigattn_fwd_noalloc's split-KV launches.  In host code the name
// `scratch` is only a stand-in for the symbol: its device address (one per
// GPU) comes from hipGetSymbolAddress and is what kernels are given.  Every
// call on a GPU uses that GPU's one array, so calls that overlap on one GPU
// (two streams, two threads) race.  No clearing is needed: the reduction reads
// exactly the partials the chunk kernel of the same call writes.
static __device__ __align__(256) float scratch[kSplitScratchBytes / sizeof(float)];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<float *> g_scratch[kMaxDevices];
std::mutex g_scratch_mu;
}  // namespace

hipError_t splitkv_scratch(float **ptr) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  float *p = g_scratch[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    // First call on this device (which is current): look the address up.
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch[dev].load(std::memory_order_relaxed);
    if (p == nullptr) {
      // The first call may come while this thread captures a graph in the
      // global mode, which refuses runtime calls it deems unsafe; the lookup
      // enqueues nothing, so it runs in the relaxed mode, and the thread's
      // mode is restored afterwards.
      hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
      e = hipThreadExchangeStreamCaptureMode(&mode);
      if (e != hipSuccess) return e;
      void *addr = nullptr;
      e = hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch));
      const hipError_t restore = hipThreadExchangeStreamCaptureMode(&mode);
      if (e == hipSuccess) e = restore;
      if (e != hipSuccess) return e;
      if (addr == nullptr) return hipErrorInvalidSymbol;
      p = static_cast<float *>(addr);
      g_scratch[dev].store(p, std::memory_order_release);
    }
  }
  *ptr = p;
  return hipSuccess;
}

// Two forms of the chunk kernel, by the waves that share a unit (one chunk
// of one (batch, head)):
//   * WPU = 4: the workgroup's waves take every fourth 32-key block of its
//     chunk and add their partials through LDS -- short caches, where there
//     are too few chunks to give every wave one of its own, or too few bytes to
//     pay for partials and a second launch;
//   * WPU = 1: every wave has a unit of its own, the units of one key range
//     in head order, so the four waves of a workgroup read the rows of four
//     neighbouring heads (4 * 2 * D contiguous bytes of every [B, T, H, D]
//     row) and never wait for each other.  What bounds the kernel is the read
//     of K and V, and how fast that goes follows from the contiguous bytes a
//     workgroup reads at a time and from the loads' cache policy.  A plain
//     read of 1 GiB by 256-byte (128-byte) rows of one head per workgroup
//     reaches 6.0 (5.0) TB/s, non-temporal 6.4 (5.7), by four heads per
//     workgroup and non-temporal 6.8 (6.8), and contiguous 6.8.  The calls
//     themselves, from WPU = 4 with plain loads: bf16 B=16 H=32 D=128 Tq=1
//     Tk=8192 493 -> 323 us (6.6 TB/s), B=1 Tk=131072 390 -> 324 us, B=32
//     H=32 D=64 Tq=4 Tk=4096 216 -> 166 us (6.9 TB/s without the calls' other
//     launches); one-wave workgroups on the heads of one XCD took 348, 364 and
//     214 us, two-wave ones 317, 317 and 191.
//     Ragged caches would leave such units uneven, so the device cuts the
//     sequences of batches of up to 64 (WaveUnits): p.rows chunks in all, of
//     about equal length.
// A wave's K and V blocks have two stages each; the K stage is refilled as
// soon as S is computed and the V stage after the output product, so three of
// the four blocks are in flight at any time.
// The cut of a batch (B <= 64, keys < 2^20 each) into at most p.rows chunks of
// equal length or nearly so, from the lengths on the device; every wave
// of the chunk kernel computes it alike (in the reduction too it took 10 us more
// at 4096 output rows: B=32 H=32 D=64 Tq=4 Tk=4096 178 -> 190 us), and leaves
// each sequence's first row and chunk length for the reduction.  The longest chunk C is the
// smallest of 64 candidates, one a lane, from total / rows (at least p.chunk)
// upwards that gives at most p.rows chunks: sum ceil(L / C) <= total / C + B,
// and the last candidate is 2.9 times the first, so one fits where B <= rows / 2.
// A sequence of L keys then has n = ceil(L / C) chunks of ceil(L / n) keys.
struct WaveUnits {
  int len, n;  // of sequence `lane`

  // ceil(L / C) by the half-integer quotient, which is off every integer by
  // 1 / 2C, more than its rounding error for L < 2^20.
  static __device__ __forceinline__ int ceil_div(int L, float rc) {
    return L > 0 ? (int)(((float)L - 0.5f) * rc) + 1 : 0;
  }
  __device__ __forceinline__ WaveUnits(const KParams &p, int lane) {
    len = lane < p.B ? p.len_k(lane) : 0;
    int total = 0;  // < 2^26
    for (int i = 0; i < p.B; ++i) total += __builtin_amdgcn_readlane(len, i);
    // Too few keys for p.rows chunks of p.chunk: one round of the GPU's waves
    // rather than a second, nearly empty one.
    int rows = p.rows;
    if (total < rows * (int64_t)p.chunk && p.round_rows > 0 && total >= p.round_rows * (int64_t)p.chunk)
      rows = p.round_rows;
    const int c0 = (max((total + rows - 1) / rows, p.chunk) + 31) / 32;  // in blocks of 32 keys
    const int c = 32 * (c0 + (c0 * lane * lane + 2047) / 2048);
    float rc = 1.0f / (float)c;
    int count = 0;
    for (int i = 0; i < p.B; ++i) count += ceil_div(__builtin_amdgcn_readlane(len, i), rc);
    const int j = __builtin_ctzll(__ballot(count <= rows) | (1ull << 63));
    rc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rc), j));
    n = ceil_div(len, rc);
  }
  // Keys of one chunk of sequence b; its last chunks may be empty.
  __device__ __forceinline__ int keys(int b) const {
    const int L = __builtin_amdgcn_readlane(len, b), m = __builtin_amdgcn_readlane(n, b);
    return ((L + m - 1) / max(m, 1) + 31) & ~31;
  }
};

// (first row, keys of a chunk) of every sequence with keys, after the partials.
__device__ __forceinline__ int2 *cut_of(const KParams &p, int D) {
  return (int2 *)(p.ws + (int64_t)p.rows * p.H * p.Tq * D);
}

template <typename T, int D, int WPU, bool SCOREMOD, bool DIRECT>
__global__ __launch_bounds__(256, 1) void fwd_splitkv_kernel(const KParams p) {
  constexpr int NW = 4;
  constexpr int KB = 32;         // keys per block (one MFMA contraction of 2 k-steps)
  constexpr int NKS = D / 16, NDB = D / 32;
  using Plan = DmaPlan<KB, D, 1>;
  constexpr int NI = Plan::NI;   // copy instructions per block of V
  constexpr int NK = NI + (SCOREMOD ? 1 : 0);  // ... of K, with its keys' score_mod

  __shared__ __attribute__((aligned(16))) uint16_t sK[NW][2][KB * D];
  __shared__ __attribute__((aligned(16))) uint16_t sV[NW][2][KB * D];
  __shared__ __attribute__((aligned(16))) float sM[SCOREMOD ? NW : 1][2][64];
  static_assert(WPU == 1 || sizeof(sK) >= NW * 32 * D * sizeof(float), "reduction buffer");

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, hi = lane >> 5;
  const int NS = p.nsplit;
  int s, b, h, C = p.chunk;
  int64_t row;  // of the partials: (chunk, batch), or the unit's of WaveUnits
  if (WPU == 1 && !DIRECT && p.rows > 0) {
    const unsigned u = blockIdx.x * NW + w, H = p.H, r = u / H;
    if (r >= (unsigned)p.rows) return;
    h = (int)(u - r * H);
    row = r;
    const WaveUnits wu(p, lane);
    s = (int)r;
    for (b = 0; b < p.B; ++b) {
      const int n = __builtin_amdgcn_readlane(wu.n, b);
      if (s < n) break;
      s -= n;
    }
    if (b == p.B) return;
    C = wu.keys(b);
    if (s == 0 && h == 0 && lane == 0) cut_of(p, D)[b] = make_int2((int)r, C);
  } else if (WPU == 1) {
    const unsigned u = blockIdx.x * NW + w, H = p.H, r = u / H;  // units fit 31 bits (sigattn_check)
    if (u >= H * (unsigned)p.B * (unsigned)NS) return;
    h = (int)(u - r * H);
    s = (int)(r % (unsigned)NS);
    b = (int)(r / (unsigned)NS);
    row = (int64_t)s * p.B + b;
  } else {
    const int bh = blockIdx.x / NS;
    s = blockIdx.x % NS, b = bh / p.H, h = bh % p.H;
    row = (int64_t)s * p.B + b;
  }
  const int wu = WPU == 1 ? 0 : w;  // the wave's place in its unit
  const int Lq = p.len_q(b), Lk = p.len_k(b);
  const int k0 = s * C, k1 = min(k0 + C, Lk);
  // A chunk past the keys has no partial (the reduction stops before it).
  if (!DIRECT && (k0 >= Lk || Lq == 0)) return;

  const int64_t qoff = p.q_base(b, h), koff = p.k_base(b, h);
  const uint16_t *Qb = (const uint16_t *)p.q + qoff;
  const uint16_t *Kb = (const uint16_t *)p.k + koff;
  const uint16_t *Vb = (const uint16_t *)p.v + koff;

  const float scale = *p.scale;
  const float bias = p.bias[b];
  const float nsl = -scale * kLog2e, nbl = -bias * kLog2e;

  // Query l32 as the B operand (k = d = 16s + 8h + j); rows past Lq are zero.
  u32x4 qf[NKS];
  {
    const bool ok = l32 < Lq;
    const uint16_t *qrow = Qb + (int64_t)l32 * p.sq_t + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) qf[ks] = ok ? *(const u32x4 *)(qrow + 16 * ks) : zero4();
  }

  f32x16 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = zero16();

  TileOffsets<D> to;
  to.init(lane);
  Plan dma;
  dma.init(0, lane);
  const int kv_stride_bytes = (int)(p.sk_t * 2);
  const int nb = k1 > k0 ? (k1 - k0 + KB - 1) / KB : 0;     // blocks of the unit
  const int nbw = nb > wu ? (nb - wu + WPU - 1) / WPU : 0;  // ... of this wave
  auto first_key = [&](int i) SIGATTN_INLINE { return k0 + KB * (wu + WPU * i); };
  const float *mod = SCOREMOD ? p.score_mod + p.mod_base(b) : nullptr;
  auto issue_k = [&](int i) SIGATTN_INLINE {
    dma.template issue<WPU == 1>(sK[w][i & 1], Kb, kv_stride_bytes, first_key(i), Lk);
    if constexpr (SCOREMOD) {
      // Keys first_key(i) + lane (the block's 32 are used; rows past Lk as in
      // the K copy): lane l writes LDS bytes dst + 4 l.
      const uint32_t off = 4u * (uint32_t)min(first_key(i) + lane, Lk - 1);
      const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)sM[w][i & 1]);
      asm volatile("s_nop 0\n\tglobal_load_lds_dword %0, %1" : : "v"(off), "s"(mod), "{m0}"(dst) : "memory");
    }
  };
  auto issue_v = [&](int i) SIGATTN_INLINE {
    dma.template issue<WPU == 1>(sV[w][i & 1], Vb, kv_stride_bytes, first_key(i), Lk);
  };

#pragma unroll
  for (int i = 0; i < 2; ++i)
    if (i < nbw) {
      issue_k(i);
      issue_v(i);
    }
  // The wait for Q (which also waits for the copies above) stays out of the loop.
#pragma unroll
  for (int ks = 0; ks < NKS; ++ks) asm volatile("" ::"v"(qf[ks]));
  for (int i = 0; i < nbw; ++i) {
    // Copies in issue order: K(i) V(i) K(i+1) V(i+1) K(i+2) ...
    if (i + 1 < nbw) wait_vm<2 * NI + NK>();
    else wait_vm<NI>();
    const uint16_t *tK = sK[w][i & 1];
    const uint16_t *tV = sV[w][i & 1];

    f32x16 sc = zero16();
    float c[16];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      f32x4 m = {nbl, nbl, nbl, nbl};
      if (SCOREMOD) {
        const f32x4 x = *(const f32x4 *)&sM[w][i & 1][8 * g + 4 * hi];
#pragma unroll
        for (int j = 0; j < 4; ++j) m[j] = -(bias + x[j]) * kLog2e;
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) c[4 * g + j] = m[j];
    }
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) sc = Elem<T>::mfma(ld_row<D>(tK, to, 0, ks), qf[ks], sc);
    if (i + 2 < nbw) {
      // Every read of K(i) has returned before the copy that replaces it.
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue_k(i + 2);
    }

    // P words: accumulator element i of lane (l32, hi) is key
    // kb + 8(i/4) + 4hi + i%4 of query l32; keys at or past k1 get P = 0.
    const int kb = first_key(i);
    uint32_t pk[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i0 = 2 * e;
      const int key = kb + 8 * (i0 / 4) + 4 * hi + (i0 % 4);
      float p0 = sigmoid_from_neg_log2(__builtin_fmaf(sc[i0], nsl, c[i0]));
      float p1 = sigmoid_from_neg_log2(__builtin_fmaf(sc[i0 + 1], nsl, c[i0 + 1]));
      p0 = key < k1 ? p0 : 0.0f;
      p1 = key + 1 < k1 ? p1 : 0.0f;
      pk[e] = Elem<T>::pack(p0, p1);
    }
    if (i + 2 < nbw) wait_vm<NI + 2 * NK>();
    else if (i + 1 < nbw) wait_vm<NI + NK>();
    else wait_vm<0>();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const u32x4 bp = (u32x4){pk[4 * j], pk[4 * j + 1], pk[4 * j + 2], pk[4 * j + 3]};
#pragma unroll
      for (int db = 0; db < NDB; ++db) acc[db] = Elem<T>::mfma(ld_tr<D>(tV, to, j, db), bp, acc[db]);
    }
    if (i + 2 < nbw) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      issue_v(i + 2);
    }
  }

  float *ws_row = nullptr;
  if (!DIRECT) ws_row = p.ws + (row * p.H + h) * p.Tq * D;
  uint16_t *Ob = (uint16_t *)p.out + qoff;
  if constexpr (WPU == 1) {
    const bool valid = l32 < Lq;
    if (l32 < (DIRECT ? min(32, p.q_rows_out(Lq)) : min(32, Lq))) {
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d0 = db * 32 + 8 * g + 4 * hi;
          const f32x4 v = {acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]};
          if (DIRECT) {
            u32x2 o = {Elem<T>::pack(v.x, v.y), Elem<T>::pack(v.z, v.w)};
            if (!valid) o = (u32x2){0u, 0u};
            *(u32x2 *)(Ob + (int64_t)l32 * p.sq_t + d0) = o;
          } else {
            *(f32x4 *)(ws_row + l32 * D + d0) = v;
          }
        }
    }
    return;
  }

  // Sum the waves' Oᵀ partials: red[w][q][d] in the tile memory.
  float *red = (float *)&sK[0][0][0];
  __syncthreads();
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int d0 = db * 32 + 8 * g + 4 * hi;
      *(float4 *)&red[(w * 32 + l32) * D + d0] =
          make_float4(acc[db][4 * g], acc[db][4 * g + 1], acc[db][4 * g + 2], acc[db][4 * g + 3]);
    }
  __syncthreads();
  const int nrows = DIRECT ? min(32, p.q_rows_out(Lq)) : min(32, Lq);
  for (int it = tid; it < nrows * (D / 4); it += 64 * NW) {
    const int q = it / (D / 4), d0 = 4 * (it % (D / 4));
    float4 v = *(const float4 *)&red[q * D + d0];
#pragma unroll
    for (int x = 1; x < NW; ++x) {
      const float4 u = *(const float4 *)&red[(x * 32 + q) * D + d0];
      v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
    }
    if (DIRECT) {
      u32x2 o;
      o.x = Elem<T>::pack(v.x, v.y);
      o.y = Elem<T>::pack(v.z, v.w);
      if (q >= Lq) o = (u32x2){0u, 0u};
      *(u32x2 *)(Ob + (int64_t)q * p.sq_t + d0) = o;
    } else {
      *(float4 *)&ws_row[q * D + d0] = v;
    }
  }
}

// O = sum of the chunks' partials; padded query rows are zero.  One output
// row per workgroup: 256 / (D/4) thread groups each add every NG-th chunk's
// partial in chunk order, and the groups' sums are added in group order, so
// the sum is deterministic and its chain of loads NG times shorter than one
// thread's over all chunks.
template <typename T, int D>
__global__ __launch_bounds__(256) void fwd_splitkv_reduce_kernel(const KParams p) {
  constexpr int CG = D / 4, NG = 256 / CG;
  __shared__ f32x4 part[NG][CG];
  const int c = threadIdx.x % CG, g = threadIdx.x / CG;
  const int q = (int)(blockIdx.x % p.Tq);
  const int bh = (int)(blockIdx.x / p.Tq), b = bh / p.H, h = bh % p.H;
  const int Lq = p.len_q(b), Lk = p.len_k(b);
  if (q >= p.q_rows_out(Lq)) return;
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if (q < Lq) {
    int C = p.chunk;
    int64_t row = b, rows = p.B;  // first partial of (b, h), and rows from one to the next
    if (p.rows > 0 && Lk > 0) {
      const int2 cut = cut_of(p, D)[b];
      row = cut.x, C = cut.y, rows = 1;
    }
    const int nvs = (Lk + C - 1) / C;
    const int64_t step = rows * p.H * p.Tq * D;
    const float *src = p.ws + ((row * p.H + h) * p.Tq + q) * D + 4 * c;
#pragma unroll 4
    for (int s = g; s < nvs; s += NG) v += *(const f32x4 *)(src + s * step);
  }
  part[g][c] = v;
  __syncthreads();
  if (g != 0) return;
#pragma unroll
  for (int x = 1; x < NG; ++x) v += part[x][c];
  const u32x2 o = {Elem<T>::pack(v.x, v.y), Elem<T>::pack(v.z, v.w)};
  *(u32x2 *)((uint16_t *)p.out + p.q_base(b, h) + (int64_t)q * p.sq_t + 4 * c) = o;
}

template <typename T, int D, int WPU>
static void launch_chunks(const KParams &p, bool scoremod, hipStream_t st) {
  const int64_t units = p.rows > 0 ? (int64_t)p.rows * p.H : (int64_t)p.B * p.H * p.nsplit;
  const dim3 grid((unsigned)(WPU == 1 ? (units + 3) / 4 : units)), block(256);
  if (p.nsplit == 1) {
    if (scoremod) fwd_splitkv_kernel<T, D, WPU, true, true><<<grid, block, 0, st>>>(p);
    else fwd_splitkv_kernel<T, D, WPU, false, true><<<grid, block, 0, st>>>(p);
  } else {
    if (scoremod) fwd_splitkv_kernel<T, D, WPU, true, false><<<grid, block, 0, st>>>(p);
    else fwd_splitkv_kernel<T, D, WPU, false, false><<<grid, block, 0, st>>>(p);
  }
}

template <typename T, int D>
static void launch_splitkv_t(const KParams &p, bool scoremod, hipStream_t st) {
  if (p.unit_waves == 1) launch_chunks<T, D, 1>(p, scoremod, st);
  else launch_chunks<T, D, 4>(p, scoremod, st);
  if (p.nsplit > 1)
    fwd_splitkv_reduce_kernel<T, D><<<dim3((unsigned)((int64_t)p.B * p.H * p.Tq)), dim3(256), 0, st>>>(p);
}

void launch_fwd_splitkv(const KParams &p, int dtype, int D, bool scoremod, hipStream_t st) {
  if (dtype == kBF16) {
    if (D == 128) launch_splitkv_t<__bf16, 128>(p, scoremod, st);
    else launch_splitkv_t<__bf16, 64>(p, scoremod, st);
  } else {
    if (D == 128) launch_splitkv_t<_Float16, 128>(p, scoremod, st);
    else launch_splitkv_t<_Float16, 64>(p, scoremod, st);
  }
}

}  // namespace sigattn
