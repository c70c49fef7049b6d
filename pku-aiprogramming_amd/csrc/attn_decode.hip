// Single-query decode attention for gfx950: o = softmax(s q K^T) V per (b, h).
//
// The reference's op chain with Lq = 1 (Q @ K^T -> * s -> softmax -> @ V,
// optimizer/operators.py:163-164, 234-239, 611-612, 416-419) is a pair of
// GEMVs over the K/V cache: about 1 flop per byte, so the kernel is bound by
// HBM bandwidth and is built to stream K and V exactly once.
//
// Split-KV: workgroup id = bh * nsplit + split owns keys [split*chunk, (split+1)*chunk)
// of one head.  (attn_decode_short_kernel below takes the problems with too
// few heads and keys to fill the chip that way.)  Phase 1 streams its K rows
// (16-byte non-temporal loads, TPR threads per row, several rows in flight per thread) and writes the log2-domain scores
// to LDS; phase 2 reduces max and sum over the chunk; phase 3 streams the V
// rows and accumulates sum_j p_j V_j.  Each split writes its sums, not yet
// divided, and its max and sum of weights (o_c, m_c, l_c) in fp32; a combine kernel
// merges them:
//   m = max_c m_c,  l = sum_c 2^(m_c - m) l_c,  o = sum_c 2^(m_c - m) o_c / l.
// When one split covers a whole head, the split kernel writes o and lse
// itself and there is no combine launch.
#include <hip/hip_runtime.h>

#include <cmath>
#include <optional>

#include "attn_common.h"
#include "attn_tiles.h"

namespace tt {

constexpr int DEC_THREADS = 256;
// Keys per split: the split kernel keeps the chunk's scores in LDS, and is
// built for chunks up to 1024 keys (4 KB of scores) and up to 8192 (32 KB).
constexpr int DEC_SMALL_CHUNK = 1024;
constexpr int DEC_MAX_CHUNK = 8192;

template <typename T> struct Vec16;  // 16 bytes of T as floats
template <> struct Vec16<u16> {
  static constexpr int N = 8;
  __device__ static void cvt(const uint4& v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f[2 * i] = __uint_as_float(w[i] << 16);
      f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};
template <> struct Vec16<float> {
  static constexpr int N = 4;
  __device__ static void cvt(const uint4& v, float* f) {
    f[0] = __uint_as_float(v.x);
    f[1] = __uint_as_float(v.y);
    f[2] = __uint_as_float(v.z);
    f[3] = __uint_as_float(v.w);
  }
};

__device__ __forceinline__ float block_reduce(float v, float* red, bool is_max) {
  // wave-level butterfly, then across the 4 waves through LDS
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    float o = __shfl_xor(v, off, 64);
    v = is_max ? fmaxf(v, o) : v + o;
  }
  const int w = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[w] = v;
  __syncthreads();
  float r = red[0];
#pragma unroll
  for (int i = 1; i < DEC_THREADS / 64; ++i) r = is_max ? fmaxf(r, red[i]) : r + red[i];
  return r;
}

// MAXC: largest chunk the LDS score buffer holds.  DIRECT (nsplit == 1): o
// and lse (natural log, may be null) are written here in the output type;
// otherwise the fp32 partials go to part_o / part_ml.
template <typename T, int D, int UNROLL, int MAXC, bool DIRECT>
__global__ __launch_bounds__(DEC_THREADS) void attn_decode_split_kernel(
    const T* __restrict__ q, const T* __restrict__ K, const T* __restrict__ V,
    float* __restrict__ part_o, float2* __restrict__ part_ml, T* __restrict__ o, float* __restrict__ lse,
    int Lkv, int nsplit, int chunk, float sl2) {
  constexpr int EPT = Vec16<T>::N;     // elements per 16-byte load
  constexpr int TPR = D / EPT;         // threads per key row
  constexpr int RPP = DEC_THREADS / TPR;  // rows per pass
  __shared__ float sS[MAXC];
  __shared__ float sAcc[RPP * D];
  __shared__ float red[DEC_THREADS / 64];

  const int split = blockIdx.x % nsplit;
  const int64_t bh = blockIdx.x / nsplit;
  const int tid = threadIdx.x, col = tid % TPR, rsub = tid / TPR;
  const int kbeg = split * chunk;
  const int n = min(chunk, Lkv - kbeg);
  const T* Kh = K + (bh * Lkv + kbeg) * D + col * EPT;
  const T* Vh = V + (bh * Lkv + kbeg) * D + col * EPT;

  float qv[EPT];
  Vec16<T>::cvt(ldg16(q + bh * D + col * EPT), qv);
#pragma unroll
  for (int e = 0; e < EPT; ++e) qv[e] *= sl2;

  // Phase 1: scores s_j = (s log2 e) q . k_j
  for (int j0 = rsub; j0 < n; j0 += RPP * UNROLL) {
    uint4 kv[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int j = j0 + u * RPP;
      kv[u] = j < n ? ldg16_stream(Kh + (int64_t)j * D) : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float kf[EPT];
      Vec16<T>::cvt(kv[u], kf);
      float dot = 0.f;
#pragma unroll
      for (int e = 0; e < EPT; ++e) dot += qv[e] * kf[e];
#pragma unroll
      for (int off = TPR / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
      const int j = j0 + u * RPP;
      if (col == 0 && j < n) sS[j] = dot;
    }
  }
  __syncthreads();

  // Phase 2: max and sum over the chunk
  float mx = -INFINITY;
  for (int j = tid; j < n; j += DEC_THREADS) mx = fmaxf(mx, sS[j]);
  mx = block_reduce(mx, red, true);
  float sm = 0.f;
  for (int j = tid; j < n; j += DEC_THREADS) {
    const float p = fast_exp2(sS[j] - mx);
    sS[j] = p;
    sm += p;
  }
  sm = block_reduce(sm, red, false);  // its barriers also publish sS

  // Phase 3: acc = sum_j p_j V_j over this thread's rows
  float acc[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) acc[e] = 0.f;
  for (int j0 = rsub; j0 < n; j0 += RPP * UNROLL) {
    uint4 vv[UNROLL];
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int j = j0 + u * RPP;
      vv[u] = j < n ? ldg16_stream(Vh + (int64_t)j * D) : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int j = j0 + u * RPP;
      const float p = j < n ? sS[j] : 0.f;
      float vf[EPT];
      Vec16<T>::cvt(vv[u], vf);
#pragma unroll
      for (int e = 0; e < EPT; ++e) acc[e] += p * vf[e];
    }
  }
#pragma unroll
  for (int e = 0; e < EPT; ++e) sAcc[rsub * D + col * EPT + e] = acc[e];
  __syncthreads();
  const float inv = 1.f / sm;
  const int64_t pidx = bh * nsplit + split;
  for (int dd = tid; dd < D; dd += DEC_THREADS) {
    float s = 0.f;
#pragma unroll 8
    for (int r = 0; r < RPP; ++r) s += sAcc[r * D + dd];
    if constexpr (!DIRECT)
      part_o[pidx * D + dd] = s;
    else if constexpr (sizeof(T) == 2)
      o[bh * D + dd] = f32_to_bf16(s * inv);
    else
      o[bh * D + dd] = s * inv;
  }
  if (tid == 0) {
    if constexpr (!DIRECT)
      part_ml[pidx] = float2{mx, sm};
    else if (lse)
      lse[bh] = (mx + __log2f(sm)) * kLn2;
  }
}

// Short splits: every K and V row of the split is loaded at once (ROWS = 8
// rows of each per thread: 32 KB of K and of V per workgroup, the same for
// every D and type), so that a split costs one memory latency instead of the
// three phases above in series.  Each wave keeps its own running softmax of its rows
// and the waves meet once, in LDS.
constexpr int kDecRows = 8;
template <typename T, int D>
constexpr int dec_short_chunk() { return kDecRows * DEC_THREADS / (D / Vec16<T>::N); }

template <typename T, int D>
__global__ __launch_bounds__(DEC_THREADS) void attn_decode_short_kernel(
    const T* __restrict__ q, const T* __restrict__ K, const T* __restrict__ V, float* __restrict__ part_o,
    float2* __restrict__ part_ml, T* __restrict__ o, float* __restrict__ lse, int Lkv, int nsplit, float sl2) {
  constexpr int EPT = Vec16<T>::N, TPR = D / EPT, RPP = DEC_THREADS / TPR, R = kDecRows;
  constexpr int NW = DEC_THREADS / 64;
  __shared__ __align__(16) float s_acc[NW][D];
  __shared__ float s_m[NW], s_l[NW];
  const int split = blockIdx.x % nsplit;
  const int64_t bh = blockIdx.x / nsplit;
  const int tid = threadIdx.x, col = tid % TPR, rsub = tid / TPR, w = tid >> 6;
  const int kbeg = split * (R * RPP), n = min(R * RPP, Lkv - kbeg);
  const T* Kh = K + (bh * Lkv + kbeg) * D + col * EPT;
  const T* Vh = V + (bh * Lkv + kbeg) * D + col * EPT;
  const uint4 qx = ldg16(q + bh * D + col * EPT);
  uint4 kx[R], vx[R];
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int j = rsub + u * RPP;
    kx[u] = j < n ? ldg16_stream(Kh + (int64_t)j * D) : uint4{0, 0, 0, 0};
  }
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const int j = rsub + u * RPP;
    vx[u] = j < n ? ldg16_stream(Vh + (int64_t)j * D) : uint4{0, 0, 0, 0};
  }
  float qv[EPT];
  Vec16<T>::cvt(qx, qv);
#pragma unroll
  for (int e = 0; e < EPT; ++e) qv[e] *= sl2;
  float sc[R], m = -INFINITY;
#pragma unroll
  for (int u = 0; u < R; ++u) {
    float kf[EPT], dot = 0.f;
    Vec16<T>::cvt(kx[u], kf);
#pragma unroll
    for (int e = 0; e < EPT; ++e) dot += qv[e] * kf[e];
#pragma unroll
    for (int off = TPR / 2; off > 0; off >>= 1) dot += __shfl_xor(dot, off, 64);
    sc[u] = rsub + u * RPP < n ? dot : -INFINITY;
    m = vmax(m, sc[u]);  // NaN scores propagate
  }
#pragma unroll
  for (int off = TPR; off < 64; off <<= 1) m = vmax(m, __shfl_xor(m, off, 64));
  const float mb = m == -INFINITY ? 0.f : m;  // no row (or none finite): every weight 0
  float l = 0.f, acc[EPT];
#pragma unroll
  for (int e = 0; e < EPT; ++e) acc[e] = 0.f;
#pragma unroll
  for (int u = 0; u < R; ++u) {
    const float p = fast_exp2(sc[u] - mb);
    float vf[EPT];
    Vec16<T>::cvt(vx[u], vf);
    l += p;
#pragma unroll
    for (int e = 0; e < EPT; ++e) acc[e] += p * vf[e];
  }
#pragma unroll
  for (int off = TPR; off < 64; off <<= 1) {
    l += __shfl_xor(l, off, 64);
#pragma unroll
    for (int e = 0; e < EPT; ++e) acc[e] += __shfl_xor(acc[e], off, 64);
  }
  if ((tid & 63) < TPR) {
#pragma unroll
    for (int e = 0; e < EPT; ++e) s_acc[w][col * EPT + e] = acc[e];
    if (col == 0) {
      s_m[w] = m;
      s_l[w] = l;
    }
  }
  __syncthreads();
  if (tid >= D) return;
  float M = s_m[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) M = vmax(M, s_m[i]);
  const float Mb = M == -INFINITY ? 0.f : M;
  float num = 0.f, den = 0.f;
#pragma unroll
  for (int i = 0; i < NW; ++i) {
    const float wgt = fast_exp2(s_m[i] - Mb);
    den += wgt * s_l[i];
    num += wgt * s_acc[i][tid];
  }
  const int64_t pidx = bh * nsplit + split;
  if (nsplit > 1) {
    // a split whose scores are all -inf: m = -inf, weight 0 in the merge
    part_o[pidx * D + tid] = num;
    if (tid == 0) part_ml[pidx] = float2{M, den};
    return;
  }
  const float inv = 1.f / den;
  if constexpr (sizeof(T) == 2)
    o[bh * D + tid] = f32_to_bf16(num * inv);
  else
    o[bh * D + tid] = num * inv;
  if (tid == 0 && lse) lse[bh] = (M + __log2f(den)) * kLn2;
}

// One workgroup of NT threads per (b, h) merges the nsplit partials: D / 4
// threads per partial row, 4 NT / D rows side by side, which meet in LDS.
// (One thread per column walking the splits in turn took 6 us for 17 splits
// and 40 us for 128.)  NT = 256, or max(64, D) for up to 8 splits: a decode of
// 928 heads in two splits each took 15.3 us with 256 threads a head, 14.9 with
// D.  The splits' weights come from their max and sum: taken from an LSE each,
// they carry its rounding (fp32 d = 128, 128 keys in two splits: 1.7e-7 from float64,
// 1.5e-7 in one).
template <typename T, int D, int NT>
__global__ __launch_bounds__(NT) void attn_decode_combine_kernel(const float* __restrict__ part_o,
                                                                  const float2* __restrict__ part_ml,
                                                                  T* __restrict__ o, float* __restrict__ lse,
                                                                  int nsplit) {
  constexpr int TPR = D / 4, G = NT / TPR;
  __shared__ __align__(16) float s_acc[G][D];
  __shared__ float s_w[G];
  const int64_t bh = blockIdx.x;
  const int tid = threadIdx.x, c = tid % TPR, g = tid / TPR;
  const float2* pl = part_ml + bh * nsplit;
  const float* po = part_o + bh * nsplit * D + 4 * c;
  float mx = -INFINITY;  // every wave forms the maximum by itself
  for (int s = tid & 63; s < nsplit; s += 64) mx = vmax(mx, pl[s].x);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = vmax(mx, __shfl_xor(mx, off, 64));
  float sw = 0.f;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = g; s < nsplit; s += G) {
    const float2 ml = pl[s];
    const float wgt = fast_exp2(ml.x - mx);
    sw += wgt * ml.y;
    acc += wgt * *reinterpret_cast<const f32x4*>(po + (int64_t)s * D);
  }
  *reinterpret_cast<f32x4*>(&s_acc[g][4 * c]) = acc;
  if (c == 0) s_w[g] = sw;
  __syncthreads();
  if (tid >= D) return;
  float num = 0.f, den = 0.f;
#pragma unroll
  for (int i = 0; i < G; ++i) {
    num += s_acc[i][tid];
    den += s_w[i];
  }
  const float val = num / den;
  if constexpr (sizeof(T) == 2)
    o[bh * D + tid] = f32_to_bf16(val);
  else
    o[bh * D + tid] = val;
  if (tid == 0 && lse) lse[bh] = (mx + __log2f(den)) * kLn2;
}

constexpr int64_t kDecShortBytes = int64_t(56) << 20;
// Scratch of the short splits' partials, of one size so that it is allocated
// once per stream: 4032 of them at d = 128.  The rule below makes at most
// 56 MB / 32 KB (a split's keys) and one more for each of fewer than 1792 heads.
constexpr size_t kDecShortWork = size_t(2) << 20;

template <typename T, int D>
static int launch_decode(const T* q, const T* k, const T* v, T* o, float* lse, int64_t BH, int64_t Lkv,
                         float scale, hipStream_t st) {
  // Split size: the longest split (fewer workgroups, each streaming more rows)
  // that still leaves >= 2048 workgroups, 8 per CU; else 256 keys.  At
  // B=64 H=32 Lkv=8192 (2048 heads) one split per head streams K/V at
  // 1.208 ms, against 1.232 / 1.244 / 1.259 / 1.301 ms for 4096 / 2048 /
  // 1024 / 512-key splits.
  auto splits = [&](int64_t c) { return BH * ((Lkv + c - 1) / c); };
  int chunk = 256;
  for (int c = DEC_MAX_CHUNK; c >= 512; c >>= 1)
    if (splits(c) >= 2048) {
      chunk = c;
      break;
    }
  // Short splits, which cost one memory latency, where 256-key ones would be
  // few or (bf16) the keys are small.  Measured (256-key splits / short, us, both
  // with the parallel merge): bf16 d = 128 [1,8] x 1024 11.4 / 6.6, [1,8] x 8192
  // 14.0 / 9.6, [1,32] x 4097 17.5 / 14.0 (544 workgroups), [16,32] x 300 18.4 /
  // 15.0 (39 MB of K), d = 32 [29,32] x 512 12.9 / 9.5 (30 MB); fp32 d = 128 [1,32] x
  // 4097 28.2 / 24.3 (544).  Beyond the line: bf16 d = 128 [1,8] x 32768 25.0 /
  // 27.6 (1024, 67 MB), [64,32] x 1024 160 / 175 against 1024-key splits; fp32 d = 64
  // [16,16] x 700 16.2 / 16.5 (768), d = 32 [40,16] x 500 13.5 / 14.6 (more
  // cross-lane steps per byte than bf16).  Nor where a head's last short split
  // is mostly empty (bf16 d = 32 [16,32] x 513 10.7 / 11.8; one split at most half
  // full of many heads, d = 32 1520 x 200 8.6 / 9.0, 2040 x 128 9.1 / 9.8, d = 64 2040 x
  // 128 11.1 / 11.8, but 1200 x 128 7.3 / 7.0 and 8.4 / 7.8, and d = 128 1520 x 64 9.6 /
  // 9.6), or two replace one long split, no merge, of many heads (d = 128 [30,32] x
  // 129 12.3 / 17.5).
  const int64_t kbytes = BH * Lkv * D * (int64_t)sizeof(T);
  bool is_short = chunk == 256 && (sizeof(T) == 2 ? splits(256) < 1024 || kbytes < kDecShortBytes : splits(256) < 640);
  const int64_t short_splits = (Lkv + dec_short_chunk<T, D>() - 1) / dec_short_chunk<T, D>();
  if (Lkv <= 256 && short_splits > 1 && BH >= 256) is_short = false;
  if (D < 128 && 2 * Lkv <= dec_short_chunk<T, D>() && BH >= 1300) is_short = false;
  if (short_splits > 1 && BH >= 64 && 10 * Lkv < 6 * short_splits * dec_short_chunk<T, D>()) is_short = false;
  if (Lkv < chunk) chunk = (int)((Lkv + 63) / 64 * 64);
  const int64_t long_splits = (Lkv + chunk - 1) / chunk;
  int64_t nsplit = is_short ? short_splits : long_splits;
  if (!grid_fits(BH * nsplit, DEC_THREADS)) return fail(TT_ERR_ARG, "attention decode: grid too large");
  const float sl2 = scale * kLog2e;
  void* ws = nullptr;
  std::optional<WorkspaceLease> lease;  // held until both kernels are launched
  auto partials = [&](int64_t n) { return (size_t)(BH * n) * (D + 2) * sizeof(float); };
  if (is_short && short_splits > 1 &&
      (partials(short_splits) > kDecShortWork || !lease.emplace().get_fixed(st, kWsDecodeShort, kDecShortWork, &ws))) {
    is_short = false;  // no scratch for them: long splits
    nsplit = long_splits;
  }
  if (!is_short && nsplit > 1) {
    const int rc = lease.emplace().get(st, kWsDecodePartials, partials(nsplit), &ws);
    if (rc) return rc;
  }
  const dim3 grid((unsigned)(nsplit * BH)), block(DEC_THREADS);
  if (nsplit == 1) {  // one split per head: no partials, no combine
    if (is_short)
      hipLaunchKernelGGL((attn_decode_short_kernel<T, D>), grid, block, 0, st, q, k, v, nullptr, nullptr, o, lse,
                         (int)Lkv, 1, sl2);
    else if (chunk <= DEC_SMALL_CHUNK)
      hipLaunchKernelGGL((attn_decode_split_kernel<T, D, 8, DEC_SMALL_CHUNK, true>), grid, block, 0, st, q, k, v,
                         nullptr, nullptr, o, lse, (int)Lkv, 1, chunk, sl2);
    else
      hipLaunchKernelGGL((attn_decode_split_kernel<T, D, 8, DEC_MAX_CHUNK, true>), grid, block, 0, st, q, k, v,
                         nullptr, nullptr, o, lse, (int)Lkv, 1, chunk, sl2);
    TT_LAUNCHED("attention decode launch", st);
    return ok();
  }
  float* part_o = (float*)ws;
  float2* part_ml = (float2*)(part_o + BH * nsplit * D);
  if (is_short)
    hipLaunchKernelGGL((attn_decode_short_kernel<T, D>), grid, block, 0, st, q, k, v, part_o, part_ml, nullptr,
                       nullptr, (int)Lkv, (int)nsplit, sl2);
  else if (chunk <= DEC_SMALL_CHUNK)
    hipLaunchKernelGGL((attn_decode_split_kernel<T, D, 8, DEC_SMALL_CHUNK, false>), grid, block, 0, st, q, k, v,
                       part_o, part_ml, nullptr, nullptr, (int)Lkv, (int)nsplit, chunk, sl2);
  else
    hipLaunchKernelGGL((attn_decode_split_kernel<T, D, 8, DEC_MAX_CHUNK, false>), grid, block, 0, st, q, k, v,
                       part_o, part_ml, nullptr, nullptr, (int)Lkv, (int)nsplit, chunk, sl2);
  TT_LAUNCHED("attention decode split launch", st);
  constexpr int kFew = D > 64 ? D : 64;
  if (nsplit <= 8)
    hipLaunchKernelGGL((attn_decode_combine_kernel<T, D, kFew>), dim3((unsigned)BH), dim3(kFew), 0, st, part_o,
                       part_ml, o, lse, (int)nsplit);
  else
    hipLaunchKernelGGL((attn_decode_combine_kernel<T, D, 256>), dim3((unsigned)BH), dim3(256), 0, st, part_o,
                       part_ml, o, lse, (int)nsplit);
  TT_LAUNCHED("attention decode combine launch", st);
  return ok();
}

template <typename T>
static int decode_entry(const char* fn, const T* q, const T* k, const T* v, T* o, float* lse, int64_t B,
                        int64_t H, int64_t Lkv, int64_t d, float scale, void* stream) {
  int rc = check_attn_shape(fn, B, H, 1, Lkv, d, 0);
  if (rc) return rc;
  const int64_t BH = B * H;
  if (BH == 0) return ok();
  if (!q || !k || !v || !o) return fail(TT_ERR_ARG, std::string(fn) + ": null pointer");
  const size_t qb = (size_t)(BH * d) * sizeof(T), kb = (size_t)(BH * Lkv * d) * sizeof(T);
  if ((rc = check_no_overlap(fn, {{q, qb, "q"}, {k, kb, "k"}, {v, kb, "v"}},
                             {{o, qb, "o"}, {lse, (size_t)BH * sizeof(float), "lse"}})))
    return rc;
  if ((rc = ensure_init())) return rc;
  hipStream_t st = stream_or_default(stream);
  switch (d) {
    case 32: return launch_decode<T, 32>(q, k, v, o, lse, BH, Lkv, scale, st);
    case 64: return launch_decode<T, 64>(q, k, v, o, lse, BH, Lkv, scale, st);
    case 128: return launch_decode<T, 128>(q, k, v, o, lse, BH, Lkv, scale, st);
    default: return fail(TT_ERR_UNSUPPORTED, std::string(fn) + ": unsupported head dim");
  }
}

}  // namespace tt

using namespace tt;

extern "C" int tt_attn_decode_bf16(const uint16_t* q, const uint16_t* k, const uint16_t* v, uint16_t* o,
                                   float* lse, int64_t B, int64_t H, int64_t Lkv, int64_t d, float scale,
                                   void* stream) {
  return decode_entry<u16>("tt_attn_decode_bf16", q, k, v, o, lse, B, H, Lkv, d, scale, stream);
}

extern "C" int tt_attn_decode_f32(const float* q, const float* k, const float* v, float* o, float* lse,
                                  int64_t B, int64_t H, int64_t Lkv, int64_t d, float scale, void* stream) {
  return decode_entry<float>("tt_attn_decode_f32", q, k, v, o, lse, B, H, Lkv, d, scale, stream);
}
