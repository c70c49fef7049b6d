// The 4096-element-tile MFMA product with a split contraction, shared by the GEMM
// and the convolution: for products too small for the 128-row tiles of
// gemm.hip to fill the chip.
//
//   acc[m][n] = sum over k of A(m, k) B(k, n)
//
// Workgroup = 4 waves, one 64 x 64 (or 32 x 128) tile, a 32 x 32 MFMA block per
// wave, and one of `nsplit` runs of whole BK-steps of k (blockIdx.z).  What bounds
// these products is the serial chain of k-steps of one workgroup (a global
// load, an LDS write, a barrier: about 1 us a step), not bandwidth or MFMA
// rate, so the contraction is cut until about two workgroups per CU exist.
// With one split the epilogue runs here; with several, each writes its fp32
// sums to `part` [nsplit][M][N] and k_split_reduce adds them in split order
// (a fixed order: results do not depend on timing).
//
// A and B are read through sources that give one 16-byte chunk of T at a
// time, zero outside the matrix:
//   kKC  = true:  chunk(at(row), k) = elements (row, k .. k + EPC - 1)
//   kKC  = false: chunk(at(row), k) = elements (row .. row + EPC - 1, k)
// so a source can be a stored matrix of either orientation or a gather.  A
// thread's rows are the same in every k-step, so at(row), what a source works
// out from the row alone, is computed once.  chunk returns the loads' raw
// registers and pack makes the 16 bytes of them only where the tile is
// written to LDS, after the step's MFMAs: nothing waits for a load in between.
// A phased product (SB::kPhased) is several products in one launch: enter(z)
// of the sources and the epilogue sets them up for product z, whose N and K
// are then B.Q and B.K (M is common).  blockIdx.z = phase * nsplit + split.
// Its epilogue returns whether an output has to be formed again, which
// again(m, n) does (rare, so that one loop behind the stores is enough).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <optional>
#include <string>

#include "attn_common.h"
#include "tt_internal.h"

namespace tt {

// Tile rows TM: 64 (64 x 64, waves 2 x 2) or 32 (32 x 128, waves side by
// side) for products of at most 32 rows.  (A 128 x 128 variant for large
// gathered products measured slower at every convolution size tried.)
constexpr int split_tile_cols(int tm) { return 4096 / tm; }

template <typename T>
struct SplitT;
template <>
struct SplitT<float> {
  static constexpr int BK = 32, EPC = 4;
  // k-contiguous tiles: 144-byte rows, so that 16 lanes' 16-byte operand
  // reads fall on distinct banks; row-contiguous tiles: 72-float k-rows, so
  // that the lane halves (4 k apart) read disjoint banks.
  static constexpr int PAD_K = 4, PAD_R = 8;
};
template <>
struct SplitT<u16> {
  static constexpr int BK = 64, EPC = 8;
  // k-contiguous tiles are swizzled (SplitTile::at), row-contiguous ones take
  // 192-byte k-rows: the 4 k-rows x 2 column halves of a transpose read cover
  // the 64 banks once.
  static constexpr int PAD_K = 0, PAD_R = 32;
};

typedef unsigned split_u32x4 __attribute__((ext_vector_type(4)));
// 16 bytes at any element alignment (the target reads unaligned global words)
typedef split_u32x4 split_u32x4_any __attribute__((aligned(2)));

// One operand tile: R rows x BK k-values.
template <typename T, bool KC, int R, class Raw = split_u32x4>
struct SplitTile {
  using S = SplitT<T>;
  static constexpr int BK = S::BK, EPC = S::EPC;
  static constexpr int CH = R * BK / EPC / 256;  // 16-byte chunks per thread
  static_assert(R * BK % (EPC * 256) == 0, "tile must split into whole chunks");
  static constexpr int LD = KC ? BK + S::PAD_K : R + S::PAD_R;
  static constexpr int ELEMS = KC ? R * LD : BK * LD;
  static constexpr int PER = (KC ? BK : R) / EPC;  // chunks per stored row
  static constexpr int ROWS = KC ? CH : 1;         // rows per thread
  static_assert(KC || 256 % PER == 0, "one row chunk per thread");

  Raw reg[CH];

  // element offset of chunk c of tile row r (KC)
  __device__ static __forceinline__ int at(int r, int c) {
    if constexpr (sizeof(T) == 2) return r * LD + ((c ^ ((r >> 1) & 7)) * EPC);
    return r * LD + c * EPC;
  }
  template <class Src>
  struct Rows {
    typename Src::At at[ROWS];
    __device__ __forceinline__ Rows(const Src& src, int r0) {
#pragma unroll
      for (int c = 0; c < ROWS; ++c) {
        const int id = (int)threadIdx.x + 256 * c;
        at[c] = src.at(r0 + (KC ? id / PER : (id % PER) * EPC));
      }
    }
  };
  template <class Src>
  __device__ __forceinline__ void load(const Src& src, const Rows<Src>& rows, int k0) {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int id = (int)threadIdx.x + 256 * c;
      reg[c] = src.chunk(rows.at[KC ? c : 0], k0 + (KC ? (id % PER) * EPC : id / PER));
    }
  }
  template <class Src>
  __device__ __forceinline__ void store(const Src& src, T* s) const {
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int id = (int)threadIdx.x + 256 * c, a = id / PER, b = id % PER;
      *reinterpret_cast<split_u32x4*>(&s[KC ? at(a, b) : a * LD + b * EPC]) = src.pack(reg[c]);
    }
  }
};

// Operand of the 32 rows at rbase for one group of k-values.  fp32: group j
// holds k = 8 j + 4 (l / 32) + e, e = 0..3, the contraction indices of four
// MFMAs; bf16: k = 16 j + 8 (l / 32) + e, e = 0..7, one MFMA.
template <bool KC, int R>
__device__ __forceinline__ f32x4 split_operand(const float* s, int rbase, int j) {
  using Tile = SplitTile<float, KC, R>;
  const int l = threadIdx.x & 63, r = rbase + (l & 31), c = 2 * j + (l >> 5);
  if constexpr (KC) {
    return *reinterpret_cast<const f32x4*>(&s[Tile::at(r, c)]);
  } else {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = s[(4 * c + e) * Tile::LD + r];
    return v;
  }
}
template <bool KC, int R>
__device__ __forceinline__ bf16x8 split_operand(const u16* s, int rbase, int j) {
  using Tile = SplitTile<u16, KC, R>;
  const int l = threadIdx.x & 63;
  if constexpr (KC) {
    return *reinterpret_cast<const bf16x8*>(&s[Tile::at(rbase + (l & 31), 2 * j + (l >> 5))]);
  } else {
    const int G = l >> 4, sl = l & 15;
    const int kr = 16 * j + 8 * (G >> 1) + (sl >> 2);
    const int col = rbase + 16 * (G & 1) + 4 * (sl & 3);
    return lds_read_tr16x2(&s[kr * Tile::LD + col], &s[(kr + 4) * Tile::LD + col]);
  }
}

// A row-major matrix as a source: rows of the tile x k.  KC: stored [row][k];
// else stored [k][row].
template <typename T, bool KC>
struct MatrixSource {
  static constexpr bool kKC = KC, kPhased = false;
  const T* p;
  int64_t ld;
  int rows, K;
  using Raw = split_u32x4;
  struct At {
    int row;
  };
  __device__ __forceinline__ At at(int row) const { return At{row}; }
  __device__ __forceinline__ split_u32x4 pack(const Raw& r) const { return r; }
  __device__ __forceinline__ Raw chunk(const At& at, int k) const {
    constexpr int EPC = SplitT<T>::EPC;
    const int a = KC ? at.row : k, b = KC ? k : at.row;  // stored row, first stored column
    const int na = KC ? rows : K, nb = KC ? K : rows;
    const T* q = p + (int64_t)a * ld + b;
    if (a < na && b + EPC <= nb) return *reinterpret_cast<const split_u32x4_any*>(q);
    T v[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e) v[e] = (a < na && b + e < nb) ? q[e] : T(0);
    return __builtin_bit_cast(split_u32x4, v);
  }
};

__device__ __forceinline__ void split_store(float* p, float v) { *p = v; }
__device__ __forceinline__ void split_store(u16* p, float v) { *p = f32_to_bf16(v); }
__device__ __forceinline__ float split_load(const float* p) { return *p; }
__device__ __forceinline__ float split_load(const u16* p) { return bf16_to_f32(*p); }

// C = alpha acc + bias + beta C, C row-major [M][N]; bias[n * bias_step]
// (null: none).  beta = 0 does not read C.
template <typename T>
struct MatrixEpilogue {
  T* C;
  const T* bias;
  int64_t bias_step;
  float alpha, beta;
  int N;
  __device__ __forceinline__ void operator()(int m, int n, float acc) const {
    T* p = C + (int64_t)m * N + n;
    float v = alpha * acc;
    if (bias) v += split_load(bias + n * bias_step);
    if (beta != 0.f) v += beta * split_load(p);
    split_store(p, v);
  }
};

template <typename T, int TM, class SA, class SB, class EP>
__global__ __launch_bounds__(256) void k_split_gemm(int M, int N, int K, int nsplit, SA A, SB B, EP ep,
                                                    float* __restrict__ part) {
  constexpr int BK = SplitT<T>::BK, GROUPS = sizeof(T) == 2 ? BK / 16 : BK / 8;
  constexpr int TN = split_tile_cols(TM);
  using TileA = SplitTile<T, SA::kKC, TM, typename SA::Raw>;
  using TileB = SplitTile<T, SB::kKC, TN, typename SB::Raw>;
  __shared__ __align__(16) T sA[2][TileA::ELEMS];
  __shared__ __align__(16) T sB[2][TileB::ELEMS];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  const int m0 = blockIdx.y * TM, n0 = blockIdx.x * TN;
  const int wm = TM == 32 ? 0 : 32 * (w >> 1), wn = TM == 32 ? 32 * w : 32 * (w & 1);
  int split = blockIdx.z;
  if (part) part += (int64_t)blockIdx.z * M * N;
  const int pitch = N;  // of a row of partial sums: the columns of the largest phase
  if constexpr (SB::kPhased) {
    const int phase = blockIdx.z / nsplit;
    split = blockIdx.z - phase * nsplit;
    A.enter(phase);
    B.enter(phase);
    N = B.Q;
    K = B.K;
    if (n0 >= N) return;  // uniform: the grid covers the largest phase
  }
  const int kper = ((K + BK - 1) / BK + nsplit - 1) / nsplit * BK;  // whole steps; a late split may be empty
  const int kbeg = min(K, split * kper), kend = min(K, kbeg + kper);
  f32x16 acc = f32x16{};
  TileA ta;
  TileB tb;
  const typename TileA::template Rows<SA> ra(A, m0);
  const typename TileB::template Rows<SB> rb(B, n0);
  if (kbeg < kend) {
    ta.load(A, ra, kbeg);
    tb.load(B, rb, kbeg);
    ta.store(A, sA[0]);
    tb.store(B, sB[0]);
  }
  __syncthreads();
  for (int k0 = kbeg, cur = 0; k0 < kend; k0 += BK, cur ^= 1) {
    const bool more = k0 + BK < kend;
    if (more) {  // the next step's chunks in flight during this step's MFMAs
      ta.load(A, ra, k0 + BK);
      tb.load(B, rb, k0 + BK);
    }
#pragma unroll
    for (int j = 0; j < GROUPS; ++j) {
      const auto a = split_operand<SA::kKC, TM>(sA[cur], wm, j);
      const auto b = split_operand<SB::kKC, TN>(sB[cur], wn, j);
      if constexpr (sizeof(T) == 2) {
        acc = mfma_bf16_32x32x16(a, b, acc);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = mfma_f32_32x32x2(a[e], b[e], acc);
      }
    }
    if (more) {
      ta.store(A, sA[cur ^ 1]);
      tb.store(B, sB[cur ^ 1]);
    }
    __syncthreads();
  }
  const int n = n0 + wn + (l & 31);
  if (n >= N) return;
  if constexpr (SB::kPhased) ep.enter(blockIdx.z / nsplit);  // here: its values need no registers during the loop
  unsigned again = 0;  // bit r: output r
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + wm + acc_row(r, l >> 5);
    if (m >= M) continue;
    if (part)
      part[(int64_t)m * pitch + n] = acc[r];
    else if constexpr (SB::kPhased)
      again |= (unsigned)ep(m, n, acc[r]) << r;
    else
      ep(m, n, acc[r]);
  }
  if constexpr (SB::kPhased)
    for (; again; again &= again - 1) ep.again(m0 + wm + acc_row(__ffs(again) - 1, l >> 5), n);
}

// Adds the splits' sums in a fixed order and runs the epilogue, phase by
// blockIdx.y.  64 outputs per wave; G waves of the workgroup take the splits
// w, w + G, ... of the same outputs and meet in LDS, 4 / G (G < 4) groups of
// outputs per workgroup.  Columns past a phase's own (PHASED) are skipped.
template <int G, bool PHASED, class EP>
__global__ __launch_bounds__(64 * (G < 4 ? 4 : G)) void k_split_reduce(const float* __restrict__ part, int M, int N,
                                                                       int nsplit, EP ep) {
  constexpr int W = G < 4 ? 4 : G, OUT = 64 * (W / G);  // waves and outputs per workgroup
  __shared__ float red[W][64];
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63, g = w % G;
  const int64_t total = (int64_t)M * N, i = (int64_t)blockIdx.x * OUT + 64 * (w / G) + l;
  const int m = (int)(i / N), n = (int)(i - (int64_t)m * N);
  int cols = N;
  if constexpr (PHASED) {
    ep.enter(blockIdx.y);
    cols = ep.columns();
    part += blockIdx.y * nsplit * total;
  }
  const bool in = i < total && n < cols;
  float s = 0.f;
  if (in) {
#pragma unroll 8
    for (int z = g; z < nsplit; z += G) s += part[z * total + i];
  }
  if constexpr (G > 1) {
    red[w][l] = s;
    __syncthreads();
    if (g != 0) return;
#pragma unroll
    for (int k = 1; k < G; ++k) s += red[w + k][l];
  }
  if (!in) return;
  if constexpr (PHASED) {
    if (ep(m, n, s)) ep.again(m, n);
  } else {
    ep(m, n, s);
  }
}

// Splits of the contraction for a grid of `tiles` tiles and nk BK-steps: to
// the nearest, two workgroups per CU in all, each with at least two steps.  (Three
// or four per CU: bf16 1536^3 22 -> 31 us, fp32 1500^3 106 -> 93 us, most sizes
// within 5 %; rounded down, fp32 900 x 1100 x 2000, 270 tiles, 76 -> 110 us;
// rounded up, bf16 300 x 5000 x 600, 395 tiles, 16.8 -> 18.6.)
inline int split_count(int64_t tiles, int64_t nk) {
  int64_t s = (512 + tiles / 2) / (tiles > 0 ? tiles : 1);
  if (s > nk / 2) s = nk / 2;
  if (s > 256) s = 256;
  return s < 1 ? 1 : (int)s;
}

// Rows that a launch takes: the grid's y extent is 16 bits.  (Splits and phases
// share z: with more than one split there are fewer than 768 of both.)
constexpr int64_t split_max_rows(int tm) { return int64_t(65535) * tm; }

// Scratch of one split product: nsplit x M x N floats, at most
// kSplitWorkBytes (with more than one split, nsplit x tiles is below 768; a
// tile is 16 KB).  One fixed size per stream, so the buffer is allocated once.
constexpr size_t kSplitWorkBytes = size_t(12) << 20;

// Launches the product on s: N columns and K contraction values (of the
// largest phase), `phases` phases (1 unless SB::kPhased).  Without scratch (a
// refused allocation, or a stream under capture, where nothing may be
// allocated and a captured address must not outlive the buffer) the
// contraction is not split.
template <typename T, int TM, class SA, class SB, class EP>
int launch_split_tiles(const char* fn, int64_t M, int64_t N, int64_t K, int phases, const SA& A, const SB& B,
                       const EP& ep, hipStream_t s) {
  constexpr int BK = SplitT<T>::BK, TN = split_tile_cols(TM);
  const int64_t gx = (N + TN - 1) / TN, gy = (M + TM - 1) / TM;
  const int64_t nk = (K + BK - 1) / BK;
  int nsplit = split_count(gx * gy * phases, nk);
  if (!grid_fits(gx, 256) || M > split_max_rows(TM) || (int64_t)phases * nsplit > 65535)
    return fail(TT_ERR_ARG, std::string(fn) + ": too large");
  float* part = nullptr;
  std::optional<WorkspaceLease> ws;  // held until the reduction is queued
  if (nsplit > 1 && !ws.emplace().get_optional(s, kWsGemmSplits, kSplitWorkBytes, (void**)&part)) nsplit = 1;
  hipLaunchKernelGGL((k_split_gemm<T, TM, SA, SB, EP>), dim3((unsigned)gx, (unsigned)gy, (unsigned)(phases * nsplit)),
                     dim3(256), 0, s, (int)M, (int)N, (int)K, nsplit, A, B, ep, part);
  TT_LAUNCHED(fn, s);
  if (nsplit > 1) {
    const int64_t waves = (M * N + 63) / 64;
    const float* p = part;
    constexpr bool PH = SB::kPhased;
    if (nsplit >= 64)
      hipLaunchKernelGGL((k_split_reduce<16, PH, EP>), dim3((unsigned)waves, (unsigned)phases), dim3(1024), 0, s, p,
                         (int)M, (int)N, nsplit, ep);
    else if (nsplit >= 16)
      hipLaunchKernelGGL((k_split_reduce<4, PH, EP>), dim3((unsigned)waves, (unsigned)phases), dim3(256), 0, s, p,
                         (int)M, (int)N, nsplit, ep);
    else
      hipLaunchKernelGGL((k_split_reduce<1, PH, EP>), dim3((unsigned)((waves + 3) / 4), (unsigned)phases), dim3(256),
                         0, s, p, (int)M, (int)N, nsplit, ep);
    TT_LAUNCHED(fn, s);
  }
  return ok();
}
template <typename T, class SA, class SB, class EP>
int launch_split_gemm(const char* fn, int64_t M, int64_t N, int64_t K, const SA& A, const SB& B, const EP& ep,
                      hipStream_t s, int phases = 1) {
  if (M <= 32) return launch_split_tiles<T, 32>(fn, M, N, K, phases, A, B, ep, s);
  return launch_split_tiles<T, 64>(fn, M, N, K, phases, A, B, ep, s);
}

}  // namespace tt
