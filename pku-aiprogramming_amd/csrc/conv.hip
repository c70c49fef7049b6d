// The convolution: its products, which gather their operands from the images
// (tt_conv_forward / tt_conv_backward, reference src/Layers.cu:160-252), the
// column matrix on its own (im2col / col2im, src/Layers.cu:81-158, kernels
// src/Layers_kernels.cu:32-105) and max pooling.
//
// Layout (the reference's): an image batch im[N][C][H][W] and its column
// matrix col[N][P][C][kh][kw], P = OH * OW output pixels in row-major order,
//   col[n][oy * OW + ox][c][ky][kx] = im[n][c][oy sh - ph + ky][ox sw - pw + kx]
// (0 outside the image), OH = (H + 2 ph - kh) / sh + 1, OW likewise.  col2im
// is its adjoint: every image element is the sum of the column entries that
// read it.  Both kernels gather (one thread per output element, a fixed
// order of the sums, no atomics), the whole batch in one launch.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "gemm_split.h"
#include "tt_internal.h"

namespace tt {

namespace {

struct ConvGeom {
  int C, H, W, kh, kw, ph, pw, sh, sw, oh, ow;
};

__device__ __forceinline__ float to_f(float x) { return x; }
__device__ __forceinline__ float to_f(uint16_t b) { return __uint_as_float(uint32_t(b) << 16); }
__device__ __forceinline__ void from_f(float v, float& out) { out = v; }
__device__ __forceinline__ void from_f(float v, uint16_t& out) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7fffffffu) > 0x7f800000u) {
    out = uint16_t((u >> 16) | 0x40);  // quiet NaN
    return;
  }
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  out = uint16_t(u >> 16);
}

// One thread per column entry (n, p, c, ky, kx), in the column's order, so
// that consecutive threads write consecutive elements.
template <typename T>
__global__ __launch_bounds__(256) void k_im2col(const T* __restrict__ im, T* __restrict__ col, int64_t total,
                                                ConvGeom g) {
  const int64_t P = (int64_t)g.oh * g.ow;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    int64_t r = i;
    const int kx = (int)(r % g.kw);
    r /= g.kw;
    const int ky = (int)(r % g.kh);
    r /= g.kh;
    const int c = (int)(r % g.C);
    r /= g.C;
    const int64_t p = r % P, n = r / P;
    const int oy = (int)(p / g.ow), ox = (int)(p % g.ow);
    const int y = oy * g.sh - g.ph + ky, x = ox * g.sw - g.pw + kx;
    T v = T(0);
    if (y >= 0 && y < g.H && x >= 0 && x < g.W) v = im[((n * g.C + c) * g.H + y) * g.W + x];
    col[i] = v;
  }
}

// One thread per image element (n, c, y, x): the sum, in float, of the column
// entries (oy, ox, ky, kx) with oy sh - ph + ky = y and ox sw - pw + kx = x,
// ky and kx ascending.
template <typename T>
__global__ __launch_bounds__(256) void k_col2im(const T* __restrict__ col, T* __restrict__ im, int64_t total,
                                                ConvGeom g) {
  const int64_t K = (int64_t)g.C * g.kh * g.kw;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    int64_t r = i;
    const int x = (int)(r % g.W);
    r /= g.W;
    const int y = (int)(r % g.H);
    r /= g.H;
    const int c = (int)(r % g.C);
    const int64_t n = r / g.C;
    const T* cn = col + n * (int64_t)g.oh * g.ow * K + (int64_t)c * g.kh * g.kw;
    float s = 0.f;
    for (int ky = 0; ky < g.kh; ++ky) {
      const int ty = y + g.ph - ky;
      if (ty < 0 || ty % g.sh != 0) continue;
      const int oy = ty / g.sh;
      if (oy >= g.oh) continue;
      for (int kx = 0; kx < g.kw; ++kx) {
        const int tx = x + g.pw - kx;
        if (tx < 0 || tx % g.sw != 0) continue;
        const int ox = tx / g.sw;
        if (ox >= g.ow) continue;
        s += to_f(cn[((int64_t)oy * g.ow + ox) * K + ky * g.kw + kx]);
      }
    }
    from_f(s, im[i]);
  }
}

// Max pooling (reference src/Layers.cu:254-322, kernels
// src/Layers_kernels.cu:109-175): one thread per output element; the window
// is clipped to the image (padding never wins), the first largest entry in
// row-major order is kept, and mask holds its index y * W + x in the (n, c)
// plane as a float (-1, and -FLT_MAX out, for a window with no image element).
__global__ __launch_bounds__(256) void k_maxpool(const float* __restrict__ in, float* __restrict__ out,
                                                 float* __restrict__ mask, int64_t total, ConvGeom g) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int ox = (int)(i % g.ow), oy = (int)((i / g.ow) % g.oh);
    const int64_t plane = i / ((int64_t)g.oh * g.ow);
    const int y0 = oy * g.sh - g.ph, x0 = ox * g.sw - g.pw;
    const int y1 = min(y0 + g.kh, g.H), x1 = min(x0 + g.kw, g.W);
    const float* pl = in + plane * g.H * g.W;
    float best = -3.402823466e38f;
    int arg = -1;
    for (int y = max(y0, 0); y < y1; ++y)
      for (int x = max(x0, 0); x < x1; ++x)
        if (pl[y * g.W + x] > best) {
          best = pl[y * g.W + x];
          arg = y * g.W + x;
        }
    out[i] = best;
    mask[i] = (float)arg;
  }
}

// Its gradient, one thread per input element: the sum of grad_out over the
// windows whose mask points at this element (the reference assigns instead,
// which with overlapping windows keeps one of them, whichever thread writes
// last; with non-overlapping windows the two agree).
__global__ __launch_bounds__(256) void k_maxpool_backward(const float* __restrict__ gout,
                                                          const float* __restrict__ mask,
                                                          float* __restrict__ gin, int64_t total, ConvGeom g) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int x = (int)(i % g.W), y = (int)((i / g.W) % g.H);
    const int64_t plane = i / ((int64_t)g.H * g.W);
    const float* gp = gout + plane * g.oh * g.ow;
    const float* mp = mask + plane * g.oh * g.ow;
    const float self = (float)(y * g.W + x);
    float s = 0.f;
    for (int ky = 0; ky < g.kh; ++ky) {
      const int ty = y + g.ph - ky;
      if (ty < 0 || ty % g.sh != 0 || ty / g.sh >= g.oh) continue;
      for (int kx = 0; kx < g.kw; ++kx) {
        const int tx = x + g.pw - kx;
        if (tx < 0 || tx % g.sw != 0 || tx / g.sw >= g.ow) continue;
        const int o = (ty / g.sh) * g.ow + tx / g.sw;
        if (mp[o] == self) s += gp[o];
      }
    }
    gin[i] = s;
  }
}

int conv_geom(const char* fn, int64_t N, int C, int H, int W, int kh, int kw, int ph, int pw, int sh, int sw,
              ConvGeom& g) {
  if (N < 0 || C < 1 || H < 1 || W < 1 || kh < 1 || kw < 1)
    return fail(TT_ERR_ARG, std::string(fn) + ": N >= 0 and C, H, W, kernel sizes >= 1 required");
  if (ph < 0 || pw < 0 || sh < 1 || sw < 1)
    return fail(TT_ERR_ARG, std::string(fn) + ": pads >= 0 and strides >= 1 required");
  if ((int64_t)H + 2 * (int64_t)ph < kh || (int64_t)W + 2 * (int64_t)pw < kw)
    return fail(TT_ERR_ARG, std::string(fn) + ": the kernel is larger than the padded image");
  g = ConvGeom{C, H, W, kh, kw, ph, pw, sh, sw, (int)((H + 2 * (int64_t)ph - kh) / sh + 1),
               (int)((W + 2 * (int64_t)pw - kw) / sw + 1)};
  return TT_OK;
}

template <typename T, bool TO_COL>
int conv_move(const char* fn, const void* src, void* dst, int64_t N, const ConvGeom& g, void* stream) {
  const int64_t total = TO_COL ? N * g.oh * g.ow * (int64_t)g.C * g.kh * g.kw : N * (int64_t)g.C * g.H * g.W;
  if (total == 0) return ok();
  if (!src || !dst) return fail(TT_ERR_ARG, std::string(fn) + ": null pointer");
  int rc = ensure_init();
  if (rc) return rc;
  hipStream_t s = stream_or_default(stream);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;  // grid-stride beyond
  if (TO_COL)
    hipLaunchKernelGGL(k_im2col<T>, dim3((unsigned)blocks), dim3(256), 0, s, (const T*)src, (T*)dst, total, g);
  else
    hipLaunchKernelGGL(k_col2im<T>, dim3((unsigned)blocks), dim3(256), 0, s, (const T*)src, (T*)dst, total, g);
  TT_LAUNCHED(fn, s);
  return ok();
}

template <bool TO_COL>
int conv_entry(const char* fn, int dtype, const void* src, void* dst, int64_t N, int C, int H, int W, int kh,
               int kw, int ph, int pw, int sh, int sw, void* stream) {
  ConvGeom g;
  int rc = conv_geom(fn, N, C, H, W, kh, kw, ph, pw, sh, sw, g);
  if (rc) return rc;
  if (dtype == TT_F32) return conv_move<float, TO_COL>(fn, src, dst, N, g, stream);
  if (dtype == TT_BF16) return conv_move<uint16_t, TO_COL>(fn, src, dst, N, g, stream);
  return fail(TT_ERR_ARG, std::string(fn) + ": dtype must be TT_F32 or TT_BF16");
}

// ---------------------------------------------------------------- the convolution products
// The convolution's three products as split-k MFMA products (gemm_split.h)
// whose operands are gathered from the image, so that no column matrix is
// written:
//   forward  out[co, q]  = sum over kk of W[co, kk] X(kk, q)     q = (n, oy, ox), kk = (c, ky, kx)
//   dW       gW[co, kk]  = sum over q of  gO[co, q] X(kk, q)
//   dX       gX[c, p]    = sum over (co, ky, kx) of W[co, c, ky, kx] gO(co, ky, kx, p)   p = (n, y, x)
// with X(kk, q) the image element under kernel position kk of output pixel q
// and gO(.., p) the output gradient that position reads p from (zero where
// there is none).  One launch covers the whole batch.
//
// They replace im2col, one GEMM per image and col2im: at small images the
// launches dominated (a product per image at 5-76 us each), at large ones the
// dW product, one or a few tiles walking every pixel.  Forward / backward
// through myLayer, us, before -> now: 64 x 8 x 14 x 14, 16 kernels 5 x 5 fp32
// 1551 / 2214 -> 12 / 35; 64 x 64 x 56 x 56, 64 kernels 3 x 3 fp32 4121 /
// 22257 -> 208 / 512 (71 / 58 TF), bf16 1660 / 7464 -> 89 / 320; 8 x 512 x
// 28 x 28, 512 kernels 3 x 3 fp32 3477 / 1617 -> 506 / 1169; 1 x 3 x 224 x 224,
// 768 kernels 16 x 16 stride 16 fp32 85 / 122 -> 17 / 33.  What bounds them now
// is the gather's index arithmetic, about ten VALU instructions an element; the
// layer leaves its widest products to the column matrix (layers.cpp).
// n / d for 0 <= n < 2^31 by a multiplication (Granlund and Montgomery's
// round-up method).
struct FastDiv {
  uint32_t d, mul, shift;
  FastDiv() = default;
  __host__ __device__ explicit FastDiv(uint32_t d_) : d(d_) {
    shift = 0;
    while ((uint64_t(1) << shift) < d) ++shift;
    mul = (uint32_t)(((uint64_t(1) << 32) * ((uint64_t(1) << shift) - d)) / d + 1);
  }
  __device__ __forceinline__ int div(int n) const { return (int)((__umulhi(mul, (uint32_t)n) + (uint32_t)n) >> shift); }
  __device__ __forceinline__ int divmod(int n, int& rem) const {
    const int q = div(n);
    rem = n - q * (int)d;
    return q;
  }
};

struct ConvDivs {
  FastDiv kk, kw, P, ow;  // kh * kw, kw, oh * ow, ow
};

// Gathers.  Every operand is im[base(v) + off(t)] for a vector position v (a
// pixel, whose EPC neighbours make one chunk) and a tap t (a kernel position
// or channel), zero unless the tap's step from the position stays inside the
// image: 0 <= y(v) + dy(t) < ylim and 0 <= x(v) + dx(t) < xlim.  The chunk's
// elements are loaded one by one without branches (element 0 where there is
// none, replaced by zero in pack): with branches around the loads (one 16-byte
// load inside an image row, predicated ones across its edge) each chunk waited
// for its own loads, 5-10 us a k-step.
struct Tap {
  int off, dy, dx;
};
template <int N>
struct Positions {
  int base[N], y[N], x[N];
};
constexpr int kOutside = -(1 << 30);  // a y or dy that no step brings inside

// a b + c for offsets of elements that may not exist
__device__ __forceinline__ int wrap_mad(int a, int b, int c) {
  return (int)((unsigned)a * (unsigned)b + (unsigned)c);
}

// Src: Positions<EPC> positions(v), Tap tap(t), data(), ylim(), xlim().
// kKC = true: v = k and t = row; false: v = row and t = k.
template <typename T, bool KC, class Src>
struct Gather {
  static constexpr bool kKC = KC;
  static constexpr int EPC = SplitT<T>::EPC;
  struct Raw {
    T v[EPC];
    bool in[EPC];
  };
  using At = std::conditional_t<KC, Tap, Positions<EPC>>;
  __device__ __forceinline__ const Src& self() const { return static_cast<const Src&>(*this); }
  __device__ __forceinline__ At at(int row) const {
    if constexpr (KC)
      return self().tap(row);
    else
      return self().positions(row);
  }
  __device__ __forceinline__ Raw chunk(const At& at, int k) const {
    if constexpr (KC)
      return load(self().positions(k), at);
    else
      return load(at, self().tap(k));
  }
  __device__ __forceinline__ Raw load(const Positions<EPC>& p, const Tap& t) const {
    Raw r;
#pragma unroll
    for (int e = 0; e < EPC; ++e) {
      r.in[e] = ((unsigned)(p.y[e] + t.dy) < (unsigned)self().ylim()) &
                ((unsigned)(p.x[e] + t.dx) < (unsigned)self().xlim());
      r.v[e] = self().data()[r.in[e] ? p.base[e] + t.off : 0];
    }
    return r;
  }
  __device__ __forceinline__ split_u32x4 pack(const Raw& r) const {
    T v[EPC];
#pragma unroll
    for (int e = 0; e < EPC; ++e) v[e] = r.in[e] ? r.v[e] : T(0);
    return __builtin_bit_cast(split_u32x4, v);
  }
};

// X(kk, q): v = output pixel q (its window's first row and column), t = kk.
template <typename T, bool KC>
struct ColumnSource : Gather<T, KC, ColumnSource<T, KC>> {
  static constexpr bool kPhased = false;
  const T* im;
  ConvGeom g;
  ConvDivs dv;
  int K, Q;
  ColumnSource(const T* im_, const ConvGeom& g_, const ConvDivs& dv_, int K_, int Q_)
      : im(im_), g(g_), dv(dv_), K(K_), Q(Q_) {}
  __device__ __forceinline__ const T* data() const { return im; }
  __device__ __forceinline__ int ylim() const { return g.H; }
  __device__ __forceinline__ int xlim() const { return g.W; }
  __device__ __forceinline__ Positions<SplitT<T>::EPC> positions(int q) const {
    Positions<SplitT<T>::EPC> r;
#pragma unroll
    for (int e = 0; e < SplitT<T>::EPC; ++e) {
      int p, ox;
      const int n = dv.P.divmod(q + e, p), oy = dv.ow.divmod(p, ox);
      r.y[e] = q + e < Q ? oy * g.sh - g.ph : kOutside;
      r.x[e] = ox * g.sw - g.pw;
      r.base[e] = wrap_mad(wrap_mad(n, g.C * g.H, r.y[e]), g.W, r.x[e]);
    }
    return r;
  }
  __device__ __forceinline__ Tap tap(int kk) const {
    int r, kx;
    const int c = dv.kk.divmod(kk, r), ky = dv.kw.divmod(r, kx);
    return Tap{wrap_mad(wrap_mad(c, g.H, ky), g.W, kx), kk < K ? ky : kOutside, kx};
  }
};

// gO[co, q] of the [N][Cout][P] output gradient: v = q, t = co.
template <typename T, bool KC>
struct GradRowSource : Gather<T, KC, GradRowSource<T, KC>> {
  static constexpr bool kPhased = false;
  const T* go;
  FastDiv P;
  int cout, Q;
  GradRowSource(const T* go_, const FastDiv& P_, int cout_, int Q_) : go(go_), P(P_), cout(cout_), Q(Q_) {}
  __device__ __forceinline__ const T* data() const { return go; }
  __device__ __forceinline__ int ylim() const { return 1; }
  __device__ __forceinline__ int xlim() const { return 1; }
  __device__ __forceinline__ Positions<SplitT<T>::EPC> positions(int q) const {
    Positions<SplitT<T>::EPC> r;
#pragma unroll
    for (int e = 0; e < SplitT<T>::EPC; ++e) {
      int p;
      const int n = P.divmod(q + e, p);
      r.base[e] = wrap_mad(n, cout * (int)P.d, p);
      r.y[e] = q + e < Q ? 0 : kOutside;
      r.x[e] = 0;
    }
    return r;
  }
  __device__ __forceinline__ Tap tap(int co) const { return Tap{wrap_mad(co, (int)P.d, 0), co < cout ? 0 : kOutside, 0}; }
};

// The same for planes of whole chunks (P % EPC = 0): rows co, k = q, one
// 16-byte load a chunk.
template <typename T>
struct GradPlaneSource {
  static constexpr bool kKC = true, kPhased = false;
  const T* go;
  FastDiv P;
  int cout, Q;
  struct Raw {
    split_u32x4 v;
    bool in;
  };
  struct At {
    int off;
    bool in;
  };
  __device__ __forceinline__ At at(int co) const { return At{wrap_mad(co, (int)P.d, 0), co < cout}; }
  __device__ __forceinline__ Raw chunk(const At& at, int q) const {
    int p;
    const int n = P.divmod(q, p);
    const bool in = at.in & (q < Q);
    return Raw{*reinterpret_cast<const split_u32x4_any*>(go + (in ? wrap_mad(n, cout * (int)P.d, p) + at.off : 0)), in};
  }
  __device__ __forceinline__ split_u32x4 pack(const Raw& r) const { return r.in ? r.v : split_u32x4{0, 0, 0, 0}; }
};

// dX by phases.  With strides sh x sw an image row y is only reached by the
// kernel rows ky = (y + ph) mod sh + sh i, so the pixels are taken by phase
// (y mod sh, x mod sw): within one phase the product is a stride-1 one over
// ny x nx pixels and nky x nkx taps, with no zero taps to multiply, and
//   oy = by + j - i   for pixel row y = fy + sh j and tap ky = ky0 + sh i.
// Stride 1 is the one phase (0, 0) with all taps.
struct ConvPhase {
  int fy, fx, ky0, kx0, ny, nx, nky, nkx, by, bx;
  __device__ __forceinline__ ConvPhase(const ConvGeom& g, int z, int phases_x) {
    fy = z / phases_x, fx = z - fy * phases_x;
    ky0 = (fy + g.ph) % g.sh, kx0 = (fx + g.pw) % g.sw;
    ny = (g.H - fy + g.sh - 1) / g.sh, nx = (g.W - fx + g.sw - 1) / g.sw;
    nky = ky0 < g.kh ? (g.kh - ky0 + g.sh - 1) / g.sh : 0;
    nkx = kx0 < g.kw ? (g.kw - kx0 + g.sw - 1) / g.sw : 0;
    by = (fy + g.ph - ky0) / g.sh, bx = (fx + g.pw - kx0) / g.sw;
  }
};

// W[co, c, ky, kx]: v = k = (co, i, j) over the phase's taps, t = row c.
template <typename T>
struct WeightSource : Gather<T, true, WeightSource<T>> {
  const T* w;
  ConvGeom g;
  int cout, z0, phases_x;
  FastDiv taps, nkx;  // nky * nkx, nkx (of the phase; at least 1)
  int K;
  WeightSource(const T* w_, const ConvGeom& g_, int cout_, int z0_, int phases_x_)
      : w(w_), g(g_), cout(cout_), z0(z0_), phases_x(phases_x_) {}
  __device__ __forceinline__ void enter(int z) {
    const ConvPhase f(g, z0 + z, phases_x);
    taps = FastDiv(max(1, f.nky * f.nkx)), nkx = FastDiv(max(1, f.nkx));
    K = cout * f.nky * f.nkx;
    w += (int64_t)f.ky0 * g.kw + f.kx0;
  }
  __device__ __forceinline__ const T* data() const { return w; }
  __device__ __forceinline__ int ylim() const { return 1; }
  __device__ __forceinline__ int xlim() const { return 1; }
  __device__ __forceinline__ Positions<SplitT<T>::EPC> positions(int k) const {
    Positions<SplitT<T>::EPC> r;
#pragma unroll
    for (int e = 0; e < SplitT<T>::EPC; ++e) {
      int t, j;
      const int co = taps.divmod(k + e, t), i = nkx.divmod(t, j);
      r.base[e] = wrap_mad(wrap_mad(co, g.C * g.kh, i * g.sh), g.kw, j * g.sw);
      r.y[e] = k + e < K ? 0 : kOutside;
      r.x[e] = 0;
    }
    return r;
  }
  __device__ __forceinline__ Tap tap(int c) const { return Tap{wrap_mad(c, g.kh * g.kw, 0), c < g.C ? 0 : kOutside, 0}; }
};

// gO(co, i, j, p): v = row p = (n, pixel of the phase), t = k = (co, i, j).
template <typename T>
struct GradImageSource : Gather<T, false, GradImageSource<T>> {
  static constexpr bool kPhased = true;
  const T* go;
  ConvGeom g;
  int cout, images, z0, phases_x;
  FastDiv taps, nkx, pix, nx;  // nky * nkx, nkx, ny * nx, nx
  int by, bx, K, Q;
  GradImageSource(const T* go_, const ConvGeom& g_, int cout_, int images_, int z0_, int phases_x_)
      : go(go_), g(g_), cout(cout_), images(images_), z0(z0_), phases_x(phases_x_) {}
  __device__ __forceinline__ void enter(int z) {
    const ConvPhase f(g, z0 + z, phases_x);
    taps = FastDiv(max(1, f.nky * f.nkx)), nkx = FastDiv(max(1, f.nkx));
    pix = FastDiv(f.ny * f.nx), nx = FastDiv(f.nx);
    by = f.by, bx = f.bx;
    K = cout * f.nky * f.nkx;
    Q = images * f.ny * f.nx;
  }
  __device__ __forceinline__ const T* data() const { return go; }
  __device__ __forceinline__ int ylim() const { return g.oh; }
  __device__ __forceinline__ int xlim() const { return g.ow; }
  __device__ __forceinline__ Positions<SplitT<T>::EPC> positions(int row) const {
    Positions<SplitT<T>::EPC> r;
#pragma unroll
    for (int e = 0; e < SplitT<T>::EPC; ++e) {
      int p, x;
      const int n = pix.divmod(row + e, p), y = nx.divmod(p, x);
      r.y[e] = row + e < Q ? by + y : kOutside;
      r.x[e] = bx + x;
      r.base[e] = wrap_mad(wrap_mad(n, cout * g.oh, by + y), g.ow, bx + x);
    }
    return r;
  }
  __device__ __forceinline__ Tap tap(int k) const {
    int r, j;
    const int co = taps.divmod(k, r), i = nkx.divmod(r, j);
    return Tap{wrap_mad(wrap_mad(co, g.oh, -i), g.ow, -j), k < K ? -i : kOutside, -j};
  }
};

// The image gradient multiplies the weights of taps that have no output pixel
// (at the image's border) by zero, which gives NaN where such a weight is
// infinite or NaN.  A sum that came out as NaN is formed again by this function
// from the other taps alone: channel c at (py, px) of the padded image, of the
// image's output gradient go; false (and no sum) where no tap is missing.  Not
// inlined: that cost the bf16 products 3-6 % (scalar registers of the k loop).
template <typename T>
__device__ __attribute__((noinline)) bool conv_dx_present(const T* w, const T* go, ConvGeom g, int cout, int c, int py,
                                                          int px, float& sum) {
  const int ky0 = py % g.sh, oy0 = py / g.sh, kx0 = px % g.sw, ox0 = px / g.sw;  // tap ky0 + sh i reads row oy0 - i
  const int nky = (g.kh - ky0 + g.sh - 1) / g.sh, nkx = (g.kw - kx0 + g.sw - 1) / g.sw;
  if (oy0 < g.oh && oy0 >= nky - 1 && ox0 < g.ow && ox0 >= nkx - 1) return false;
  const int64_t kk = (int64_t)g.kh * g.kw, P = (int64_t)g.oh * g.ow;
  sum = 0.f;
  for (int co = 0; co < cout; ++co) {
    const T *wc = w + ((int64_t)co * g.C + c) * kk + ky0 * g.kw + kx0, *plane = go + co * P;
    for (int i = max(0, oy0 - g.oh + 1); i < nky && i <= oy0; ++i)
      for (int j = max(0, ox0 - g.ow + 1); j < nkx && j <= ox0; ++j)
        sum = fmaf(split_load(wc + i * g.sh * g.kw + j * g.sw), split_load(plane + (oy0 - i) * g.ow + ox0 - j), sum);
  }
  return true;
}

// gX[n][c][y][x] for product column p = (n, pixel of the phase).
template <typename T>
struct PhaseEpilogue {
  T* gx;
  const T *w, *go;
  ConvGeom g;
  int cout, images, z0, phases_x;
  FastDiv pix, nx;
  int fy, fx;
  __device__ __forceinline__ int columns() const { return images * (int)pix.d; }
  __device__ __forceinline__ void enter(int z) {
    const ConvPhase f(g, z0 + z, phases_x);
    pix = FastDiv(f.ny * f.nx), nx = FastDiv(f.nx);
    fy = f.fy, fx = f.fx;
  }
  __device__ __forceinline__ T* at(int m, int n, int y, int x) const {
    return gx + ((int64_t)n * g.C + m) * g.H * g.W + (int64_t)(fy + y * g.sh) * g.W + fx + x * g.sw;
  }
  __device__ __forceinline__ bool operator()(int m, int q, float acc) const {
    int p, x;
    const int n = pix.divmod(q, p), y = nx.divmod(p, x);
    split_store(at(m, n, y, x), acc);
    return acc != acc;
  }
  __device__ __forceinline__ void again(int m, int q) const {
    int p, x;
    const int n = pix.divmod(q, p), y = nx.divmod(p, x);
    float s;
    if (conv_dx_present(w, go + (int64_t)n * cout * g.oh * g.ow, g, cout, m, fy + y * g.sh + g.ph, fx + x * g.sw + g.pw, s))
      split_store(at(m, n, y, x), s);
  }
};

// dX where the windows do not overlap (sh >= kh and sw >= kw): every pixel is
// under at most one kernel position, so the product of W^T (rows kk = (c, ky,
// kx)) and gO (columns q) scatters straight into the image.
template <typename T>
struct WindowEpilogue {
  T* gx;
  ConvGeom g;
  FastDiv kk, kw, P, ow;
  __device__ __forceinline__ void operator()(int m, int q, float acc) const {
    int r, kx, p, ox;
    const int c = kk.divmod(m, r), ky = kw.divmod(r, kx), n = P.divmod(q, p), oy = ow.divmod(p, ox);
    const int y = oy * g.sh - g.ph + ky, x = ox * g.sw - g.pw + kx;
    if (y >= 0 && y < g.H && x >= 0 && x < g.W)
      split_store(gx + (((int64_t)n * g.C + c) * g.H + y) * g.W + x, acc);
  }
};

// y[n][m][p] for product column q = (n, p): [N][M][P] planes.
template <typename T>
struct PlaneEpilogue {
  T* y;
  FastDiv P;
  int M;
  __device__ __forceinline__ void operator()(int m, int q, float acc) const {
    int p;
    const int n = P.divmod(q, p);
    split_store(y + ((int64_t)n * M + m) * P.d + p, acc);
  }
};

// dX at stride 1 with few input channels.  The product's rows are the input
// channels, so that with one of them 31 of 32 rows of its tiles are padding.
// Here a lane owns a pixel (and all C channels), four groups of lanes of the workgroup take
// the output channels in turn and meet in LDS, and the weights lie in LDS,
// read by all lanes of a wave at once.  What is left are the reads of gO: kh kw of
// them per pixel and output channel, all but the first from the caches.
constexpr int kFewChannels = 4;

template <typename T, int C>
__global__ __launch_bounds__(256) void k_conv_dx_few(const T* __restrict__ w, const T* __restrict__ go, T* __restrict__ gx,
                                                     ConvGeom g, int cout, int64_t pixels) {
  extern __shared__ float s_w[];  // [cout][kh kw][C]
  __shared__ float red[4][C][64];
  const int kk = g.kh * g.kw, l = threadIdx.x & 63, grp = threadIdx.x >> 6, P = g.oh * g.ow;
  for (int i = threadIdx.x; i < cout * C * kk; i += 256) {
    const int co = i / (C * kk), r = i - co * (C * kk), c = r / kk;
    s_w[co * C * kk + (r - c * kk) * C + c] = split_load(w + i);
  }
  __syncthreads();
  const int64_t p = (int64_t)blockIdx.x * 64 + l, HW = (int64_t)g.H * g.W;
  const int64_t n = p / HW;
  const int q = (int)(p - n * HW), y = q / g.W + g.ph, x = q % g.W + g.pw;
  float acc[C];
#pragma unroll
  for (int c = 0; c < C; ++c) acc[c] = 0.f;
  if (p < pixels) {
    const T* gon = go + n * cout * P;
    for (int co = grp; co < cout; co += 4) {
      const T* plane = gon + (int64_t)co * P;
      const float* wc = s_w + co * C * kk;
      for (int ky = 0; ky < g.kh; ++ky) {
        const int oy = y - ky;
        const bool row = oy >= 0 && oy < g.oh;
#pragma unroll 5
        for (int kx = 0; kx < g.kw; ++kx) {
          const int ox = x - kx;
          const bool in = row && ox >= 0 && ox < g.ow;
          const float v = split_load(plane + (in ? oy * g.ow + ox : 0));
#pragma unroll
          for (int c = 0; c < C; ++c) acc[c] = fmaf(wc[(ky * g.kw + kx) * C + c], in ? v : 0.f, acc[c]);
        }
      }
    }
  }
#pragma unroll
  for (int c = 0; c < C; ++c) red[grp][c][l] = acc[c];
  __syncthreads();
  if (grp < C && p < pixels) {  // C <= 4 groups: one channel each
    float v = (red[0][grp][l] + red[1][grp][l]) + (red[2][grp][l] + red[3][grp][l]);
    if (v != v) conv_dx_present(w, go + n * cout * P, g, cout, grp, y, x, v);
    split_store(gx + (n * C + grp) * HW + q, v);
  }
}

// Whether k_conv_dx_few takes the image gradient.  Measured (the whole
// backward, us, product / this kernel): fp32 64 x 1 x 28 x 28, 8 kernels 5 x 5 46 /
// 23; 64 x 3 x 32 x 32, 64 3 x 3 78 / 61; 16 x 3 x 224 x 224, 64 3 x 3 730 / 479; one
// 28 x 28 image 26 / 15; bf16 alike (697 / 417 at 224 x 224).  The error against
// float64 is half of the product's.  A lane's loads are one chain, kw of them in
// flight at a time, where the product splits its contraction: on grids below
// three workgroups per CU the chain stays near the longest measured there (75, ten
// 28 x 28 images with 10 kernels 5 x 5: 25.5 / 17.0), beyond near 144 (64 x 3 x 32 x
// 32 above), or 512 for one channel, where nearly all of the product is padding.  Longer
// ones lost in bf16 (8 x 4 x 64 x 64, 80 kernels 4 x 4, chain 320, 78 / 95; 8 x 1 x 64 x
// 64, 512 kernels, chain 2048, 354 / 417), and kernels narrower than three columns
// stay on the product.  The weights in LDS are then at most 10 KB.
bool few_channels(const ConvGeom& g, int64_t N, int cout) {
  const int64_t chain = (int64_t)((cout + 3) / 4) * g.kh * g.kw, workgroups = (N * g.H * g.W + 63) / 64;
  return g.C <= kFewChannels && g.sh == 1 && g.sw == 1 && g.kw >= 3 &&
         chain <= (workgroups < 768 ? 96 : g.C == 1 ? 512 : 160) && grid_fits(workgroups, 256);
}

template <typename T>
int launch_few_channels(const char* fn, const T* w, const T* go, T* gin, int64_t N, int cout, const ConvGeom& g,
                        hipStream_t s) {
  const int64_t pixels = N * g.H * g.W;
  const dim3 grid((unsigned)((pixels + 63) / 64));
  const size_t lds = sizeof(float) * cout * g.C * g.kh * g.kw;
  switch (g.C) {
    case 1: hipLaunchKernelGGL((k_conv_dx_few<T, 1>), grid, dim3(256), lds, s, w, go, gin, g, cout, pixels); break;
    case 2: hipLaunchKernelGGL((k_conv_dx_few<T, 2>), grid, dim3(256), lds, s, w, go, gin, g, cout, pixels); break;
    case 3: hipLaunchKernelGGL((k_conv_dx_few<T, 3>), grid, dim3(256), lds, s, w, go, gin, g, cout, pixels); break;
    default: hipLaunchKernelGGL((k_conv_dx_few<T, 4>), grid, dim3(256), lds, s, w, go, gin, g, cout, pixels); break;
  }
  TT_LAUNCHED(fn, s);
  return ok();
}

ConvDivs conv_divs(const ConvGeom& g) {
  return ConvDivs{FastDiv(g.kh * g.kw), FastDiv(g.kw), FastDiv(g.oh * g.ow), FastDiv(g.ow)};
}

constexpr int64_t kConvPhases = 32768;  // phases per launch (the grid's z extent is 16 bits)

// Images per launch: the product's columns (n, pixel) and the offsets of the
// images' elements stay below 2^30.
int64_t conv_slab(int64_t N, int cout, const ConvGeom& g) {
  const int64_t image = std::max((int64_t)g.C * g.H * g.W, (int64_t)cout * g.oh * g.ow);
  return std::min(N, std::max<int64_t>(1, (int64_t(1) << 30) / image));
}

template <typename T>
int conv_forward(const char* fn, const T* in, const T* w, T* out, int64_t N, int cout, const ConvGeom& g,
                 hipStream_t s) {
  const int64_t P = (int64_t)g.oh * g.ow, K = (int64_t)g.C * g.kh * g.kw, slab = conv_slab(N, cout, g);
  const ConvDivs dv = conv_divs(g);
  for (int64_t n = 0; n < N; n += slab) {
    const int64_t Q = std::min(slab, N - n) * P;
    const int rc = launch_split_gemm<T>(
        fn, cout, Q, K, MatrixSource<T, true>{w, K, cout, (int)K},
        ColumnSource<T, false>(in + n * g.C * g.H * g.W, g, dv, (int)K, (int)Q),
        PlaneEpilogue<T>{out + n * cout * P, dv.P, cout}, s);
    if (rc) return rc;
  }
  return ok();
}

template <typename T>
int conv_backward(const char* fn, const T* in, const T* w, const T* go, T* gin, T* gw, int64_t N, int cout,
                  const ConvGeom& g, hipStream_t s) {
  const int64_t P = (int64_t)g.oh * g.ow, K = (int64_t)g.C * g.kh * g.kw, HW = (int64_t)g.H * g.W;
  const ConvDivs dv = conv_divs(g);
  const int64_t slab = conv_slab(N, cout, g);
  for (int64_t n = 0; n < N; n += slab) {
    const int64_t Q = std::min(slab, N - n) * P;
    const ColumnSource<T, true> col(in + n * g.C * HW, g, dv, (int)K, (int)Q);
    const MatrixEpilogue<T> ep{gw, nullptr, 0, 1.f, n == 0 ? 0.f : 1.f, (int)K};
    const T* gon = go + n * cout * P;
    const int rc = P % SplitT<T>::EPC == 0
                       ? launch_split_gemm<T>(fn, cout, K, Q, GradPlaneSource<T>{gon, dv.P, cout, (int)Q}, col, ep, s)
                       : launch_split_gemm<T>(fn, cout, K, Q, GradRowSource<T, true>(gon, dv.P, cout, (int)Q), col, ep, s);
    if (rc) return rc;
  }
  if (g.sh >= g.kh && g.sw >= g.kw) {
    // pixels outside every window are not written by the product
    const bool tiled = g.sh == g.kh && g.sw == g.kw && g.ph == 0 && g.pw == 0 && g.oh * g.kh == g.H && g.ow * g.kw == g.W;
    if (!tiled) {
      const int rc = tt_elementwise(TT_EW_FILL, sizeof(T) == 2 ? TT_BF16 : TT_F32, gin, nullptr, nullptr,
                                    N * g.C * HW, 0.0, 0.0, 0, s);
      if (rc) return rc;
    }
    for (int64_t n = 0; n < N; n += slab) {
      const int64_t Q = std::min(slab, N - n) * P;
      const int rc = launch_split_gemm<T>(
          fn, K, Q, cout, MatrixSource<T, false>{w, K, (int)K, cout},
          GradRowSource<T, false>(go + n * cout * P, dv.P, cout, (int)Q),
          WindowEpilogue<T>{gin + n * g.C * HW, g, dv.kk, dv.kw, dv.P, dv.ow}, s);
      if (rc) return rc;
    }
    return ok();
  }
  if (few_channels(g, N, cout)) return launch_few_channels(fn, w, go, gin, N, cout, g, s);
  const int phases_x = std::min(g.sw, g.W);
  const int64_t phases = (int64_t)std::min(g.sh, g.H) * phases_x;
  const int64_t pixels = (int64_t)((g.H + g.sh - 1) / g.sh) * ((g.W + g.sw - 1) / g.sw);  // of the largest phase
  const int64_t taps = (int64_t)((g.kh + g.sh - 1) / g.sh) * ((g.kw + g.sw - 1) / g.sw);    // likewise
  for (int64_t n = 0; n < N; n += slab) {
    const int64_t images = std::min(slab, N - n);
    for (int64_t z0 = 0; z0 < phases; z0 += kConvPhases) {
      const int rc = launch_split_gemm<T>(
          fn, g.C, images * pixels, cout * taps, WeightSource<T>(w, g, cout, (int)z0, phases_x),
          GradImageSource<T>(go + n * cout * P, g, cout, (int)images, (int)z0, phases_x),
          PhaseEpilogue<T>{gin + n * g.C * HW, w, go + n * cout * P, g, cout, (int)images, (int)z0, phases_x}, s,
          (int)std::min<int64_t>(kConvPhases, phases - z0));
      if (rc) return rc;
    }
  }
  return ok();
}

// Clamps strides to the padded extent (a longer one also leaves one output)
// and returns whether the products' 32-bit indices and grids cover the shape
// (their rows: cout forward and for dW; C, or C kh kw under windows that do not
// overlap, for dX).
bool conv_fits(ConvGeom& g, int cout) {
  const int64_t lim = int64_t(1) << 30, kk = (int64_t)g.kh * g.kw, P = (int64_t)g.oh * g.ow;
  const int64_t eh = (int64_t)g.H + 2 * (int64_t)g.ph, ew = (int64_t)g.W + 2 * (int64_t)g.pw;
  // (each product below is of factors within 2^31, checked from the left)
  if (eh >= lim / 2 || ew >= lim / 2 || P > lim || (int64_t)g.H * g.W > lim || kk > lim || g.C * ((int64_t)g.H * g.W) > lim ||
      cout * P > lim || g.C * kk > lim || cout * (g.C * kk) > lim)
    return false;
  const bool apart = g.sh >= g.kh && g.sw >= g.kw;
  if (std::max<int64_t>(cout, apart ? g.C * kk : g.C) > split_max_rows(64)) return false;
  g.sh = std::min(g.sh, (int)eh + 1);
  g.sw = std::min(g.sw, (int)ew + 1);
  return true;
}

}  // namespace

}  // namespace tt

using namespace tt;

extern "C" int tt_im2col(int dtype, const void* im, void* col, int64_t N, int C, int H, int W, int kh, int kw,
                         int pad_h, int pad_w, int stride_h, int stride_w, void* stream) {
  return conv_entry<true>("tt_im2col", dtype, im, col, N, C, H, W, kh, kw, pad_h, pad_w, stride_h, stride_w, stream);
}

extern "C" int tt_conv_forward(int dtype, const void* in, const void* weight, void* out, int64_t N, int C, int H,
                               int W, int cout, int kh, int kw, int pad_h, int pad_w, int stride_h, int stride_w,
                               void* stream) {
  const char* fn = "tt_conv_forward";
  ConvGeom g;
  int rc = conv_geom(fn, N, C, H, W, kh, kw, pad_h, pad_w, stride_h, stride_w, g);
  if (rc) return rc;
  if (cout < 0) return fail(TT_ERR_ARG, std::string(fn) + ": negative output channels");
  if (dtype != TT_F32 && dtype != TT_BF16) return fail(TT_ERR_ARG, std::string(fn) + ": dtype must be TT_F32 or TT_BF16");
  if (N == 0 || cout == 0) return ok();
  if (!in || !weight || !out) return fail(TT_ERR_ARG, std::string(fn) + ": null pointer");
  if (!conv_fits(g, cout)) return fail(TT_ERR_UNSUPPORTED, std::string(fn) + ": one image, its output or the weights above 2^30 elements, an axis above 2^29 or the channels above 65535 * 64");
  if ((rc = ensure_init())) return rc;
  hipStream_t s = stream_or_default(stream);
  if (dtype == TT_F32) return conv_forward(fn, (const float*)in, (const float*)weight, (float*)out, N, cout, g, s);
  return conv_forward(fn, (const uint16_t*)in, (const uint16_t*)weight, (uint16_t*)out, N, cout, g, s);
}

extern "C" int tt_conv_backward(int dtype, const void* in, const void* weight, const void* grad_out, void* grad_in,
                                void* grad_weight, int64_t N, int C, int H, int W, int cout, int kh, int kw,
                                int pad_h, int pad_w, int stride_h, int stride_w, void* stream) {
  const char* fn = "tt_conv_backward";
  ConvGeom g;
  int rc = conv_geom(fn, N, C, H, W, kh, kw, pad_h, pad_w, stride_h, stride_w, g);
  if (rc) return rc;
  if (N < 1 || cout < 1) return fail(TT_ERR_ARG, std::string(fn) + ": N and output channels >= 1 required");
  if (dtype != TT_F32 && dtype != TT_BF16) return fail(TT_ERR_ARG, std::string(fn) + ": dtype must be TT_F32 or TT_BF16");
  if (!in || !weight || !grad_out || !grad_in || !grad_weight)
    return fail(TT_ERR_ARG, std::string(fn) + ": null pointer");
  if (!conv_fits(g, cout)) return fail(TT_ERR_UNSUPPORTED, std::string(fn) + ": one image, its output or the weights above 2^30 elements, an axis above 2^29 or the channels (times the kernel under separate windows) above 65535 * 64");
  if ((rc = ensure_init())) return rc;
  hipStream_t s = stream_or_default(stream);
  if (dtype == TT_F32)
    return conv_backward(fn, (const float*)in, (const float*)weight, (const float*)grad_out, (float*)grad_in,
                         (float*)grad_weight, N, cout, g, s);
  return conv_backward(fn, (const uint16_t*)in, (const uint16_t*)weight, (const uint16_t*)grad_out,
                       (uint16_t*)grad_in, (uint16_t*)grad_weight, N, cout, g, s);
}

extern "C" int tt_col2im(int dtype, const void* col, void* im, int64_t N, int C, int H, int W, int kh, int kw,
                         int pad_h, int pad_w, int stride_h, int stride_w, void* stream) {
  return conv_entry<false>("tt_col2im", dtype, col, im, N, C, H, W, kh, kw, pad_h, pad_w, stride_h, stride_w,
                           stream);
}

namespace tt {
namespace {

// backward: (a, b, c) = (grad_out, mask, grad_in); forward: (in, out, mask).
int pool_launch(const char* fn, bool backward, const float* a, float* b, float* c, int64_t planes, int H, int W,
                int kh, int kw, int ph, int pw, int sh, int sw, void* stream) {
  ConvGeom g;
  int rc = conv_geom(fn, planes, 1, H, W, kh, kw, ph, pw, sh, sw, g);
  if (rc) return rc;
  const int64_t total = backward ? planes * (int64_t)H * W : planes * (int64_t)g.oh * g.ow;
  if (total == 0) return ok();
  if (!a || !b || !c) return fail(TT_ERR_ARG, std::string(fn) + ": null pointer");
  rc = ensure_init();
  if (rc) return rc;
  hipStream_t s = stream_or_default(stream);
  int64_t blocks = (total + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  if (backward)
    hipLaunchKernelGGL(k_maxpool_backward, dim3((unsigned)blocks), dim3(256), 0, s, a, b, c, total, g);
  else
    hipLaunchKernelGGL(k_maxpool, dim3((unsigned)blocks), dim3(256), 0, s, a, b, c, total, g);
  TT_LAUNCHED(fn, s);
  return ok();
}

}  // namespace
}  // namespace tt

extern "C" int tt_maxpool_f32(const float* in, float* out, float* mask, int64_t planes, int H, int W, int kh,
                              int kw, int pad_h, int pad_w, int stride_h, int stride_w, void* stream) {
  return tt::pool_launch("tt_maxpool_f32", false, in, out, mask, planes, H, W, kh, kw, pad_h, pad_w, stride_h,
                         stride_w, stream);
}

extern "C" int tt_maxpool_backward_f32(const float* grad_out, const float* mask, float* grad_in, int64_t planes,
                                       int H, int W, int kh, int kw, int pad_h, int pad_w, int stride_h,
                                       int stride_w, void* stream) {
  // the mask is only read; the helper's middle pointer is writable for the forward's output
  return tt::pool_launch("tt_maxpool_backward_f32", true, grad_out, const_cast<float*>(mask), grad_in, planes, H, W,
                         kh, kw, pad_h, pad_w, stride_h, stride_w, stream);
}

