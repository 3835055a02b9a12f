// Kernels of the image structure function path (gfx950, wave64).
//
//   k_rows  stage (a), row pass: pixel convert (+ frame-0 subtraction) x window,
//           two frames packed as one complex row, length-nx FFT, split into the
//           two half spectra, blocked store R[tb][kx][y][ti].
//   k_cols  stage (a) column pass + stage (b) transpose: length-ny FFT of Tb
//           frames of one kx column at once, store q-major S[q][t] in runs of
//           Tb consecutive frames.
//
// The time stages live in fddm_time_wave.hip, fddm_time_pair.hip,
// fddm_time_p2.hip and fddm_time_long.hip (fft mode) and fddm_diff.hip.
//
// Semantics follow the reference cores: spectra and normalisation
// src/cpp/ddm.cc:288-323, correlation and two-ended sums ddm.cc:344-426,
// differences ddm.cc:117-171, output shift src/cpp/helper_ddm.cc:41-103.
#include <type_traits>

#include "fddm_fft.hpp"
#include "fddm_kernels.hpp"
#include "fddm_spatial.hpp"

namespace fddm {

constexpr int kThreads = 256;

int fft_bucket(long long work) {
  const long long e = (work + kThreads - 1) / kThreads;
  if (e <= 4) return 4;
  if (e <= 8) return 8;
  if (e <= 16) return 16;
  if (e <= 32) return 32;
  if (e <= 64) return 64;
  return 0;
}

// ---------------------------------------------------------------------------
// Pixel conversion.  Integer frame differences are formed exactly in integer
// arithmetic before the conversion to T.
// ---------------------------------------------------------------------------
template <typename Tin, typename T>
__device__ __forceinline__ T load_pixel(const Tin* __restrict__ img, const Tin* __restrict__ ref, size_t idx, size_t idx0,
                                        bool sub) {
  if constexpr (std::is_integral_v<Tin> && sizeof(Tin) <= 2) {
    int v = static_cast<int>(img[idx]);
    if (sub) v -= static_cast<int>(ref[idx0]);
    return static_cast<T>(v);
  } else if constexpr (std::is_integral_v<Tin> && sizeof(Tin) == 4) {
    long long v = static_cast<long long>(img[idx]);
    if (sub) v -= static_cast<long long>(ref[idx0]);
    return static_cast<T>(v);
  } else if constexpr (std::is_integral_v<Tin>) {
    double v = static_cast<double>(img[idx]);
    if (sub) v -= static_cast<double>(ref[idx0]);
    return static_cast<T>(v);
  } else {
    // floating pixels: the difference in the wider of the two types
    using Wd = std::conditional_t<(sizeof(Tin) > sizeof(T)), Tin, T>;
    Wd v = static_cast<Wd>(img[idx]);
    if (sub) v -= static_cast<Wd>(ref[idx0]);
    return static_cast<T>(v);
  }
}

// ---------------------------------------------------------------------------
// Stage (a): row pass.
// ---------------------------------------------------------------------------
template <typename Tin, typename T, int E>
__global__ void __launch_bounds__(kThreads) k_rows(RowArgs a) {
  using C = cplx_t<T>;
  extern __shared__ __align__(16) unsigned char smem[];
  C* buf = reinterpret_cast<C*>(smem);
  const int tid = threadIdx.x;
  const int H = a.H, W = a.W, nx = a.nx, Tb = a.Tb, G = a.G;
  const int nxh = nx / 2 + 1;
  const int y = blockIdx.x % H;
  const uint64_t tb = blockIdx.x / H;
  const uint64_t t0 = tb * Tb;
  const Tin* __restrict__ img = static_cast<const Tin*>(a.img);
  const Tin* __restrict__ ref = static_cast<const Tin*>(a.img0);  // the subtracted frame
  const T* __restrict__ win = static_cast<const T*>(a.window);
  const T half_norm = static_cast<T>(0.5 * a.norm);
  const int bstride = nx + 1;
  const size_t plane = static_cast<size_t>(H) * W;
  C* __restrict__ R = static_cast<C*>(a.R);
  const C* __restrict__ tw = static_cast<const C*>(a.twx);

  const sp::BlockFrames<sizeof(T) == 8> fr(a, t0, Tb, plane);
  const bool sub = a.subtract0 != 0;
  for (int g0 = 0; g0 < Tb / 2; g0 += G) {
    for (int w = tid; w < G * nx; w += kThreads) {
      const int p = w / nx, x = w - p * nx;
      T va = 0, vb = 0;
      if (x < W) {
        const int ka = 2 * (g0 + p), kb = ka + 1;
        const size_t i0 = static_cast<size_t>(y) * W + x;
        if (fr.here(ka)) va = load_pixel<Tin, T>(img, ref, fr.at(ka, plane) + i0, i0, sub && !fr.is_raw(ka));
        if (kb < fr.n) vb = load_pixel<Tin, T>(img, ref, fr.first + kb * plane + i0, i0, sub);
        if (win) {
          const T wv = win[i0];
          va *= wv;
          vb *= wv;
        }
      }
      buf[lds_pad(p * bstride + x)] = C{va, vb};
    }
    __syncthreads();
    fft_lds<T, E, false>(buf, 0, a.dx, G, 0, bstride, 1, tw, tid, kThreads);
    // Z = A + i B with A, B the spectra of the two real rows:
    // A(k) = (Z(k) + conj Z(-k)) / 2, B(k) = (Z(k) - conj Z(-k)) / 2i.
    const int nti = 2 * G;
    for (int w = tid; w < nxh * nti; w += kThreads) {
      const int tl = w % nti, k = w / nti;
      const int p = tl >> 1;
      const C zk = buf[lds_pad(p * bstride + k)];
      const C zn = buf[lds_pad(p * bstride + (k == 0 ? 0 : nx - k))];
      C o;
      if ((tl & 1) == 0) {
        o = C{(zk.x + zn.x) * half_norm, (zk.y - zn.y) * half_norm};
      } else {
        o = C{(zk.y + zn.y) * half_norm, (zn.x - zk.x) * half_norm};
      }
      const int ti = 2 * g0 + tl;
      R[((tb * nxh + k) * static_cast<size_t>(H) + y) * Tb + ti] = o;
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Stage (a) columns + (b) q-major store.  PAIRS: the plan may hold passes of
// radix 10 or 6.  Lengths without them (96: 3 x 4 x 8) keep a kernel without
// their loops, which took 5 % (400 frames of 96^2 in FP64 22.6 us, without 21.3).
// ---------------------------------------------------------------------------
template <typename T, int E, bool PAIRS>
__global__ void __launch_bounds__(kThreads) k_cols(ColArgs a) {
  using C = cplx_t<T>;
  extern __shared__ __align__(16) unsigned char smem[];
  C* buf = reinterpret_cast<C*>(smem);
  const int tid = threadIdx.x;
  const int nxh = a.nxh, H = a.H, ny = a.ny, Tb = a.Tb;
  const int kx = blockIdx.x % nxh;
  const uint64_t tb = blockIdx.x / nxh;
  const C* __restrict__ src = static_cast<const C*>(a.R) + (tb * nxh + kx) * static_cast<size_t>(H) * Tb;
  const int nin = H * Tb, nall = ny * Tb;
  for (int w = tid; w < nall; w += kThreads) buf[lds_pad(w)] = w < nin ? src[w] : C{0, 0};
  __syncthreads();
  const C* __restrict__ tw = static_cast<const C*>(a.twy);
  const int logG = __builtin_ctz(a.G);
  for (int g0 = 0; g0 < Tb; g0 += a.G) fft_lds<T, E, true, PAIRS>(buf, g0, a.dy, a.G, logG, 1, Tb, tw, tid, kThreads);
  C* __restrict__ S = static_cast<C*>(a.S);
  for (int w = tid; w < nall; w += kThreads) {
    const int ti = w % Tb, ky = w / Tb;
    S[(static_cast<size_t>(ky) * nxh + kx) * a.Lp + tb * Tb + ti] = buf[lds_pad(w)];
  }
}

// ---------------------------------------------------------------------------
// FFT engine test kernel: one forward transform per workgroup, in place.
// ---------------------------------------------------------------------------
template <typename T, int E>
__global__ void __launch_bounds__(kThreads) k_fft_test(cplx_t<T>* data, FftDesc d, const cplx_t<T>* tw) {
  using C = cplx_t<T>;
  extern __shared__ __align__(16) unsigned char smem[];
  C* buf = reinterpret_cast<C*>(smem);
  C* p = data + static_cast<size_t>(blockIdx.x) * d.n;
  for (int t = threadIdx.x; t < d.n; t += kThreads) buf[lds_pad(t)] = p[t];
  __syncthreads();
  fft_lds<T, E, false>(buf, 0, d, 1, 0, d.n, 1, tw, threadIdx.x, kThreads);
  for (int t = threadIdx.x; t < d.n; t += kThreads) p[t] = buf[lds_pad(t)];
}

// ---------------------------------------------------------------------------
// Launchers.
// ---------------------------------------------------------------------------
namespace {

template <typename K, typename... Args>
hipError_t launch(K kernel, unsigned grid, size_t lds, hipStream_t s, Args... args) {
  if (grid == 0) return hipSuccess;
  if (lds > 64 * 1024) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(kThreads), lds, s, args...);
  return hipGetLastError();
}

template <typename Tin, typename T>
hipError_t rows_e(const RowArgs& a, unsigned grid, size_t lds, int e, hipStream_t s) {
  switch (e) {
    case 16: return launch(k_rows<Tin, T, 16>, grid, lds, s, a);
    case 32: return launch(k_rows<Tin, T, 32>, grid, lds, s, a);
    default: return hipErrorInvalidValue;
  }
}

template <typename T>
hipError_t rows_t(const RowArgs& a, unsigned grid, size_t lds, int e, hipStream_t s) {
  switch (a.in_dtype) {
    case IN_U8: return rows_e<uint8_t, T>(a, grid, lds, e, s);
    case IN_I16: return rows_e<int16_t, T>(a, grid, lds, e, s);
    case IN_U16: return rows_e<uint16_t, T>(a, grid, lds, e, s);
    case IN_I32: return rows_e<int32_t, T>(a, grid, lds, e, s);
    case IN_U32: return rows_e<uint32_t, T>(a, grid, lds, e, s);
    case IN_I64: return rows_e<int64_t, T>(a, grid, lds, e, s);
    case IN_U64: return rows_e<uint64_t, T>(a, grid, lds, e, s);
    case IN_F32: return rows_e<float, T>(a, grid, lds, e, s);
    case IN_F64: return rows_e<double, T>(a, grid, lds, e, s);
    default: return hipErrorInvalidValue;
  }
}

int rc_bucket(long long work) {
  const int e = fft_bucket(work);
  return e <= 16 ? 16 : e;
}

}  // namespace

hipError_t launch_rows(const RowArgs& a, int precision, hipStream_t s) {
  if (!a.generic && rows_mr_ok(a, precision)) return launch_rows_mr(a, precision, s);
  const uint64_t nblocks = (a.frames + a.Tb - 1) / a.Tb;
  const unsigned grid = static_cast<unsigned>(nblocks * a.H);
  const int e = rc_bucket(static_cast<long long>(a.G) * a.nx);
  if (precision == PREC_FP64) {
    return rows_t<double>(a, grid, sizeof(double2) * lds_padded_size(a.G * (a.nx + 1)), e, s);
  }
  return rows_t<float>(a, grid, sizeof(float2) * lds_padded_size(a.G * (a.nx + 1)), e, s);
}

hipError_t launch_cols(const ColArgs& a, int precision, hipStream_t s) {
  if (!a.generic && cols_mr_ok(a, precision)) return launch_cols_mr(a, precision, s);
  const unsigned grid = static_cast<unsigned>(a.nblocks * a.nxh);
  const int e = rc_bucket(static_cast<long long>(a.G) * a.ny);
  const bool pairs = a.dy.c10 + a.dy.c6 > 0;
  if (precision == PREC_FP64) {
    const size_t lds = sizeof(double2) * lds_padded_size(a.ny * a.Tb);
    if (e == 16) return launch(pairs ? k_cols<double, 16, true> : k_cols<double, 16, false>, grid, lds, s, a);
    if (e == 32) return launch(pairs ? k_cols<double, 32, true> : k_cols<double, 32, false>, grid, lds, s, a);
  } else {
    const size_t lds = sizeof(float2) * lds_padded_size(a.ny * a.Tb);
    if (e == 16) return launch(pairs ? k_cols<float, 16, true> : k_cols<float, 16, false>, grid, lds, s, a);
    if (e == 32) return launch(pairs ? k_cols<float, 32, true> : k_cols<float, 32, false>, grid, lds, s, a);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_fft_test(void* data, int n, int batch, const FftDesc& d, const void* tw, int precision,
                           hipStream_t s) {
  const int e = fft_bucket(n);
  if (precision == PREC_FP64) {
    using C = double2;
    const size_t lds = sizeof(C) * lds_padded_size(n);
    C* p = static_cast<C*>(data);
    const C* t = static_cast<const C*>(tw);
    switch (e) {
      case 4: return launch(k_fft_test<double, 4>, batch, lds, s, p, d, t);
      case 8: return launch(k_fft_test<double, 8>, batch, lds, s, p, d, t);
      case 16: return launch(k_fft_test<double, 16>, batch, lds, s, p, d, t);
      case 32: return launch(k_fft_test<double, 32>, batch, lds, s, p, d, t);
      default: return hipErrorInvalidValue;
    }
  }
  using C = float2;
  const size_t lds = sizeof(C) * lds_padded_size(n);
  C* p = static_cast<C*>(data);
  const C* t = static_cast<const C*>(tw);
  switch (e) {
    case 4: return launch(k_fft_test<float, 4>, batch, lds, s, p, d, t);
    case 8: return launch(k_fft_test<float, 8>, batch, lds, s, p, d, t);
    case 16: return launch(k_fft_test<float, 16>, batch, lds, s, p, d, t);
    case 32: return launch(k_fft_test<float, 32>, batch, lds, s, p, d, t);
    case 64: return launch(k_fft_test<float, 64>, batch, lds, s, p, d, t);
    default: return hipErrorInvalidValue;
  }
}

namespace {

// Device buffer -> pinned host buffer, 16 bytes per lane and four in flight
// per lane: the GPU writes the host pages itself over the host link.
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(256) void k_copy_out(const u32x4* __restrict__ src, u32x4* __restrict__ dst,
                                                  uint64_t n16) {
  const uint64_t stride = uint64_t(gridDim.x) * 256;
  uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const u32x4 a = src[i], b = src[i + stride], c = src[i + 2 * stride], d = src[i + 3 * stride];
    dst[i] = a;
    dst[i + stride] = b;
    dst[i + 2 * stride] = c;
    dst[i + 3 * stride] = d;
  }
  for (; i < n16; i += stride) dst[i] = src[i];
}

}  // namespace

hipError_t launch_copy_out(void* dst, const void* src, uint64_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  if (n % 16 || reinterpret_cast<uintptr_t>(src) % 16 || reinterpret_cast<uintptr_t>(dst) % 16)
    return hipErrorInvalidValue;
  const uint64_t n16 = n / 16;
  const unsigned blocks = static_cast<unsigned>(std::min<uint64_t>((n16 + 255) / 256, 1024));
  hipLaunchKernelGGL(k_copy_out, dim3(blocks), dim3(256), 0, s, static_cast<const u32x4*>(src),
                     static_cast<u32x4*>(dst), n16);
  return hipGetLastError();
}

}  // namespace fddm
