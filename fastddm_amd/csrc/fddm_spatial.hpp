// Helpers shared by the spatial (row-pass) kernels of every size class.
#pragma once

#include <type_traits>

#include "fddm_kernels.hpp"

namespace fddm {
namespace sp {

// The frames t0 + k, k < Tb, of one block of a row launch.  All of it is uniform
// over a workgroup, so a lane is left with 32-bit compares of k.  EDGES: the
// launch may set split, gap and raw (RowArgs).  The scalar registers for them
// have the arguments loaded one after the other, a microsecond a launch (8 x 8^2
// in FP32 6.1 -> 5.5 us without), so kernels whose launches do not leave them out.
template <bool EDGES>
struct BlockFrames {
  int n;          // frames k < n lie one after the other from pixel `first` of img on
  int raw;        // frame k == raw (even; none: < 0) is frame 0 of img, nothing subtracted
  uint64_t first;

  __device__ __forceinline__ BlockFrames(const RowArgs& a, uint64_t t0, int Tb, uint64_t plane)
      : n(static_cast<int>(a.L < t0 ? 0 : a.L - t0 < static_cast<uint64_t>(Tb) ? a.L - t0 : Tb)), raw(-1) {
    if constexpr (EDGES) {
      const uint32_t t = static_cast<uint32_t>(t0);
      if (a.raw - t < static_cast<uint32_t>(Tb)) raw = static_cast<int>(a.raw - t);
      if (t >= a.split) t0 += a.gap;
    }
    first = t0 * plane;
  }
  __device__ __forceinline__ bool is_raw(int k) const { return EDGES && k == raw; }
  __device__ __forceinline__ bool here(int k) const { return k < n || is_raw(k); }
  // first pixel of frame k
  __device__ __forceinline__ uint64_t at(int k, uint64_t plane) const {
    return is_raw(k) ? 0 : first + static_cast<uint64_t>(k) * plane;
  }
};

// Pixel (p, x) of a pair row: converted, frame 0 subtracted in integer
// arithmetic where the type allows, times the window value.
template <typename Tin, typename T>
__device__ __forceinline__ T pixel_value(Tin v, Tin v0, bool sub, T w) {
  if constexpr (std::is_integral_v<Tin> && sizeof(Tin) <= 2) {
    return static_cast<T>(static_cast<int>(v) - (sub ? static_cast<int>(v0) : 0)) * w;
  } else if constexpr (std::is_integral_v<Tin> && sizeof(Tin) == 4) {
    return static_cast<T>(static_cast<long long>(v) - (sub ? static_cast<long long>(v0) : 0)) * w;
  } else if constexpr (std::is_integral_v<Tin>) {
    return static_cast<T>(static_cast<double>(v) - (sub ? static_cast<double>(v0) : 0.0)) * w;
  } else {
    // floating pixels: the difference in the wider of the two types (a
    // float32 difference would round where the FP64 transform is exact)
    using Wd = std::conditional_t<(sizeof(Tin) > sizeof(T)), Tin, T>;
    return static_cast<T>(sub ? static_cast<Wd>(v) - static_cast<Wd>(v0) : static_cast<Wd>(v)) * w;
  }
}

// Split of pair row p at frequency k, Z = FFT(frame 2p + i frame 2p+1):
// A(k) = (Z(k) + conj Z(-k)) / 2 and B(k) = (Z(k) - conj Z(-k)) / 2i (times
// the norm), stored together at dst (frames 2p and 2p+1 are neighbours in R):
// one 16-byte store in FP32, and one read of the two Z values per pair.
template <typename T>
__device__ __forceinline__ void split_store(cplx_t<T>* dst, cplx_t<T> zk, cplx_t<T> zn, T half_norm) {
  const T ax = (zk.x + zn.x) * half_norm, ay = (zk.y - zn.y) * half_norm;
  const T bx = (zk.y + zn.y) * half_norm, by = (zn.x - zk.x) * half_norm;
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4*>(dst) = make_float4(ax, ay, bx, by);
  } else {
    dst[0] = cplx_t<T>{ax, ay};
    dst[1] = cplx_t<T>{bx, by};
  }
}

}  // namespace sp
}  // namespace fddm
