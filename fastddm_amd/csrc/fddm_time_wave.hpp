// Transforms held in the registers of one wave, shared by the time kernels
// of fddm_time_wave.hip (one wave per transform pair) and fddm_time_pair.hip
// (the even and odd bins on two waves).
//
// An M-point transform is worked on by P lanes of one wave holding R points
// each (M = P R, sample t = p + P r in register r of lane p): a radix-R DFT in
// registers, the twiddles W_M^(p k1), an exchange through the wave's own LDS,
// and the P-point transforms over p in registers again (one pass for P <= R,
// one radix-2 step between the wave's halves and one pass for P = 64, R = 32,
// two passes otherwise).  The result is in natural order, bin k = p + P r in
// register r of lane p.  All LDS addresses are one base per lane plus
// immediate offsets.
#pragma once

#include <cmath>
#include <type_traits>
#include <vector>

#include "fddm_kernels.hpp"
#include "fddm_p2.hpp"
#include "fddm_wave.hpp"

namespace fddm {
namespace tw {
using namespace p2;

constexpr int kEdge = 32;  // lags of at most this many pairs: direct sums

// The last kEdge samples as the direct sums read them: sample L - n + t, the
// later one of pair t < n of the lag with n pairs, is in place late_place(n, t).
// The sums run over the same t for every lag and drop t >= n, so they read up
// to place late_place(1, kEdge - 1); the places from kEdge on hold zeros.
constexpr int kLast = 2 * kEdge;
__host__ __device__ constexpr int late_place(int n, int t) { return kEdge - n + t; }

// Shape and LDS layout of M = P R.  Elements are 8 bytes: a float complex
// value, or one component of a double one (exchanged one after the other).
template <int R_, int P_, int W_ = 4>
struct WaveLay {
  static constexpr int R = R_, P = P_, M = R * P, GROUPS = 64 / P, W = W_, Q = W * GROUPS;  // W: waves per workgroup
  // second stage, P points per k1: one pass (P <= R), a radix-2 step between
  // the halves of the wave and one pass (P = 2R = 64), or two passes R R3
  static constexpr bool LANE2 = P == 64 && R == 32;
  static constexpr int R3 = P > R && !LANE2 ? P / R : 1;
  static_assert(LANE2 || (P <= R ? R % P == 0 : R % R3 == 0), "plan");
  // exchange: rows of NC elements, read back 16 bytes at a time; blocks of
  // NC + 2 put eight such reads in distinct banks (three passes: R3 blocks
  // of R a row, then R3 rows of R^2)
  static constexpr int NC = LANE2 || R3 > 1 ? R : P, RS = R3 > 1 ? R3 * (R + 2) + 2 : R == 64 ? NC + 4 : NC + 2;
  static constexpr int ROWS = R3 > 1 ? R : M / NC, RS3 = R * R + 16;
  static constexpr int GS0 = ROWS * RS > R3 * RS3 || R3 == 1 ? ROWS * RS : R3 * RS3;
  static constexpr int GS = GS0 + (GROUPS > 2 ? P : 0);  // groups start in distinct banks
  // chunks of R consecutive samples, stride R + 2
  static constexpr int CS = R + 2, CG = P * CS;
  static constexpr int NB = P >= R ? 1 : R / P;  // register rows per chunk, where a chunk is longer than a row
  static constexpr int chunk_row(int r) { return P >= R ? r * (P / R) * CS : (r / NB) * CS + (r % NB) * P; }
  // the exchange buffer or the chunks, then the last samples of each group
  static constexpr int BUF = GROUPS * (GS > CG ? GS : CG), WAVE = BUF + GROUPS * kLast;
  static constexpr size_t bytes = sizeof(double) * W * WAVE;
  // tables, complex of the compute type: W_M^(p k1) at [k1][p],
  // W_M^(p (k1 + 1/2)) at [k1][p], then W_P^j (j < R; LANE2) or W_P^(p0 k2) at
  // [k2][p0] (R3 > 1), (cos, sin)(2 pi d / N) for d < M / 2; in double
  // 1 / (L - d) for d < M
  static constexpr int TW_E = 0, TW_O = M, TW_2 = 2 * M, TW_CS = TW_2 + (LANE2 ? R : R3 > 1 ? P : 0);
  static constexpr int TW_END = TW_CS + M / 2;
  // R = 64: real and imaginary parts one after the other also in FP32 (4-byte elements)
  template <typename T>
  static constexpr bool by_part() {
    return sizeof(T) == 8 || R == 64;
  }
};

// Position of sample t in the chunk layout.
template <int R>
__host__ __device__ __forceinline__ int chunk_pos(int t) {
  constexpr int LR = R == 32 ? 5 : R == 16 ? 4 : 3;
  static_assert(R == 1 << LR, "R");
  return t + ((t >> LR) << 1);
}

// Orders this wave's LDS writes before its later reads (the hardware keeps a
// wave's LDS accesses in order; this keeps the compiler from moving them).
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// a: [a of lanes 0..31 | b of lanes 0..31], b: [a of 32..63 | b of 32..63]
__device__ __forceinline__ void swap32(float& a, float& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap32(double& a, double& b) {
  const uint64_t ua = static_cast<uint64_t>(__double_as_longlong(a)), ub = static_cast<uint64_t>(__double_as_longlong(b));
  const auto lo = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(ua), static_cast<unsigned>(ub), false, false);
  const auto hi =
      __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(ua >> 32), static_cast<unsigned>(ub >> 32), false, false);
  a = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi[0]) << 32) | lo[0]));
  b = __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi[1]) << 32) | lo[1]));
}

__device__ __forceinline__ float from_lane(float v, int addr) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(addr, __float_as_int(v)));
}
__device__ __forceinline__ double from_lane(double v, int addr) {
  const uint64_t u = static_cast<uint64_t>(__double_as_longlong(v));
  const unsigned lo = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(addr, static_cast<int>(u & 0xffffffffull)));
  const unsigned hi = static_cast<unsigned>(__builtin_amdgcn_ds_bpermute(addr, static_cast<int>(u >> 32)));
  return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// Inclusive scan over the P lanes of a group, and the group's total in every lane.
template <int P>
__device__ __forceinline__ double group_scan(double v, int p) {
  if constexpr (P == 64) return wave::incl_scan(v);
#pragma unroll
  for (int s = 1; s < P; s *= 2) {
    const double u = __shfl_up(v, s, P);
    v += p >= s ? u : 0.0;
  }
  return v;
}
template <int P>
__device__ __forceinline__ double group_last(double v) {
  if constexpr (P == 64) return wave::lane63(v);
  return __shfl(v, P - 1, P);
}

// Keeps what is written before it (a batch of loads) ahead of what follows:
// left alone, the scheduler sinks each load to its use to save registers and
// waits for them one by one.
__device__ __forceinline__ void issued() { __builtin_amdgcn_sched_barrier(0); }

// Adds the squared differences of the pairs t = s0, s0 + STEP, ... of the lag
// with n pairs, t < end and t < n, B pairs in flight: sample t of a block from
// t0 on is early[t - t0 + pos(t0)].  late and early are arrays, or stand-ins
// that check their indices (the test of the ranges).
template <int STEP, int B, typename Late, typename Early, typename Pos, typename F>
__host__ __device__ __forceinline__ void few_pairs(double& sum, int n, int s0, int end, const Late& late, const Early& early,
                                                   Pos&& pos, F&& square) {
#pragma nounroll
  for (int t0 = 0; t0 < end; t0 += B * STEP) {
    std::decay_t<decltype(late[0])> x1[B], x0[B];
#pragma unroll
    for (int b = 0; b < B; ++b) {
      x1[b] = late[late_place(n, s0) + t0 + b * STEP];
      x0[b] = early[s0 + b * STEP + pos(t0)];
    }
#if defined(__HIP_DEVICE_COMPILE__)
    issued();
#endif
#pragma unroll
    for (int b = 0; b < B; ++b) sum += t0 + b * STEP + s0 < n ? square(x1[b], x0[b]) : 0.0;
  }
}

// Element i + p of a table (i the same for all lanes).
template <typename E>
__device__ __forceinline__ E entry(const E* __restrict__ table, int i, unsigned p) {
  return *reinterpret_cast<const E*>(reinterpret_cast<const char*>(table + i) + p * static_cast<unsigned>(sizeof(E)));
}

// Exchange between two passes: register i written to position wpos(i), then
// runs of NC registers read from consecutive positions from rpos(run) on
// (16 bytes at a time where NC > 1).
template <int R, int NC, typename E, typename FR>
__device__ __forceinline__ void read_rows(const E* b, E (&x)[R], FR&& rpos) {
  if constexpr (NC == 1) {
#pragma unroll
    for (int i = 0; i < R; ++i) x[i] = b[rpos(i)];
  } else {
    constexpr int V = 16 / sizeof(E);
    struct alignas(16) Vec {
      E e[V];
    };
#pragma unroll
    for (int i = 0; i < R; i += V) {
      const Vec t = *reinterpret_cast<const Vec*>(b + rpos(i / NC) + i % NC);
#pragma unroll
      for (int k = 0; k < V; ++k) x[i + k] = t.e[k];
    }
  }
}
// BY_PART: real parts, then imaginary parts (elements of T), else complex values.
template <typename T, int R, int NC, bool BY_PART, typename FW, typename FR>
__device__ __forceinline__ void exchange(cplx_t<T> (&v)[R], double* lds, FW&& wpos, FR&& rpos) {
  if constexpr (!BY_PART) {
    auto* const b = reinterpret_cast<cplx_t<T>*>(lds);
#pragma unroll
    for (int i = 0; i < R; ++i) b[wpos(i)] = v[i];
    wave_sync();
    read_rows<R, NC>(b, v, rpos);
    wave_sync();
  } else {
    T* const b = reinterpret_cast<T*>(lds);
    T x[R];
#pragma unroll
    for (int i = 0; i < R; ++i) b[wpos(i)] = v[i].x;
    wave_sync();
    read_rows<R, NC>(b, x, rpos);
    wave_sync();
#pragma unroll
    for (int i = 0; i < R; ++i) b[wpos(i)] = v[i].y;
    wave_sync();
#pragma unroll
    for (int i = 0; i < R; ++i) v[i].x = x[i];
    read_rows<R, NC>(b, x, rpos);
#pragma unroll
    for (int i = 0; i < R; ++i) v[i].y = x[i];
    wave_sync();
  }
}

// Forward M-point transform, natural order in and out.  odd: of x(t) W_N^t,
// the odd bins of the N-point one (in the first DFT W_R^(r / 2), the rest in
// the twiddle table).  t1, t2: twiddles of the first and second stage.  mid()
// runs after the exchange (the place to issue loads for what follows).
// The twiddles are read before the first DFT if they take at most 64 VGPRs;
// otherwise in batches of 16 VGPRs, each ahead of the one in use.
template <typename T, typename Lay, typename Odd, typename F>
__device__ __forceinline__ void wave_fft(cplx_t<T> (&v)[Lay::R], double* lds, const cplx_t<T>* __restrict__ t1,
                                         const cplx_t<T>* __restrict__ t2, int p, Odd odd, F&& mid) {
  using C = cplx_t<T>;
  constexpr int R = Lay::R, P = Lay::P, RS = Lay::RS, R3 = Lay::R3;
  constexpr int WB = sizeof(C) * R <= 256 ? R : static_cast<int>(64 / sizeof(C)), NW = R / WB;
  constexpr bool BY_PART = Lay::template by_part<T>();
  if (odd) sfor<1, R>([&](auto rc) {
      constexpr int r = decltype(rc)::value;
      v[r] = mul_w<T, r, 2 * R>(v[r]);
    });
  C w[NW > 1 ? 2 : 1][WB];
#pragma unroll
  for (int k = 0; k < WB; ++k) w[0][k] = entry(t1, k * P, p);
  C wl{};
  if constexpr (Lay::LANE2) wl = entry(t2, 0, p & (R - 1));
  issued();
  dft<T, R>(v);
#pragma unroll
  for (int b = 0; b < NW; ++b) {
    if (b + 1 < NW) {
#pragma unroll
      for (int k = 0; k < WB; ++k) w[(b + 1) % 2][k] = entry(t1, ((b + 1) * WB + k) * P, p);
      issued();
    }
#pragma unroll
    for (int k = 0; k < WB; ++k)
      if (b + k > 0 || !std::is_same_v<Odd, std::false_type>) v[b * WB + k] = cmul(v[b * WB + k], w[b % 2][k]);
  }
  if constexpr (Lay::LANE2) {
    // bins k1 + R k2, k2 = 2 kappa + g: sums (g = 0) and differences (g = 1)
    // of samples j and j + R of the P-point transforms; lanes below 32 take
    // the even k1, the others the odd ones
    const int j = p & (R - 1), hi = p >> 5;
    static_assert(R == 32, "the halves of the wave");
#pragma unroll
    for (int i = 0; i < R; i += 2) {
      swap32(v[i].x, v[i + 1].x);
      swap32(v[i].y, v[i + 1].y);
      const C a = v[i], b = v[i + 1];
      v[i] = cadd(a, b);
      v[i + 1] = cmul(csub(a, b), wl);
    }
    const int wb = hi * RS + j, rb = p * RS;
    // register i + g holds (k1 = i + hi, g): row k1 + R g
    exchange<T, R, R, BY_PART>(v, lds, [&](int i) { return wb + ((i & ~1) + R * (i & 1)) * RS; }, [&](int) { return rb; });
    mid();
    dft<T, R>(v);
  } else if constexpr (R3 > 1) {
    // sample p = p0 + R3 p1 of the P-point transforms: radix R over p1 (lane
    // p0 R + k1), twiddles, then radix R3 over p0 of the bins j = k1 + R k2
    // = p + P i, which leaves bin j + R^2 k3 in register i + (R / R3) k3
    const int k1 = p & (R - 1), p0 = p / R;
    const int wb = (p & (R3 - 1)) * (R + 2) + p / R3, rb = k1 * RS + p0 * (R + 2);
    exchange<T, R, R, BY_PART>(v, lds, [&](int i) { return wb + i * RS; }, [&](int) { return rb; });
#pragma unroll
    for (int k = 1; k < R; ++k) w[0][k] = entry(t2, k * R3, p0);
    issued();
    static_assert(WB == R, "one batch");
    dft<T, R>(v);
#pragma unroll
    for (int k = 1; k < R; ++k) v[k] = cmul(v[k], w[0][k]);
    const int wb3 = p0 * Lay::RS3 + k1;
    constexpr int NI = R / R3;
    exchange<T, R, 1, BY_PART>(v, lds, [&](int i) { return wb3 + i * R; },
                      [&](int i) { return p + (i % NI) * P + (i / NI) * Lay::RS3; });
    mid();
    // register i + NI p0 holds sample p0 of butterfly i
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      C u[R3];
#pragma unroll
      for (int k = 0; k < R3; ++k) u[k] = v[i + NI * k];
      dft<T, R3>(u);
#pragma unroll
      for (int k = 0; k < R3; ++k) v[i + NI * k] = u[k];
    }
  } else {
    constexpr int CN = R / P;
    const int rb = p * RS;
    exchange<T, R, P, BY_PART>(v, lds, [&](int i) { return p + i * RS; }, [&](int i) { return rb + i * P * RS; });
    mid();
    C o[R];
#pragma unroll
    for (int i = 0; i < CN; ++i) {
      C u[P];
#pragma unroll
      for (int k = 0; k < P; ++k) u[k] = v[i * P + k];
      dft<T, P>(u);
#pragma unroll
      for (int k = 0; k < P; ++k) o[i + CN * k] = u[k];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = o[r];
  }
}

// Every requested lag's row of the workgroup's Q neighbouring columns, from
// the results by column and lag in LDS (column stride SS).  A lane writes up to
// 16 bytes of a row (4 or 2 columns) at once where the output is aligned for it.
template <typename OutT, int NT, int Q, int M>
struct LagRows {
  static constexpr int V = Q * sizeof(OutT) < 16 ? Q : static_cast<int>(16 / sizeof(OutT)), CG = Q / V;  // columns per lane, lanes per row
  static constexpr int STEP = NT / CG, B = 8;  // rows per round of the workgroup, rounds in flight
  static constexpr int SS = M + (CG > 1 ? 16 / CG : 0);  // the lanes of one row read LDS in different banks
  static_assert(Q % V == 0 && CG <= 16, "whole rows");
  typedef OutT Vec __attribute__((ext_vector_type(V)));

  static __device__ __forceinline__ void write(const TimeArgs& a, const OutT* stage, int c0, int tid) {
    const int cg = tid % CG, i0 = tid / CG, c = c0 + cg * V;
    const OutT* const st = stage + cg * V * SS;
    OutT* dst = static_cast<OutT*>(a.out) + static_cast<size_t>(i0) * a.ldo + col_out(a, c);
    const size_t step = STEP * a.ldo;
    const bool aligned = (reinterpret_cast<uintptr_t>(a.out) | (a.ldo * sizeof(OutT)) |
                          (col_out(a, c0) * sizeof(OutT))) % sizeof(Vec) == 0 && c0 + Q <= a.cols;  // uniform
    for (int ib = 0; ib < a.nl; ib += B * STEP) {
      uint32_t d[B];
#pragma unroll
      for (int b = 0; b < B; ++b) d[b] = a.lags[min(ib + i0 + b * STEP, a.nl - 1)];
      issued();
      Vec val[B];
#pragma unroll
      for (int b = 0; b < B; ++b)
#pragma unroll
        for (int k = 0; k < V; ++k) val[b][k] = st[d[b] + k * SS];
      if (aligned && ib + B * STEP <= a.nl) {
#pragma unroll
        for (int b = 0; b < B; ++b) {
          *reinterpret_cast<Vec*>(dst) = val[b];
          dst += step;
        }
      } else {
        const int left = a.nl - ib - i0;  // rows of this lane from here on: b STEP < left
#pragma unroll
        for (int b = 0; b < B; ++b) {
          if (b * STEP < left) {
            if (aligned) {
              *reinterpret_cast<Vec*>(dst) = val[b];
            } else {
#pragma unroll
              for (int k = 0; k < V; ++k)
                if (c + k < a.cols) dst[k] = val[b][k];
            }
          }
          dst += step;
        }
      }
    }
  }
};

// Host side: table entries of the compute type, exp(-2 pi i num / den).
inline void put_value(std::vector<unsigned char>& out, long double v, bool f64) {
  const double d = static_cast<double>(v);
  const float f = static_cast<float>(v);
  const unsigned char* b = f64 ? reinterpret_cast<const unsigned char*>(&d) : reinterpret_cast<const unsigned char*>(&f);
  out.insert(out.end(), b, b + (f64 ? 8 : 4));
}
inline void put_root(std::vector<unsigned char>& out, long long num, long long den, bool f64) {
  const long double ang = -6.283185307179586476925286766559005768L * static_cast<long double>(num) / static_cast<long double>(den);
  put_value(out, cosl(ang), f64);
  put_value(out, sinl(ang), f64);
}
// Tables of an M-point transform on P lanes: first stage (with the odd one), second stage.
inline void put_transform(std::vector<unsigned char>& out, long long M, long long P, bool f64, bool with_odd) {
  const long long R = M / P;
  for (long long k = 0; k < R; ++k)
    for (long long p = 0; p < P; ++p) put_root(out, p * k, M, f64);
  for (long long k = 0; with_odd && k < R; ++k)
    for (long long p = 0; p < P; ++p) put_root(out, p * (2 * k + 1), 2 * M, f64);
  if (P == 64 && R == 32) {
    for (long long j = 0; j < R; ++j) put_root(out, j, P, f64);
  } else if (P > R) {
    for (long long k = 0; k < R; ++k)
      for (long long p0 = 0; p0 < P / R; ++p0) put_root(out, p0 * k, P, f64);
  }
}
// 1 / (L - d), d < M, in double.
inline void put_reciprocals(std::vector<unsigned char>& out, long long M, uint64_t L) {
  for (uint64_t d = 0; d < static_cast<uint64_t>(M); ++d)
    put_value(out, d < L ? 1.0L / static_cast<long double>(L - d) : 0.0L, true);
}

}  // namespace tw
}  // namespace fddm
