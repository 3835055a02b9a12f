// Stages (c) + (e), fft mode, for series of 2049 to 4096 frames (FP32) and
// 1025 to 2048 (FP64): one column on two waves.
//
// As in fddm_time_wave.hip, the zero-padded transform of length N = 2M splits
// into its even and odd bins, two M-point transforms of the M samples; here
// one wave computes the even bins and another the odd ones, R = M / 64 points
// per lane, because the registers of one wave do not hold one of them beside
// the other's result.  Re C(d) splits the same way, with P_e(m) = |G(2m)|^2 and
// P_o(m) = |G(2m + 1)|^2:
//   Re C(d) N = a(d) + b(d),  a(d) = Re FFT_M(P_e)(d),  b(d) = Re W_N^d FFT_M(P_o)(d),
//   a(M - d) = a(d),  b(M - d) = -b(d).
// Each wave transforms its real sequence as M / 2 complex points, Z = FFT of
// P(2n) + i P(2n + 1), and untangles its a or b for d < M / 2 from Z(d) and
// Z(M / 2 - d).  The waves trade these through LDS; the even wave then forms D
// of the lags below M / 2, the odd one of those above.
//
// Bound: VALU issue (60 % busy in FP32, 48 % in FP64), and the scattered lag
// rows: 16-byte pieces of rows half a megabyte apart leave at about 110 G
// pieces per second (a write-only probe), 1.2 of 5.3 ms for 131584 columns of
// 4000 FP32 samples and lags.  Eight waves per workgroup (four columns, one
// workgroup per CU) write longer pieces than four and measured faster in FP32
// (20.8 -> 19.9 ms at 525312 columns); in FP64 two workgroups of four waves
// overlap better (3.4 -> 3.0 ms).  A persistent form that read the next
// series ahead was slower (2.4 against 1.8 ms in fddm_time_wave.hip at 2000
// samples): its loads queue behind the stores.
// Kernel time against the workgroup form (fddm_time_p2.hip at these lengths):
// 22.3 -> 18.5 ms for 525312 columns of 4000 samples in compensated FP32, 5.46
// -> 3.0 ms for 131584 of 2000 in FP64.
#include <vector>

#include "fddm_time_wave.hpp"

namespace fddm {
namespace {
using namespace tw;

template <typename T, int R_, int W_>
struct PairLay {
  using C = cplx_t<T>;
  static constexpr int R = R_, P = 64, M = R * P, H = M / 2, R2 = R / 2;
  using First = WaveLay<R, P>;
  using Second = WaveLay<R2, P>;
  static constexpr int W = W_, Q = W / 2;  // waves and columns per workgroup
  // 8-byte elements per wave: an exchange of the first transform (by parts),
  // P, Z, a or b, and half of the column's samples or prefix sums
  static constexpr int REG = 2176;
  static_assert(R * First::RS * sizeof(T) * (sizeof(T) == 4 ? 1 : 2) <= REG * 8 && M * sizeof(T) <= REG * 8, "REG");
  static_assert(Second::GS <= REG && H <= REG, "REG");
  // sample chunks of R2: 16 bytes of padding each; prefix sums: two doubles
  static constexpr int XC = R2 + 16 / sizeof(C), CS = R2 + 2;
  static_assert(128 * XC * sizeof(C) <= 2 * REG * 8 && 128 * CS <= 2 * REG, "REG");
  static constexpr int EXTRA = kLast * sizeof(C) / 8 + 2;  // last samples, total, flag
  static constexpr size_t bytes = sizeof(double) * W * (REG + EXTRA);
  // tables: W_M^(p k1), W_M^(p (k1 + 1/2)), second stage; the same of FFT_H
  // (even only); (cos, sin)(2 pi d / M), (2 pi d / N), (6 pi d / N) for d < M / 4;
  // in double 1 / (L - d) for d < M
  static constexpr int T_E = 0, T_O = M, T_2 = 2 * M, T_H = T_2 + (First::LANE2 ? R : 0);
  static constexpr int T_H2 = T_H + H, T_CS = T_H2 + (Second::LANE2 ? R2 : Second::R3 > 1 ? P : 0);
  static constexpr int T_END = T_CS + 3 * (M / 4);
};

template <int PAD, int R>
__host__ __device__ __forceinline__ int padded(int t) {
  constexpr int LR = R == 32 ? 5 : 4;
  static_assert(R == 1 << LR, "R");
  return t + (t >> LR) * PAD;
}

template <typename T, typename OutT, int R, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2, 2)))
    k_time_pair(TimeArgs a, int wg_per_xcd, int wgs, int subtract_mean) {
  using C = cplx_t<T>;
  using Lay = PairLay<T, R, W>;
  constexpr int M = Lay::M, H = Lay::H, R2 = Lay::R2, R4 = R / 4, Q = Lay::Q;
  constexpr bool F64 = sizeof(T) == 8;

  extern __shared__ __align__(16) unsigned char smem[];

  const int wgi = (blockIdx.x & 7) * wg_per_xcd + (blockIdx.x >> 3);  // XCD-contiguous columns
  if (wgi >= wgs) return;                                             // whole workgroup: before any barrier
  const int tid = threadIdx.x, p = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int e = wave & 1, qi = wave >> 1;  // 0: even bins, 1: odd bins; column of the workgroup
  const int c0 = wgi * Q;
  const bool active = c0 + qi < a.cols;
  const int c = active ? c0 + qi : a.cols - 1;  // (an idle pair repeats the last column and stores nothing)
  const int q = __builtin_amdgcn_readfirstlane(col_q(a, c));
  const int L = a.L;
  const C* __restrict__ src = static_cast<const C*>(a.S) + static_cast<size_t>(q - a.s_q0) * a.Lp;
  const C* __restrict__ tab = static_cast<const C*>(a.twt);
  const double* __restrict__ inv = reinterpret_cast<const double*>(tab + Lay::T_END);
  double* const base = reinterpret_cast<double*>(smem);
  double* const mine = base + wave * Lay::REG;
  double* const pair = base + (wave - e) * Lay::REG;  // both waves' regions
  double* const extra = base + W * Lay::REG + wave * Lay::EXTRA;
  double* const total = extra + Lay::EXTRA - 2;
  double* const pair_total = total - e * Lay::EXTRA;
  const double rl = inv[0];

  // 1. the whole series on either wave, without its mean (compensated paths)
  C v[R];
#pragma unroll
  for (int r = 0; r < R; ++r) v[r] = r < R2 ? entry(src, 64 * r, p) : entry(src, 0, min(p + 64 * r, L - 1));
  const C first = frame0_spectrum<C>(a, q);  // F(0) of the raw first frame
  issued();
#pragma unroll
  for (int r = R2; r < R; ++r) v[r] = p + 64 * r < L ? v[r] : C{0, 0};
  double sr = 0, si = 0;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    sr += static_cast<double>(v[r].x);
    si += static_cast<double>(v[r].y);
  }
  sr = group_last<64>(group_scan<64>(sr, p));
  si = group_last<64>(group_scan<64>(si, p));
  T m_r = 0, m_i = 0;
  if (subtract_mean) {
    m_r = static_cast<T>(sr * rl);
    m_i = static_cast<T>(si * rl);
  }
  // sum of the subtracted series, for VAR and PS
  const double fsr = sr - static_cast<double>(L) * static_cast<double>(m_r);
  const double fsi = si - static_cast<double>(L) * static_cast<double>(m_i);
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const C f{v[r].x - m_r, v[r].y - m_i};
    v[r] = r < R2 || p + 64 * r < L ? f : C{0, 0};
  }

  // 2. |G|^2 of this wave's bins, then Z of them as P(2n) + i P(2n + 1)
  wave_fft<T, typename Lay::First>(v, mine, tab + (e ? Lay::T_O : Lay::T_E), tab + Lay::T_2, p, e != 0, [] {});
  C z[R2];
  {
    T* const b = reinterpret_cast<T*>(mine);
#pragma unroll
    for (int r = 0; r < R; ++r) b[p + 64 * r] = v[r].x * v[r].x + v[r].y * v[r].y;
    wave_sync();
    const C* const bz = reinterpret_cast<const C*>(mine);
#pragma unroll
    for (int r = 0; r < R2; ++r) z[r] = bz[p + 64 * r];
    wave_sync();
  }
  C w1[R4], w3[R4];
  wave_fft<T, typename Lay::Second>(z, mine, tab + Lay::T_H, tab + Lay::T_H2, p, std::false_type{}, [&] {
    const C* const t1 = tab + Lay::T_CS + (e ? M / 4 : 0);
#pragma unroll
    for (int r = 0; r < R4; ++r) w1[r] = entry(t1, 64 * r, p);
    if (e) {
#pragma unroll
      for (int r = 0; r < R4; ++r) w3[r] = entry(tab + Lay::T_CS, M / 2 + 64 * r, p);
    }
    issued();
  });

  // 3. 2 a or 2 b at u = p + 64 r < M / 4 (va) and M / 2 - u (vb), from
  // A = Z(u), B = Z(M / 2 - u) (lane 64 - p, register R2 - 1 - r; lane 0:
  // register R2 - r), (c1, s1), (c3, s3):
  //   2 a = A.x + B.x +- (c1 (A.y + B.y) - s1 (A.x - B.x))
  //   2 b(u) = c1 (A.x + B.x) + s1 (A.y - B.y) + c3 (A.y + B.y) - s3 (A.x - B.x)
  //   2 b(M / 2 - u) = s1 (A.x + B.x) - c1 (A.y - B.y) - s3 (A.y + B.y) - c3 (A.x - B.x)
  // Lane 0, r = 0 holds u = 0 only for M / 2; its va is that of M / 4 instead,
  // A = B = Z(M / 4) with the angles pi / 2, pi / 4 and 3 pi / 4.
  double va[R4], vb[R4];
  {
    const int other = ((64 - p) & 63) * 4;
    constexpr T h = static_cast<T>(0.70710678118654752440084436210485);
    const double qx = z[R4].x, qy = z[R4].y;
    constexpr int B = 4;  // values fetched from other lanes at once
#pragma unroll
    for (int rb = 0; rb < R4; rb += B) {
      C o[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int r = rb + i, r0 = r == 0 ? 0 : R2 - r;
        o[i].x = from_lane(p == 0 ? z[r0].x : z[R2 - 1 - r].x, other);
        o[i].y = from_lane(p == 0 ? z[r0].y : z[R2 - 1 - r].y, other);
      }
      issued();
      if (e == 0) {
#pragma unroll
        for (int i = 0; i < B; ++i) {
          const int r = rb + i;
          const double ax = z[r].x, ay = z[r].y, bx = o[i].x, by = o[i].y, c1 = w1[r].x, s1 = w1[r].y;
          const double sx = ax + bx, w = c1 * (ay + by) - s1 * (ax - bx);
          va[r] = sx + w;
          vb[r] = sx - w;
        }
      } else {
#pragma unroll
        for (int i = 0; i < B; ++i) {
          const int r = rb + i;
          const double ax = z[r].x, ay = z[r].y, bx = o[i].x, by = o[i].y;
          const double c1 = w1[r].x, s1 = w1[r].y, c3 = w3[r].x, s3 = w3[r].y;
          const double sx = ax + bx, dx = ax - bx, sy = ay + by, dy = ay - by;
          va[r] = c1 * sx + s1 * dy + (c3 * sy - s3 * dx);
          vb[r] = s1 * sx - c1 * dy - (s3 * sy + c3 * dx);
        }
      }
    }
    va[0] = p == 0 ? (e ? 2 * static_cast<double>(h) * (qx - qy) : 2 * qx) : va[0];
#pragma unroll
    for (int r = 0; r < R4; ++r) {
      mine[p + 64 * r] = va[r];
      mine[p + 64 * (R4 + r)] = vb[r];
    }
  }
  // this wave's half of the series again, for the prefix sums
  C x[R2];
  {
    const int t0 = e * H + p;
#pragma unroll
    for (int r = 0; r < R2; ++r) x[r] = entry(src, 0, min(t0 + 64 * r, L - 1));
    issued();
  }
  __syncthreads();
  {
    const double* const o = pair + (1 - e) * Lay::REG;
    const double sg = e ? -1.0 : 1.0;
#pragma unroll
    for (int r = 0; r < R4; ++r) {
      va[r] = o[p + 64 * r] + sg * va[r];
      vb[r] = o[p + 64 * (R4 + r)] + sg * vb[r];
    }
  }
  __syncthreads();

  // 4. prefix sums of |x|^2 over both waves and the lags with few pairs (four
  // lanes share a lag's pairs)
  double ptot, de = 0;
  double ia[R4], ib[R4];  // 1 / (L - d)
  {
    C* const xs = reinterpret_cast<C*>(pair);
    constexpr int XP = 16 / sizeof(C);
    const int t0 = e * H + p, wb = padded<XP, R2>(t0), ch = e * 64 + p;
#pragma unroll
    for (int r = 0; r < R2; ++r) {
      const C f{x[r].x - m_r, x[r].y - m_i};
      xs[wb + r * (64 / R2) * Lay::XC] = t0 + 64 * r < L ? f : C{0, 0};
    }
    __syncthreads();
    {
      C* const last = reinterpret_cast<C*>(extra);
      static_assert(kLast == 64, "one per lane");
      last[p] = p < kEdge ? xs[padded<XP, R2>(L - kEdge + p)] : C{0, 0};
      wave_sync();
      few_pairs<4, 4>(de, ch / 4 + 1, ch % 4, kEdge, static_cast<const C*>(last), static_cast<const C*>(xs),
                      [](int t0) { return padded<XP, R2>(t0); }, [](C u, C w) {
                        const double dr = static_cast<double>(u.x) - static_cast<double>(w.x);
                        const double di = static_cast<double>(u.y) - static_cast<double>(w.y);
                        return dr * dr + di * di;
                      });
      de += __shfl_xor(de, 1, 64);
      de += __shfl_xor(de, 2, 64);
    }
    double s[R2];
    double run = 0;
    {
      const C* const rx = xs + ch * Lay::XC;
      constexpr int V = 16 / sizeof(C);
      struct alignas(16) Vec {
        C c[V];
      };
#pragma unroll
      for (int i = 0; i < R2; i += V) {
        const Vec f = *reinterpret_cast<const Vec*>(rx + i);
#pragma unroll
        for (int k = 0; k < V; ++k) {
          const double fx = f.c[k].x, fy = f.c[k].y;
          s[i + k] = fx * fx + fy * fy;
          run += s[i + k];
        }
      }
    }
    const double inc = group_scan<64>(run, p);
    if (p == 63) *total = inc;
    __syncthreads();
    const double first = pair_total[0];
    ptot = first + pair_total[Lay::EXTRA];
    double acc = inc - run + (e ? first : 0.0);
    double* const rb = pair + ch * Lay::CS;
#pragma unroll
    for (int i = 0; i < R2; i += 2) {
      const double e0 = acc, e1 = e0 + s[i];
      acc = e1 + s[i + 1];
      *reinterpret_cast<f64x2*>(rb + i) = f64x2{e0, e1};
    }
#pragma unroll
    for (int r = 0; r < R4; ++r) {
      // u and M / 2 - u, or M - u and M / 2 + u (lane 0, r = 0: M / 4 in place of u = 0)
      const int u = r == 0 && p == 0 ? M / 4 : p + 64 * r;
      ia[r] = entry(inv, 0, e ? M - u : u);
      ib[r] = entry(inv, 0, r == 0 && p == 0 ? H : e ? H + u : H - u);
    }
    issued();
  }
  __syncthreads();

  // 5. D as in fddm_time_wave.hip
  bool flag = false;
  {
    const double thr = ptot * kWkFlag;
    constexpr double k = -0.5 / M;
    constexpr int ROW = (64 / R2) * Lay::CS;
    const int sg = e ? -1 : 1;
    const int p1 = e ? M - p : p, p2 = e ? H + p : H - p;  // lags of r = 0
    const int tail1 = padded<2, R2>(p1), tail2 = padded<2, R2>(p2);
    const int head1 = padded<2, R2>(L - p1), head2 = padded<2, R2>(L - p2);
    auto value = [&](double cc, int d, double tail, double head, double rn) {
      const double num = head + (ptot - tail) + k * cc;
      if constexpr (!F64) flag |= num < thr && d < L - kEdge;
      return num * rn;
    };
    constexpr int B = 4;  // lag pairs whose sums are read at once
#pragma unroll
    for (int rb = 0; rb < R4; rb += B) {
      double t1[B], h1[B], t2[B], h2[B];
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int s = sg * (rb + i);  // lags p1 + 64 s and p2 - 64 s
        int t = tail1 + ROW * s, hd = max(head1 - ROW * s, 0);
        if (rb + i == 0) {
          const int d = e ? M - M / 4 : M / 4;
          t = p == 0 ? padded<2, R2>(d) : t;
          hd = p == 0 ? padded<2, R2>(max(L - d, 0)) : hd;
        }
        t1[i] = pair[t];
        h1[i] = pair[hd];
        t2[i] = pair[tail2 - ROW * s];
        h2[i] = pair[max(head2 + ROW * s, 0)];
      }
      issued();
#pragma unroll
      for (int i = 0; i < B; ++i) {
        const int r = rb + i, s = sg * r;
        const int d1 = r == 0 && p == 0 ? (e ? M - M / 4 : M / 4) : p1 + 64 * s;
        va[r] = value(va[r], d1, t1[i], h1[i], ia[r]);
        vb[r] = value(vb[r], p2 - 64 * s, t2[i], h2[i], ib[r]);
      }
    }
  }
  if constexpr (!F64) {
    const bool any = __ballot(flag) != 0;  // (by every lane: outside the branch)
    if (p == 0) total[1] = any ? 1.0 : 0.0;
  }
  OutT* __restrict__ out = static_cast<OutT*>(a.out);
  const size_t ldo = a.ldo;
  if (active && e == 0 && p == 0) {
    const size_t oq = col_out(a, c);
    const double mr2 = fsr * rl, mi2 = fsi * rl;
    const double var = ptot * rl - (mr2 * mr2 + mi2 * mi2);
    const double fr = static_cast<double>(m_r) + mr2 + static_cast<double>(first.x);
    const double fi = static_cast<double>(m_i) + mi2 + static_cast<double>(first.y);
    const double ps = var + fr * fr + fi * fi;
    out[static_cast<size_t>(a.nl) * ldo + oq] = static_cast<OutT>(ps);
    out[static_cast<size_t>(a.nl + 1) * ldo + oq] = static_cast<OutT>(var);
  }

  using Rows = LagRows<OutT, 64 * W, Q, M>;
  static_assert(Q * Rows::SS * sizeof(OutT) <= Lay::bytes, "results fit the exchange buffers");

  // 6. results to LDS by column and lag, then every requested lag's row
  __syncthreads();
  if constexpr (!F64) {
    if (a.flags && active && e == 0 && p == 0) a.flags[q] = total[1] + total[1 + Lay::EXTRA] != 0.0;
  }
  OutT* const stage = reinterpret_cast<OutT*>(smem);
  {
    OutT* const st = stage + qi * Rows::SS;
#pragma unroll
    for (int r = 0; r < R4; ++r) {
      const int u = r == 0 && p == 0 ? M / 4 : p + 64 * r;
      st[e ? M - u : u] = static_cast<OutT>(va[r]);
      st[r == 0 && p == 0 ? H : e ? H + u : H - u] = static_cast<OutT>(vb[r]);
    }
    __syncthreads();  // (the direct sums replace values of either wave)
    const int ch = e * 64 + p, n = ch / 4 + 1;
    if (ch % 4 == 0) st[L - n] = static_cast<OutT>(de / n);
  }
  __syncthreads();
  Rows::write(a, stage, c0, tid);
}

template <typename T, typename OutT, int R, int W>
hipError_t launch_one(const TimeArgs& a, bool subtract_mean, hipStream_t s) {
  using Lay = PairLay<T, R, W>;
  if (a.cols <= 0) return hipSuccess;
  const int wgs = (a.cols + Lay::Q - 1) / Lay::Q;
  const int wpx = (wgs + 7) / 8;
  auto kernel = k_time_pair<T, OutT, R, W>;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     static_cast<int>(Lay::bytes));
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kernel, dim3(8u * wpx), dim3(64 * W), Lay::bytes, s, a, wpx, wgs, subtract_mean ? 1 : 0);
  return hipGetLastError();
}

}  // namespace

int time_pair_log(int precision) { return precision == PREC_FP64 ? 11 : 12; }

std::vector<unsigned char> time_pair_tables(int precision, uint64_t L) {
  const bool f64 = precision == PREC_FP64;
  const int logm = time_pair_log(precision);
  const long long M = 1ll << logm, H = M / 2;
  std::vector<unsigned char> out;
  put_transform(out, M, 64, f64, true);
  put_transform(out, H, 64, f64, false);
  for (int k : {2, 1, 3})
    for (long long d = 0; d < M / 4; ++d) put_root(out, -k * d, 2 * M, f64);
  put_reciprocals(out, M, L);
  return out;
}

hipError_t launch_time_pair(const TimeArgs& a, int precision, int out_dtype, hipStream_t s) {
  const bool f32 = out_dtype == OUT_F32;
  switch (precision) {
    case PREC_FP64: return f32 ? launch_one<double, float, 32, 4>(a, true, s) : launch_one<double, double, 32, 4>(a, true, s);
    case PREC_FP32:
    case PREC_FP32C: {
      const bool sub = precision == PREC_FP32C;
      return f32 ? launch_one<float, float, 64, 8>(a, sub, s) : launch_one<float, double, 64, 8>(a, sub, s);
    }
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fddm
