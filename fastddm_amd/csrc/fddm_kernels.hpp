// Host-side launchers of the fastddm_amd kernels.
#pragma once

#include <vector>

#include "fddm_common.hpp"

namespace fddm {

// Stage (a), row pass.  Frames [0, L) of the (L, H, W) stack `img` (pixel
// type in_dtype) -> per-row half spectra along x, scaled by `norm`, stored in
// the blocked layout R[tb][kx][y][ti] (t = tb * Tb + ti, kx < nx/2+1, y < H).
// `window` (H*W of T) may be null.  subtract0: use I(t) - I0 in place of I(t),
// where I0 is the frame at img0 (the stack's frame 0; img itself when the
// launch starts at frame 0).  `frames` limits how many leading frames are
// transformed (>= 1).  In FP64 frames t >= split (a multiple of Tb) come from
// frame t + gap of img, and frame t == raw (even; none: 2^32 - 1) is frame 0 of
// img without the subtraction (BlockFrames in fddm_spatial.hpp).
struct RowArgs {
  const void* img;
  const void* img0;
  int in_dtype;
  uint64_t L;       // frames present (t < L; besides raw)
  uint64_t frames;  // frames to transform
  int H, W, nx, Tb, G;
  int logn;  // > 0: power-of-two kernel for nx = 2^logn (twx holds its tables)
  const void* window;
  int subtract0;
  double norm;
  FftDesc dx;
  const void* twx;
  void* R;
  int generic;  // 1: the generic workgroup kernel even where k_rows_mr applies
  uint32_t split = 0, gap = 0, raw = ~uint32_t(0);
};

// Stage (a) column pass + q-major store: R -> S[q][t], q = ky * nxh + kx,
// row pitch Lp (multiple of Tb).  Transforms blocks tb in [0, nblocks).
struct ColArgs {
  const void* R;
  uint64_t nblocks;
  int H, ny, nxh, Tb, G;
  int logn;  // > 0: power-of-two kernel for ny = 2^logn (twy holds its tables)
  uint64_t Lp;
  FftDesc dy;
  const void* twy;
  void* S;
  int generic;  // 1: the generic workgroup kernel even where k_cols_mr applies
};

// Stage (c)/(d): per-q time series -> D(q, lags), PS, VAR in the y-shifted
// output (NL+2, ny, nxh).
struct TimeArgs {
  const void* S;
  uint64_t Lp;
  int L, ny, nxh;
  const void* S0;  // frame-0 spectra (stride s0_stride, in double when s0_f64) or null
  uint64_t s0_stride;
  int s0_f64;
  const uint32_t* lags;
  int nl;
  FftDesc dt;
  const void* twt;
  void* out;
  unsigned char* flags;  // fft mode, compensated FP32: per q, 1 = some lag needs launch_fix
  // Columns of this launch, c in [0, cols).  local = 0: column c is output
  // column c0 + c of the y-shifted plane (row pitch ldo) and reads the q at
  // that position; local = 1: column c reads q = c0 + c and is stored
  // unshifted at out[i ldo + c].  S holds the rows of q >= s_q0 (row q - s_q0).
  int c0, cols, local;
  uint64_t ldo;
  int s_q0;
};

// Whole-plane launch: every q, y-shifted output of row pitch ny (nx/2+1).
inline void time_full(TimeArgs& a) {
  a.c0 = 0;
  a.cols = a.ny * a.nxh;
  a.local = 0;
  a.ldo = static_cast<uint64_t>(a.ny) * a.nxh;
  a.s_q0 = 0;
}

// q read by column c of a launch, and the column's output offset in a row.
__device__ __forceinline__ int col_q(const TimeArgs& a, int c) {
  if (a.local) return a.c0 + c;
  const int o = a.c0 + c, yo = o / a.nxh, kx = o - yo * a.nxh;
  return ((yo + a.ny - a.ny / 2) % a.ny) * a.nxh + kx;
}
__device__ __forceinline__ size_t col_out(const TimeArgs& a, int c) {
  return static_cast<size_t>(a.local ? c : a.c0 + c);
}

// F(0) of the raw first frame at q, in the compute type (zero without S0).
template <typename C>
__device__ __forceinline__ C frame0_spectrum(const TimeArgs& a, int q) {
  if (!a.S0) return C{0, 0};
  const size_t i = static_cast<size_t>(q) * a.s0_stride;
  if (!a.s0_f64) return static_cast<const C*>(a.S0)[i];
  const double2 z = static_cast<const double2*>(a.S0)[i];
  using T = decltype(C{}.x);
  return C{static_cast<T>(z.x), static_cast<T>(z.y)};
}

hipError_t launch_rows(const RowArgs& a, int precision, hipStream_t s);
hipError_t launch_cols(const ColArgs& a, int precision, hipStream_t s);
hipError_t launch_diff(const TimeArgs& a, int precision, int out_dtype, hipStream_t s);
// Time kernel with a column's transforms in LDS (fddm_time_p2.hip), N = 2^logn,
// logn in [kTimeMinLog, kShortMaxLog] or time_p2_log.
int time_p2_log(int precision);
hipError_t launch_time_p2(const TimeArgs& a, int logn, int precision, int out_dtype, hipStream_t s);
// Time kernel with every transform in the registers of one wave
// (fddm_time_wave.hip): M = 2^logm samples (zero-padded, M >= L), logm in
// [7, time_wave_max_log].  time_wave_tables: the tables it reads from a.twt.
int time_wave_max_log(int precision);
std::vector<unsigned char> time_wave_tables(int logm, int precision, uint64_t L);
hipError_t launch_time_wave(const TimeArgs& a, int logm, int precision, int out_dtype, hipStream_t s);
// The same with a column's even and odd bins on two waves
// (fddm_time_pair.hip), M = 2^time_pair_log samples.
int time_pair_log(int precision);
std::vector<unsigned char> time_pair_tables(int precision, uint64_t L);
hipError_t launch_time_pair(const TimeArgs& a, int precision, int out_dtype, hipStream_t s);
// Power-of-two spatial kernels (256 <= n <= 4096): plan radices and launchers.
bool p2_spatial_ok(int logn);
int p2_spatial_plan(int logn, bool cols, int* r0, int* r1, int* r2);
hipError_t launch_rows_p2(const RowArgs& a, int precision, hipStream_t s);
hipError_t launch_cols_p2(const ColArgs& a, int precision, hipStream_t s);
// Mixed-radix row kernel (a frame pair's row on a wave, a half or a quarter of
// one, 2 <= nx <= 2048, Tb 4, 8 or 16); launch_rows uses it where rows_mr_ok holds.
bool rows_mr_ok(const RowArgs& a, int precision);
hipError_t launch_rows_mr(const RowArgs& a, int precision, hipStream_t s);
// Mixed-radix column kernel (one wave per frame of the block, 256 <= ny <= 2048,
// in FP64 up to 768); launch_cols uses it where cols_mr_ok holds.
bool cols_mr_ok(const ColArgs& a, int precision);
hipError_t launch_cols_mr(const ColArgs& a, int precision, hipStream_t s);
hipError_t launch_fft_test(void* data, int n, int batch, const FftDesc& d, const void* tw,
                           int precision, hipStream_t s);

// n bytes from device memory to pinned host memory addressed by the device
// (hipHostGetDevicePointer), by a kernel; n and both addresses multiples of 16.
hipError_t launch_copy_out(void* dst, const void* src, uint64_t n, hipStream_t s);

// Corrections of the compensated path (fddm_edge.hip), in the y-shifted
// output: the lags lags[i0 .. nl) (n = L - dt <= E pairs) by direct sums from
// the FP64 spectra S64[q][c] (pitch lp; null: none) of the first and last E
// frames; of the q marked in a.flags (null: none) the lags with (L - dt) D <
// kWkFlag L VAR and L - dt > 32 by direct differences of the float series
// S[q][t] (pitch Lp) in double.
constexpr int kEdgeFrames = 8;
// What the float transforms leave in (L - dt) D, against direct differences of
// the same float spectra: at most 1.4e-7 sum |G|^2 on white noise (8e8 cells) and
// 5.6e-7 on slow speckle (1.2e8 cells, 120 to 4000 frames), with transforms in
// registers (fddm_time_wave.hip, fddm_time_pair.hip) as in LDS (fddm_time_p2.hip:
// 6.2e-7).  So a lag that is not marked is off by 2.8e-4 at most; 1.7e-4 was the
// largest found.
constexpr double kWkFlag = 2e-3;
hipError_t launch_fix(const TimeArgs& a, const void* S64, uint64_t lp, int E, int i0, int out_dtype, hipStream_t s);

// Time stage for series longer than the LDS-resident plans allow
// (fddm_time_long.hip): N = 2^logn in (2^12, 2^long_max_log] as a four-step
// transform, one workgroup per q at a time, each with a scratch slot of
// long_slot_bytes in `scratch` (slots slots).  long_twiddles: the table the
// kernel reads from a.twt (complex, converted to the compute type).
int long_max_log(int precision);
uint64_t long_slot_bytes(int logn, int precision, uint64_t L);
std::vector<double> long_twiddles(int logn);
hipError_t launch_time_long(const TimeArgs& a, int logn, int precision, int out_dtype, void* scratch,
                            uint64_t slot_bytes, int slots, hipStream_t s);

// Elements-per-thread template bucket for a transform of `work` points
// cooperatively done by 256 threads; 0 if too large.
int fft_bucket(long long work);

}  // namespace fddm
