// Shared device/host helpers for the gfx950 CSR step library.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <cmath>

#include "dfcsr.h"

#define DFCSR_WAVE 64

namespace dfcsr {

// Records the message for dfcsr_last_error() and returns code.
int set_error(int code, const char *fmt, ...);

#define DFCSR_CHECK_HIP(expr)                                                    \
  do {                                                                           \
    hipError_t _e = (expr);                                                      \
    if (_e != hipSuccess)                                                        \
      return ::dfcsr::set_error(DFCSR_EHIP, "%s failed: %s", #expr,              \
                                hipGetErrorString(_e));                          \
  } while (0)

#define DFCSR_LAUNCH_CHECK(name)                                                 \
  do {                                                                           \
    hipError_t _e = hipGetLastError();                                           \
    if (_e != hipSuccess)                                                        \
      return ::dfcsr::set_error(DFCSR_EHIP, "launch of %s failed: %s", name,     \
                                hipGetErrorString(_e));                          \
  } while (0)

// launch(first, n) for each launch of `blocks` workgroups of `threads`: a launch
// of 2^32 threads or more (along x) runs the remainder alone, with no error, so
// they are cut at 2^31.
template <typename F>
void launch_blocks(int64_t blocks, int threads, const F &launch) {
  const int64_t most = ((int64_t)1 << 31) / threads;
  for (int64_t at = 0; at < blocks; at += most)
    launch((int)at, (unsigned)(blocks - at < most ? blocks - at : most));
}

// np.linspace(start, stop, num)[i]: y = i*step + start with step =
// (stop - start)/(num - 1), two roundings (no fused multiply-add), and the
// last point pinned to stop.  num == 1 gives start.
__host__ __device__ inline double linspace_at(double start, double stop, int num, int i) {
#pragma clang fp contract(off)
  if (num <= 1) return start;
  if (i == num - 1) return stop;
  double step = (stop - start) / (double)(num - 1);
  double y = (double)i * step;
  return y + start;
}

// Index rule of pyDFCSR's interpolate3D / interpolate1D (interp3D.py:30-52):
// i0 = int(u) (truncation), i1 = i0 at the last plane else i0 + 1, valid iff
// i0 >= 0 and i1 < size.  Equivalent to -1 < u < size; NaN is invalid.
struct TruncIdx {
  int i0, i1;
  double frac;
  bool ok;
};

__host__ __device__ inline TruncIdx trunc_index(double u, int size) {
#pragma clang fp contract(off)
  TruncIdx r;
  r.ok = (u > -1.0) && (u < (double)size);
  double f = r.ok ? trunc(u) : 0.0;
  r.i0 = (int)f;
  r.i1 = (r.i0 == size - 1) ? r.i0 : r.i0 + 1;
  r.frac = r.ok ? (u - f) : 0.0;
  return r;
}

// Interval search of scipy's RegularGridInterpolator on a linspace axis:
// the i with g[i] <= v < g[i+1], clipped to [0, num-2] (v == g[num-1] gives
// num-2), using the exact linspace values.  Caller handles out-of-bounds.
__host__ __device__ inline int rgi_interval(double v, double g0, double g1, int num) {
#pragma clang fp contract(off)
  double step = (g1 - g0) / (double)(num - 1);
  double u = (v - g0) / step;
  int i = (u >= 0.0) ? (int)u : 0;
  if (i > num - 2) i = num - 2;
  if (i < 0) i = 0;
  while (i > 0 && linspace_at(g0, g1, num, i) > v) --i;
  while (i < num - 2 && linspace_at(g0, g1, num, i + 1) <= v) ++i;
  return i;
}

// Lane exchanges of a double as register moves (permlane swaps between and
// within the halves of a wave, DPP rotations within a row of 16 lanes), not
// through the LDS unit as ds_bpermute: a wave's sum is 18 vector
// instructions, and the waves of a workgroup do not queue for the LDS.  Every
// lane of the wave takes part.
typedef unsigned Words __attribute__((ext_vector_type(2)));

__device__ inline double from_words(unsigned lo, unsigned hi) {
  return __hiloint2double((int)hi, (int)lo);
}

// a <- (lower half of a, lower half of b), b <- (upper half of a, of b)
__device__ inline void swap_halves(double &a, double &b) {
  const Words lo = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                    (unsigned)__double2loint(b), false, false);
  const Words hi = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                    (unsigned)__double2hiint(b), false, false);
  a = from_words(lo[0], hi[0]);
  b = from_words(lo[1], hi[1]);
}

// rows (16 lanes) 0..3: a <- (a0, b0, a2, b2), b <- (a1, b1, a3, b3)
__device__ inline void swap_rows(double &a, double &b) {
  const Words lo = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                    (unsigned)__double2loint(b), false, false);
  const Words hi = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                    (unsigned)__double2hiint(b), false, false);
  a = from_words(lo[0], hi[0]);
  b = from_words(lo[1], hi[1]);
}

// v of the lane N below in the row, cyclic
template <int N>
__device__ inline double row_rotate(double v) {
  const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), 0x120 + N, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), 0x120 + N, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// Sum of a row's 16 lanes, in each of them.
__device__ inline double row_sum(double v) {
  v += row_rotate<8>(v);
  v += row_rotate<4>(v);
  v += row_rotate<2>(v);
  v += row_rotate<1>(v);
  return v;
}

__device__ inline double wave_sum(double v) {
  double u = v;
  swap_halves(v, u);
  v += u;
  u = v;
  swap_rows(v, u);
  return row_sum(v + u);
}

// Sums over the wave of four values with the moves of one and a half: row r
// of the result holds the sum of value wave_sum4_of(r).
__device__ inline double wave_sum4(double a, double b, double c, double d) {
  swap_halves(a, b);
  a += b;
  swap_halves(c, d);
  c += d;
  swap_rows(a, c);
  return row_sum(a + c);
}
__device__ inline int wave_sum4_of(int row) { return (row >> 1) | ((row & 1) << 1); }

__device__ inline double wave_max(double v) {
  double u = v;
  swap_halves(v, u);
  v = fmax(v, u);
  u = v;
  swap_rows(v, u);
  v = fmax(v, u);
  v = fmax(v, row_rotate<8>(v));
  v = fmax(v, row_rotate<4>(v));
  v = fmax(v, row_rotate<2>(v));
  return fmax(v, row_rotate<1>(v));
}

// Deterministic block sum (fixed tree), result valid in all threads.
// smem: at least blockDim.x/64 doubles.
__device__ inline double block_sum(double v, double *smem) {
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  double r = 0.0;
  for (int i = 0; i < nw; ++i) r += smem[i];
  __syncthreads();
  return r;
}

__device__ inline double block_max(double v, double *smem) {
  int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) smem[wid] = v;
  __syncthreads();
  double r = smem[0];
  for (int i = 1; i < nw; ++i) r = fmax(r, smem[i]);
  __syncthreads();
  return r;
}

inline hipStream_t as_stream(void *s) { return reinterpret_cast<hipStream_t>(s); }

}  // namespace dfcsr
