// a8-a10: re-gridding of density-function slices into the device history.
//
// Replaces DF_tracker.DF_interp (deposit.py:296-309) as used by
// append_interpolant for the new slice (deposit.py:328-337) and for a full
// re-grid of every logged slice (deposit.py:379-390).  Each target point
// (xi, zi) of the common interp grid takes scipy RegularGridInterpolator's
// linear value on the slice's own linspace grids: interval search, norm
// distances y0, y1 and the corner sum
//   v00(1-y0)(1-y1) + v01(1-y0)y1 + v10 y0(1-y1) + v11 y0 y1,
// with fill 0 outside the grid (mean(vx_x) of the slice for vx_x).
//
// History layout: corner-packed records (record (x, z) holds field f at
// (x, z), (x, z1), (x1, z), (x1, z1) in elements f*4 + 0..3, x1 and z1
// clamped to the last plane).  float64: whole records [x][z][slot][20];
// float32 chunked: 16-byte chunks (one field's four corners each) stored
// [x][slot][f][z], where threads of consecutive z write consecutive chunks;
// float32 time-innermost: whole records [x][z][slot][20].  Any of the three
// rings may be absent.
#include "common.h"

namespace dfcsr {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxJobs = 4096;

// Jobs of one launch, as a kernel argument: no copy of them on the stream.  A
// step has one or two; a whole history's go 64 a launch (3 KB of the 4 KB that
// arguments may take), or a small grid's launches would be all its time: 64
// slices onto 37 x 70 52 us with 16 a launch, 31 with 64.
constexpr int kJobs = 16, kManyJobs = 64;
template <int kN>
struct RegridJobs {
  DfcsrRegridJob j[kN];
};
static_assert(sizeof(RegridJobs<kManyJobs>) <= 3072, "kernel arguments");

// per-job mean of the raw vx_x field (np.mean(vx_x), deposit.py:332, 384):
// one workgroup a job, wide enough that a 100 x 100 slice is ten loads in
// flight a thread (12 us as 256 threads, 4 us now)
constexpr int kMeanThreads = 1024;

template <int kN>
__global__ __launch_bounds__(kMeanThreads) void vxx_mean_kernel(const double *__restrict__ src,
                                                                int64_t slot_stride,
                                                                RegridJobs<kN> jobs,
                                                                double *__restrict__ means) {
  __shared__ double red[kMeanThreads / 64];
  const DfcsrRegridJob &J = jobs.j[blockIdx.x];
  const int64_t N = (int64_t)J.nbx * J.nbz;
  const double *f = src + (int64_t)J.src_slot * slot_stride + (int64_t)DFCSR_F_VX_X * N;
  double s = 0.0;
#pragma unroll 8
  for (int64_t e = threadIdx.x; e < N; e += kMeanThreads) s += f[e];
  s = block_sum(s, red);
  if (threadIdx.x == 0) means[blockIdx.x] = s / (double)N;
}

// Where a target coordinate lies on an axis of the slice: its interval and
// norm distance, i < 0 outside.
struct AxisAt {
  int i;
  double y;
};

__device__ inline AxisAt axis_at(double q, double g0, double g1, int n) {
#pragma clang fp contract(off)
  if (!(q >= g0 && q <= g1) || n < 2) return {-1, 0.0};
  const int i = rgi_interval(q, g0, g1, n);
  const double a = linspace_at(g0, g1, n, i), b = linspace_at(g0, g1, n, i + 1);
  return {i, (q - a) / (b - a)};
}

// A tile of kTX x kTZ records a workgroup.  The interval searches and norm
// distances are one per row and column of the tile, the five fields one per
// node (the records' last row and column of corners included), held in LDS;
// the rings are then written in their own order, so that neighbouring lanes
// store neighbouring bytes: ten lanes a 160-byte record of the float64 ring,
// whole row pieces of the cell-major rings (their pad cell, a copy of the
// last one, is the clamped column past the edge).  Bound by the
// stores, whose records are cap apart (tiles from 4 x 32 to 4 x 128 take the
// same): one 500 x 500 slice into the float64 rings 23 us (MI355X; 32 with a
// lane per record evaluating its four corners), into the float32 ones 19 (25).
constexpr int kTX = 8, kTZ = 32, kNodeX = kTX + 1, kNodeZ = kTZ + 1;

template <int kN>
__global__ __launch_bounds__(kThreads) void regrid_kernel(
    const double *__restrict__ src, int64_t slot_stride, RegridJobs<kN> jobs, int first,
    const double *__restrict__ means, double *__restrict__ h64, float *__restrict__ h32,
    float *__restrict__ h32t, double *__restrict__ c64, float *__restrict__ c32, int Xi, int Zi,
    int cap, double xi0, double xi1, double zi0, double zi1) {
#pragma clang fp contract(off)
  __shared__ AxisAt ax[kNodeX + kNodeZ];
  __shared__ double v[kNodeX * kNodeZ * 5];
  const DfcsrRegridJob &J = jobs.j[blockIdx.y];
  const int across = (Zi + kTZ - 1) / kTZ;
  const int tile = first + (int)blockIdx.x;
  const int x0 = tile / across * kTX, z0 = tile % across * kTZ;
  const int rows = min(kTX, Xi - x0), cols = min(kTZ, Zi - z0);
  const int t = threadIdx.x;
  if (t < kNodeX)
    ax[t] = axis_at(linspace_at(xi0, xi1, Xi, min(x0 + t, Xi - 1)), J.x0, J.x1, J.nbx);
  else if (t < kNodeX + kNodeZ)
    ax[t] = axis_at(linspace_at(zi0, zi1, Zi, min(z0 + t - kNodeX, Zi - 1)), J.z0, J.z1, J.nbz);
  const double fill_vxx = means[blockIdx.y];
  const int64_t Nsrc = (int64_t)J.nbx * J.nbz;
  const double *base = src + (int64_t)J.src_slot * slot_stride;
  __syncthreads();
  for (int e = t; e < kNodeX * kNodeZ; e += kThreads) {
    const AxisAt px = ax[e / kNodeZ], pz = ax[kNodeX + e % kNodeZ];
    const bool in = px.i >= 0 && pz.i >= 0;
    const double y0 = px.y, y1 = pz.y;
    const int64_t o = (int64_t)px.i * J.nbz + pz.i;
#pragma unroll
    for (int f = 0; f < 5; ++f) {
      double r = f == DFCSR_F_VX_X ? fill_vxx : 0.0;
      if (in) {
        const double *F = base + (int64_t)f * Nsrc + o;
        r = F[0] * (1 - y0) * (1 - y1);
        r = r + F[1] * (1 - y0) * y1;
        r = r + F[J.nbz] * y0 * (1 - y1);
        r = r + F[J.nbz + 1] * y0 * y1;
      }
      v[e * 5 + f] = r;
    }
  }
  __syncthreads();
  // corner (dx, dz) of field f of record (r, c)
  auto at = [&](int r, int c, int f) { return v[(r * kNodeZ + c) * 5 + f]; };
  if (h64)
    for (int e = t; e < rows * cols * 10; e += kThreads) {
      const int rec = e / 10, h = e - rec * 10, r = rec / cols, c = rec - r * cols;
      const int f = h >> 1, d = h & 1;
      const int64_t cell = (int64_t)(x0 + r) * Zi + (z0 + c);
      double2 *out = reinterpret_cast<double2 *>(h64 + (cell * cap + J.dst_slot) * DFCSR_HIST_REC64);
      out[h] = make_double2(at(r + d, c, f), at(r + d, c + 1, f));
    }
  if (h32t)
    for (int e = t; e < rows * cols * 5; e += kThreads) {
      const int rec = e / 5, f = e - rec * 5, r = rec / cols, c = rec - r * cols;
      const int64_t cell = (int64_t)(x0 + r) * Zi + (z0 + c);
      float4 *out = reinterpret_cast<float4 *>(h32t + (cell * cap + J.dst_slot) * DFCSR_HIST_REC32);
      out[f] = make_float4((float)at(r, c, f), (float)at(r, c + 1, f), (float)at(r + 1, c, f),
                           (float)at(r + 1, c + 1, f));
    }
  if (h32)
    for (int e = t; e < rows * 5 * cols; e += kThreads) {
      const int q = e / cols, c = e - q * cols, r = q / 5, f = q - r * 5;
      const int64_t blk = (int64_t)(x0 + r) * cap + J.dst_slot;
      float4 *out = reinterpret_cast<float4 *>(h32) + (blk * DFCSR_HIST_CHUNKS32 + f) * Zi + z0 + c;
      *out = make_float4((float)at(r, c, f), (float)at(r, c + 1, f), (float)at(r + 1, c, f),
                         (float)at(r + 1, c + 1, f));
    }
  if (c64 || c32) {
    const int w = (cols + (z0 + cols == Zi ? 1 : 0)) * DFCSR_CELL;   // with the pad cell
    for (int e = t; e < rows * w; e += kThreads) {
      const int r = e / w, k = e - r * w;
      const int64_t to =
          (((int64_t)J.dst_slot * Xi + x0 + r) * DFCSR_CELL_ROW(Zi) + z0) * DFCSR_CELL + k;
      const double u = v[r * kNodeZ * 5 + k];
      if (c64) c64[to] = u;
      if (c32) c32[to] = (float)u;
    }
  }
}

// dcells32 plane of logical slice i (first <= i < nt): cells32 of slice
// i + 1 minus that of slice i, 0 for the newest.  n: floats per plane, read
// as float4 when kVec (n % 4 == 0, so every plane starts 16-byte aligned).
template <bool kVec>
__global__ __launch_bounds__(kThreads) void tdiff_kernel(const float *__restrict__ c,
                                                         float *__restrict__ d, int64_t n,
                                                         int cap, int head, int nt, int first) {
  for (int i = first + (int)blockIdx.y; i < nt; i += (int)gridDim.y) {
    const int s0 = (head + i) % cap, s1 = (head + i + 1) % cap;
    const bool last = i == nt - 1;
    if (kVec) {
      const float4 *a = reinterpret_cast<const float4 *>(c + (int64_t)s0 * n);
      const float4 *b = reinterpret_cast<const float4 *>(c + (int64_t)s1 * n);
      float4 *o = reinterpret_cast<float4 *>(d + (int64_t)s0 * n);
      for (int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x; e < n / 4;
           e += (int64_t)gridDim.x * kThreads) {
        if (last) {
          o[e] = make_float4(0.f, 0.f, 0.f, 0.f);
        } else {
          const float4 u = a[e], v = b[e];
          o[e] = make_float4(v.x - u.x, v.y - u.y, v.z - u.z, v.w - u.w);
        }
      }
    } else {
      const float *a = c + (int64_t)s0 * n, *b = c + (int64_t)s1 * n;
      float *o = d + (int64_t)s0 * n;
      for (int64_t e = (int64_t)blockIdx.x * kThreads + threadIdx.x; e < n;
           e += (int64_t)gridDim.x * kThreads)
        o[e] = last ? 0.f : b[e] - a[e];
    }
  }
}

// Whether a cell can contribute to a wake integrand: density, density_x or
// density_z nonzero, or vx or vx_x not finite (beyond the float32 range for
// a float64 cell, so that a span holds for float32 copies too).
template <typename T>
__device__ inline bool cell_contributes(const T *c) {
  const T big = (T)3.4028234663852886e38;   // FLT_MAX
  const T vx = c[DFCSR_F_VX], vxx = c[DFCSR_F_VX_X];
  // no short circuit: the five loads go out together
  return (c[DFCSR_F_DENSITY] != (T)0) | (c[DFCSR_F_DENSITY_X] != (T)0) |
         (c[DFCSR_F_DENSITY_Z] != (T)0) | !((vx <= big) & (vx >= -big)) |
         !((vxx <= big) & (vxx >= -big));
}

// x rows per workgroup of zspan_kernel: a step refreshes two slices, so 4
// rows give 2 x 125 workgroups on a 500-row grid, and 16 waves take the ten
// rows of cells these read at once, all fields of four cells a lane together
// (9 us float64, 6 float32; 17 and 16 with 4 waves and a test field by field)
constexpr int kSpanRows = 4;
constexpr int kSpanThreads = 1024;

// zspan entries (x, slot of slice i) for x in one block of kSpanRows rows:
// each wave finds the z span of whole rows (its own cells) of slices i and
// i + 1 into LDS, then each entry joins rows x, x + 1 of both slices.
template <typename T>
__global__ __launch_bounds__(kSpanThreads) void zspan_kernel(const T *__restrict__ cells,
                                                         uint32_t *__restrict__ zspan, int Xi,
                                                         int Zi, int cap, int head, int nt,
                                                         int first, int block0) {
  __shared__ int lo_s[2][kSpanRows + 1], hi_s[2][kSpanRows + 1];
  const int xb = (block0 + (int)blockIdx.x) * kSpanRows;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nwave = kSpanThreads / 64;
  const int nrow = min(kSpanRows + 1, Xi - xb);   // rows xb .. xb + nrow - 1 (x + 1 clamped)
  const int64_t plane = (int64_t)Xi * DFCSR_CELL_ROW(Zi) * DFCSR_CELL;
  for (int i = first + (int)blockIdx.y; i < nt; i += (int)gridDim.y) {
    const int np = i + 1 < nt ? 2 : 1;
    for (int w = wave; w < np * nrow; w += nwave) {
      const int p = w / nrow, r = w - p * nrow;
      const T *row = cells + (int64_t)((head + i + p) % cap) * plane +
                     (int64_t)(xb + r) * DFCSR_CELL_ROW(Zi) * DFCSR_CELL;
      int lo = 0x7fffffff, hi = -1;
#pragma unroll 4
      for (int z = lane; z < Zi; z += 64) {
        if (cell_contributes(row + (int64_t)z * DFCSR_CELL)) {
          lo = min(lo, z);
          hi = max(hi, z);
        }
      }
#pragma unroll
      for (int d = 32; d >= 1; d >>= 1) {
        lo = min(lo, __shfl_xor(lo, d, 64));
        hi = max(hi, __shfl_xor(hi, d, 64));
      }
      if (lane == 0) {
        lo_s[p][r] = lo;
        hi_s[p][r] = hi;
      }
    }
    __syncthreads();
    if ((int)threadIdx.x < min(kSpanRows, Xi - xb)) {
      const int r = threadIdx.x, r1 = min(r + 1, nrow - 1);
      int lo = min(lo_s[0][r], lo_s[0][r1]), hi = max(hi_s[0][r], hi_s[0][r1]);
      if (np == 2) {
        lo = min(lo, min(lo_s[1][r], lo_s[1][r1]));
        hi = max(hi, max(hi_s[1][r], hi_s[1][r1]));
      }
      // no contributing cell: zlo = 0xffff > zhi = 0
      const uint32_t e = hi < 0 ? 0xffffu : ((uint32_t)lo | ((uint32_t)hi << 16));
      zspan[(int64_t)(xb + r) * cap + (head + i) % cap] = e;
    }
    __syncthreads();   // before the next slice overwrites the row spans
  }
}

}  // namespace
}  // namespace dfcsr

using namespace dfcsr;

extern "C" int dfcsr_history_zspan(const double *cells, const float *cells32, uint32_t *zspan,
                                   int Xi, int Zi, int cap, int head, int nt, int first,
                                   void *stream) {
  if ((!cells && !cells32) || !zspan) return set_error(DFCSR_EINVAL, "history_zspan: NULL ring");
  if (Xi < 1 || Zi < 1 || Zi > 0xffff)
    return set_error(DFCSR_EINVAL, "history_zspan: grid %d x %d (Zi <= 65535)", Xi, Zi);
  if (cap < 1 || nt < 0 || nt > cap || head < 0 || head >= cap)
    return set_error(DFCSR_EINVAL, "history_zspan: cap %d head %d nt %d", cap, head, nt);
  if (first < 0) first = 0;
  if (first >= nt) return DFCSR_OK;
  const int gx = (Xi + kSpanRows - 1) / kSpanRows;
  int gy = nt - first;
  if (gy > 1024) gy = 1024;
  hipStream_t s = as_stream(stream);
  launch_blocks(gx, kSpanThreads, [&](int at, unsigned g) {
    if (cells)
      hipLaunchKernelGGL(zspan_kernel<double>, dim3(g, gy), dim3(kSpanThreads), 0, s, cells, zspan,
                         Xi, Zi, cap, head, nt, first, at);
    else
      hipLaunchKernelGGL(zspan_kernel<float>, dim3(g, gy), dim3(kSpanThreads), 0, s, cells32,
                         zspan, Xi, Zi, cap, head, nt, first, at);
  });
  DFCSR_LAUNCH_CHECK("history_zspan");
  return DFCSR_OK;
}

extern "C" int dfcsr_cells32_tdiff(const float *cells32, float *dcells32, int Xi, int Zi, int cap,
                                   int head, int nt, int first, void *stream) {
  if (!cells32 || !dcells32) return set_error(DFCSR_EINVAL, "cells32_tdiff: NULL ring");
  if (Xi < 1 || Zi < 1) return set_error(DFCSR_EINVAL, "cells32_tdiff: grid %d x %d", Xi, Zi);
  if (cap < 1 || nt < 0 || nt > cap || head < 0 || head >= cap)
    return set_error(DFCSR_EINVAL, "cells32_tdiff: cap %d head %d nt %d", cap, head, nt);
  if (first < 0) first = 0;
  if (first >= nt) return DFCSR_OK;
  const int64_t n = (int64_t)Xi * DFCSR_CELL_ROW(Zi) * DFCSR_CELL;   // the row copies too
  const bool vec = n % 4 == 0;
  const int64_t per = vec ? n / 4 : n;
  int gx = (int)((per + kThreads - 1) / kThreads);
  if (gx > 512) gx = 512;
  int gy = nt - first;
  if (gy > 1024) gy = 1024;
  hipStream_t s = as_stream(stream);
  if (vec)
    hipLaunchKernelGGL(tdiff_kernel<true>, dim3(gx, gy), dim3(kThreads), 0, s, cells32, dcells32,
                       n, cap, head, nt, first);
  else
    hipLaunchKernelGGL(tdiff_kernel<false>, dim3(gx, gy), dim3(kThreads), 0, s, cells32, dcells32,
                       n, cap, head, nt, first);
  DFCSR_LAUNCH_CHECK("cells32_tdiff");
  return DFCSR_OK;
}

extern "C" int64_t dfcsr_regrid_workspace_bytes(int njobs) {
  if (njobs < 1) njobs = 1;
  return (int64_t)njobs * (int64_t)(sizeof(DfcsrRegridJob) + sizeof(double)) + 256;
}

extern "C" int dfcsr_regrid(const double *src, int64_t src_slot_stride, const DfcsrRegridJob *jobs,
                            int njobs, double *hist64, float *hist32, float *hist32t,
                            double *cells, float *cells32, int Xi, int Zi, int cap, double xi0,
                            double xi1, double zi0, double zi1, void *ws, int64_t ws_bytes,
                            void *stream) {
  if (!src || !jobs || !ws) return set_error(DFCSR_EINVAL, "regrid: NULL pointer");
  if (!hist64 && !hist32 && !hist32t && !cells && !cells32)
    return set_error(DFCSR_EINVAL, "regrid: no history ring");
  if (njobs < 1) return DFCSR_OK;
  if (njobs > kMaxJobs) return set_error(DFCSR_ERANGE, "regrid: %d jobs > %d", njobs, kMaxJobs);
  if (Xi < 2 || Zi < 2) return set_error(DFCSR_EINVAL, "regrid: interp grid %d x %d", Xi, Zi);
  if (cap < 1) return set_error(DFCSR_EINVAL, "regrid: ring capacity %d", cap);
  if (ws_bytes < dfcsr_regrid_workspace_bytes(njobs))
    return set_error(DFCSR_ENOWS, "regrid: workspace too small");
  for (int k = 0; k < njobs; ++k) {
    const DfcsrRegridJob &J = jobs[k];
    if (J.nbx < 1 || J.nbz < 1 || (int64_t)5 * J.nbx * J.nbz > src_slot_stride || J.src_slot < 0 ||
        J.dst_slot < 0 || J.dst_slot >= cap)
      return set_error(DFCSR_EINVAL, "regrid: bad job %d (nbx %d nbz %d src %d dst %d)", k, J.nbx,
                       J.nbz, J.src_slot, J.dst_slot);
  }
  hipStream_t s = as_stream(stream);
  double *means = static_cast<double *>(ws);
  const int64_t tiles = (int64_t)((Xi + kTX - 1) / kTX) * ((Zi + kTZ - 1) / kTZ);
  const auto launch = [&](auto J) {
    constexpr int N = sizeof(J.j) / sizeof(J.j[0]);
    for (int k = 0; k < njobs; k += N) {
      const int m = njobs - k < N ? njobs - k : N;
      for (int i = 0; i < m; ++i) J.j[i] = jobs[k + i];
      hipLaunchKernelGGL(vxx_mean_kernel<N>, dim3(m), dim3(kMeanThreads), 0, s, src,
                         src_slot_stride, J, means + k);
      launch_blocks(tiles, kThreads, [&](int first, unsigned g) {
        hipLaunchKernelGGL(regrid_kernel<N>, dim3(g, m), dim3(kThreads), 0, s, src,
                           src_slot_stride, J, first, (const double *)(means + k), hist64, hist32,
                           hist32t, cells, cells32, Xi, Zi, cap, xi0, xi1, zi0, zi1);
      });
    }
  };
  if (njobs > kJobs) launch(RegridJobs<kManyJobs>{});
  else launch(RegridJobs<kJobs>{});
  DFCSR_LAUNCH_CHECK("regrid");
  return DFCSR_OK;
}
