// a16: mesh -> particle kick.
//
// Replaces Beam.apply_wakes (beams.py:108-131): the wake grids are scaled
// (step_size * W * 1e6 / E0, numpy's left-to-right order) and interpolated
// with scipy RegularGridInterpolator's linear rule on the linspace axes
// (xrange, zrange) at (x_transform, z), fill 0 outside; pz and (if
// transverse_on) px are incremented in place.
//
// Four to six rows of 8 bytes a particle pass through memory; beside them a
// particle reads the four corners of its cell from each wake, at random
// places.  From global memory a wave's lanes go through the cache a line at a
// time (512 cycles for the eight corners), so the wakes are held in LDS,
// scaled once per mesh point: all of them, or the middle of the mesh that
// fits, around which a bunch gathers, and the few particles outside read
// global memory.  3e6 particles, both kicks of a 128 x 128 mesh, MI355X: 33.5
// us, 4.3 TB/s (58 from global memory, every corner divided by the beam energy
// for each particle).
#include <algorithm>

#include "common.h"

namespace dfcsr {
namespace {

constexpr int kThreads = 256;

constexpr int kLdsThreads = 1024;
constexpr int kLdsBytes = 160 * 1024;

// Particles from which holding the mesh in LDS pays for staging it in every
// workgroup: both kicks, or dE alone.  Measured (rows from HBM, us, global
// memory / LDS), both: 64 x 64 at 1e6 17 / 19, at 2e6 29 / 27; 100 x 100 at
// 4e5 8 / 12, at 1e6 21 / 19; 256 x 256 at 1e6 28 / 25.  dE alone: 64 x 64 at
// 2e6 19 / 19, at 3e6 27 / 25; 128 x 128 at 3e6 28 / 29, at 8e6 83 / 60.
constexpr int64_t kLdsFromTwo = 1250000, kLdsFromOne = 4000000;
// ... on meshes of at most this many times the points that LDS holds: past it
// too few particles are in the middle.  Both kicks: 512 x 512 (26 times) at
// 2e6 42 / 38, at 1e7 262 / 205; 850 x 850 (71) 46 / 49, 285 / 259; 1024 x 1024
// (102) 49 / 53, 294 / 277; 2048 x 2048 96 / 105, 475 / 491.
constexpr int64_t kLdsMeshes = 64;

// A linspace axis with its step formed once: the interval of v as
// rgi_interval finds it (its guess may come from the reciprocal of the step,
// the search corrects it), and v's norm distance in it.
struct MeshAxis {
  double g0, g1, step, inv;
  int n;
  __device__ double at(int i) const {
#pragma clang fp contract(off)
    return i == n - 1 ? g1 : (double)i * step + g0;
  }
  __device__ int find(double v, double &y) const {
#pragma clang fp contract(off)
    const double u = (v - g0) * inv;
    int i = (u >= 0.0) ? (int)u : 0;
    if (i > n - 2) i = n - 2;
    if (i < 0) i = 0;
    double a = at(i), b = at(i + 1);
    while (i > 0 && a > v) b = a, a = at(--i);
    while (i < n - 2 && b <= v) a = b, b = at(++i + 1);
    y = (v - a) / (b - a);
    return i;
  }
};

MeshAxis make_axis(double g0, double g1, int n) {
#pragma clang fp contract(off)
  const double step = n > 1 ? (g1 - g0) / (double)(n - 1) : 0.0;
  return {g0, g1, step, 1.0 / step, n};
}

__device__ inline double scaled(double w, double step, double E0) {
#pragma clang fp contract(off)
  double v = step * w;
  v = v * 1e6;
  return v / E0;
}

// The cell of a particle and its norm distances; i < 0 outside the mesh.
struct MeshCell {
  int i, j;
  double y0, y1;
};

__device__ inline MeshCell cell_of(const MeshAxis &ax, const MeshAxis &az, double xv, double zv,
                                   double p0, double p1) {
#pragma clang fp contract(off)
  double pv = p0 * zv;
  pv = pv + p1;
  const double xt = xv - pv;   // x - np.polyval(slope, z)
  MeshCell c = {-1, 0, 0.0, 0.0};
  if (!(xt >= ax.g0 && xt <= ax.g1 && zv >= az.g0 && zv <= az.g1 && ax.n >= 2 && az.n >= 2))
    return c;
  c.i = ax.find(xt, c.y0);
  c.j = az.find(zv, c.y1);
  return c;
}

__device__ inline double bilinear(double v00, double v01, double v10, double v11,
                                  const MeshCell &c) {
#pragma clang fp contract(off)
  double r = v00 * (1 - c.y0) * (1 - c.y1);
  r = r + v01 * (1 - c.y0) * c.y1;
  r = r + v10 * c.y0 * (1 - c.y1);
  return r + v11 * c.y0 * c.y1;
}

// A wake's kick in a cell from global memory, scaled for the particle.
__device__ inline double kick_at(const double *W, int nz, const MeshCell &c, double step,
                                 double E0) {
  const double *w = W + (int64_t)c.i * nz + c.j, *u = w + nz;
  return bilinear(scaled(w[0], step, E0), scaled(w[1], step, E0), scaled(u[0], step, E0),
                  scaled(u[1], step, E0), c);
}

__global__ __launch_bounds__(kThreads) void kick_kernel(
    double *__restrict__ px, double *__restrict__ pz, const double *__restrict__ x,
    const double *__restrict__ z, int64_t n, const double *__restrict__ dE,
    const double *__restrict__ xk, MeshAxis ax, MeshAxis az, double p0, double p1, double step,
    double E0, int transverse_on) {
  for (int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x; p < n;
       p += (int64_t)gridDim.x * kThreads) {
    const MeshCell c = cell_of(ax, az, x[p], z[p], p0, p1);
    double dEv = 0.0, dxv = 0.0;
    if (c.i >= 0) {
      dEv = kick_at(dE, az.n, c, step, E0);
      if (transverse_on) dxv = kick_at(xk, az.n, c, step, E0);
    }
    pz[p] = pz[p] + dEv;
    if (transverse_on) px[p] = px[p] + dxv;
  }
}

// The mesh points held in LDS: ni x nj of them from (i0, j0), one value each
// (dE), or two side by side.
struct MeshPart {
  int i0, j0, ni, nj;
};

// The middle of an nx x nz mesh (both 2 or more), its sides in proportion, of
// at most `most` points.  Each side keeps 2 points, one cell, however thin the
// mesh is.
MeshPart middle(int nx, int nz, int most) {
  MeshPart m = {0, 0, nx, nz};
  if ((int64_t)nx * nz > most) {
    const double f = std::sqrt((double)most / ((double)nx * nz));
    m.ni = std::clamp((int)(nx * f), 2, std::min(nx, most / 2));
    m.nj = std::min(nz, most / m.ni);
    m.ni = std::min(nx, most / m.nj);
  }
  m.i0 = (nx - m.ni) / 2;
  m.j0 = (nz - m.nj) / 2;
  return m;
}

template <bool kX>
__global__ __launch_bounds__(kLdsThreads) void kick_lds_kernel(
    double *__restrict__ px, double *__restrict__ pz, const double *__restrict__ x,
    const double *__restrict__ z, int64_t n, const double *__restrict__ dE,
    const double *__restrict__ xk, MeshAxis ax, MeshAxis az, MeshPart part, double p0, double p1,
    double step, double E0) {
  extern __shared__ __align__(16) double lds[];
  double2 *const two = reinterpret_cast<double2 *>(lds);
  for (int e = threadIdx.x; e < part.ni * part.nj; e += kLdsThreads) {
    const int i = e / part.nj, j = e - i * part.nj;
    const int64_t at = (int64_t)(part.i0 + i) * az.n + part.j0 + j;
    const double a = scaled(dE[at], step, E0);
    if (kX) two[e] = make_double2(a, scaled(xk[at], step, E0));
    else lds[e] = a;
  }
  __syncthreads();
  const auto kick = [&](double xv, double zv, double &pzv, double &pxv) {
    const MeshCell c = cell_of(ax, az, xv, zv, p0, p1);
    const int i = c.i - part.i0, j = c.j - part.j0;
    double dEv = 0.0, dxv = 0.0;
    if (i >= 0 && i + 1 < part.ni && j >= 0 && j + 1 < part.nj) {
      const int o = i * part.nj + j;
      if (kX) {
        const double2 *w = two + o, *u = w + part.nj;
        const double2 a = w[0], b = w[1], d = u[0], f = u[1];
        dEv = bilinear(a.x, b.x, d.x, f.x, c);
        dxv = bilinear(a.y, b.y, d.y, f.y, c);
      } else {
        const double *w = lds + o, *u = w + part.nj;
        dEv = bilinear(w[0], w[1], u[0], u[1], c);
      }
    } else if (c.i >= 0) {
      dEv = kick_at(dE, az.n, c, step, E0);
      if (kX) dxv = kick_at(xk, az.n, c, step, E0);
    }
    pzv = pzv + dEv;
    pxv = pxv + dxv;
  };
  // two particles a turn, so that the second's rows load over the first
  const int64_t stride = (int64_t)gridDim.x * kLdsThreads;
  int64_t p = (int64_t)blockIdx.x * kLdsThreads + threadIdx.x;
  for (; p + stride < n; p += 2 * stride) {
    const int64_t q = p + stride;
    const double xp = x[p], zp = z[p], xq = x[q], zq = z[q];
    double ap = pz[p], aq = pz[q], bp = kX ? px[p] : 0.0, bq = kX ? px[q] : 0.0;
    kick(xp, zp, ap, bp);
    pz[p] = ap;
    if (kX) px[p] = bp;
    kick(xq, zq, aq, bq);
    pz[q] = aq;
    if (kX) px[q] = bq;
  }
  if (p < n) {
    double a = pz[p], b = kX ? px[p] : 0.0;
    kick(x[p], z[p], a, b);
    pz[p] = a;
    if (kX) px[p] = b;
  }
}

}  // namespace
}  // namespace dfcsr

using namespace dfcsr;

extern "C" int dfcsr_apply_wakes(double *px, double *pz, const double *x, const double *z,
                                 int64_t n, const double *dE_dct, const double *x_kick, int xbins,
                                 int zbins, double xr0, double xr1, double zr0, double zr1,
                                 double slope0, double slope1, double step_size,
                                 double init_energy, int transverse_on, void *stream) {
  if (!pz || !x || !z || !dE_dct || (transverse_on && (!px || !x_kick)))
    return set_error(DFCSR_EINVAL, "apply_wakes: NULL pointer");
  if (xbins < 1 || zbins < 1) return set_error(DFCSR_EINVAL, "apply_wakes: bad mesh");
  if (n <= 0) return DFCSR_OK;
  const MeshAxis ax = make_axis(xr0, xr1, xbins), az = make_axis(zr0, zr1, zbins);
  hipStream_t s = as_stream(stream);
  // (a mesh one point wide has no cells: no particle is kicked)
  const int value = transverse_on ? 16 : 8;
  if (n >= (transverse_on ? kLdsFromTwo : kLdsFromOne) && xbins >= 2 && zbins >= 2 &&
      (int64_t)xbins * zbins <= kLdsMeshes * (kLdsBytes / value)) {
    const MeshPart part = middle(xbins, zbins, kLdsBytes / value);
    const int64_t bytes = (int64_t)part.ni * part.nj * value;
    int64_t b = (n + kLdsThreads - 1) / kLdsThreads;
    const int64_t most = 256 * (bytes <= kLdsBytes / 2 ? 2 : 1);   // what the CUs' LDS holds
    if (b > most) b = most;
    if (transverse_on)
      hipLaunchKernelGGL(kick_lds_kernel<true>, dim3((int)b), dim3(kLdsThreads), (size_t)bytes, s,
                         px, pz, x, z, n, dE_dct, x_kick, ax, az, part, slope0, slope1, step_size,
                         init_energy);
    else
      hipLaunchKernelGGL(kick_lds_kernel<false>, dim3((int)b), dim3(kLdsThreads), (size_t)bytes, s,
                         px, pz, x, z, n, dE_dct, x_kick, ax, az, part, slope0, slope1, step_size,
                         init_energy);
  } else {
    int64_t b = (n + kThreads - 1) / kThreads;
    if (b > 8192) b = 8192;
    hipLaunchKernelGGL(kick_kernel, dim3((int)b), dim3(kThreads), 0, s, px, pz, x, z, n, dE_dct,
                       x_kick, ax, az, slope0, slope1, step_size, init_energy, transverse_on);
  }
  DFCSR_LAUNCH_CHECK("apply_wakes");
  return DFCSR_OK;
}
