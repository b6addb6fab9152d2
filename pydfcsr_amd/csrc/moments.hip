// a1: beam moments with a fixed reduction tree (deterministic).
//
// Replaces the numpy statistics the CSR step reads: Beam.update_status and
// its properties (beams.py:88-98, 137-215), get_CSR_mesh's std/mean of
// x_transform (CSR.py:368-374) and get_DF's slice std (deposit.py:147-159).
// Means are sums over n and spreads centred sums of squares, as numpy's std;
// the least-squares slope is cov(x, z)/var(z), intercept
// mean_x - slope*mean_z.
//
// Bound by memory: the moments read x and z twice (the residual spread and
// the slice need the slope and sigma_z of the first pass, and forming them
// from raw products would cancel for a tilted beam), the statistics read six
// rows once.  One workgroup of 16 waves a compute unit (kMaxBlocks) keeps
// 64 KB or more of loads in flight on each, and leaves few partial sums for
// the next pass: the second pass's workgroups each add the first's 256 by
// themselves.  At 1e7 particles (MI355X) the moments take 61 us, 27 + 29 us of
// them reading 160 MB twice at 5.7 TB/s (four passes over x and z with a
// one-workgroup kernel after each: 132 us), the statistics 80 us, 75 of them
// reading 480 MB at 6.4 TB/s (145 + 43 us with 27 block sums, one after the
// other, at the end of each of 1024 workgroups).  At 1e5 both are latency: 15
// and 11 us (38 and 54).
#include "common.h"

namespace dfcsr {
namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr int kMaxBlocks = 256;
constexpr int kPair = 2;                     // neighbouring particles a lane loads at once
constexpr int kTile = kThreads * kPair;

// Two neighbouring values of a row; rows start at any multiple of 8 bytes.
typedef double Pair __attribute__((ext_vector_type(2), aligned(8)));

__device__ inline Pair load_pair(const double *p) { return *reinterpret_cast<const Pair *>(p); }

int nblocks_for(int64_t n) {
  int64_t b = (n + kTile - 1) / kTile;
  if (b < 1) b = 1;
  if (b > kMaxBlocks) b = kMaxBlocks;
  return (int)b;
}

// Each wave's sums of K values into its row of smem (kWaves * K doubles).
template <int K>
__device__ inline void wave_sums(const double (&v)[K], double *smem) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < K; k += 4) {
    const double s = wave_sum4(v[k], k + 1 < K ? v[k + 1] : 0.0, k + 2 < K ? v[k + 2] : 0.0,
                               k + 3 < K ? v[k + 3] : 0.0);
    const int of = k + wave_sum4_of(lane >> 4);
    if ((lane & 15) == 0 && of < K) smem[wid * K + of] = s;
  }
}

// Sums of K values over the workgroup (fixed tree), in every thread.
// smem: kWaves * K doubles.
template <int K>
__device__ inline void block_sums(double (&v)[K], double *smem) {
  __syncthreads();
  wave_sums<K>(v, smem);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    double r = 0.0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) r += smem[w * K + k];
    v[k] = r;
  }
}

// stats layout in workspace (doubles):
//   [0..9] results (same order as the public output)
//   [16 ...] workgroup partials of both passes, kPart a workgroup each
enum { S_MX = 0, S_MZ, S_SX, S_SZ, S_P0, S_P1, S_MXT, S_SXT, S_SSL, S_NSL };
constexpr int kPartOff = 16;
constexpr int kPart = 6;
constexpr int kWsPartials = 1024 * 4;        // doubles of partials a caller's workspace holds
static_assert(2 * kMaxBlocks * kPart <= kWsPartials, "partials fit the workspace");

// Centred sums of a thread, joined to the next batch's by the pairwise rule:
// with nt values before and nb in the batch, means m and mb,
// M2 = M2 + M2b + (mb - m)^2 nt nb / (nt + nb).  No large squares cancel.
struct Joint {
  double n = 0.0, mx = 0.0, mz = 0.0, xx = 0.0, xz = 0.0, zz = 0.0;

  __device__ void join(double nb, double bx, double bz, double bxx, double bxz, double bzz) {
    const double r = nb / (n + nb), f = n * r, dx = bx - mx, dz = bz - mz;
    n += nb;
    mx += dx * r;
    mz += dz * r;
    xx += bxx + dx * dx * f;
    xz += bxz + dx * dz * f;
    zz += bzz + dz * dz * f;
  }

  __device__ void pair(Pair x, Pair z) {
    const double dx = 0.5 * (x[1] - x[0]), dz = 0.5 * (z[1] - z[0]);
    join(2.0, x[0] + dx, z[0] + dz, 2.0 * dx * dx, 2.0 * dx * dz, 2.0 * dz * dz);
  }

  __device__ void one(double x, double z) { join(1.0, x, z, 0.0, 0.0, 0.0); }
};

// pass 0, per workgroup: sum x, sum z, count, centred xx, xz, zz
__global__ __launch_bounds__(kThreads) void moments_first(const double *__restrict__ x,
                                                          const double *__restrict__ z,
                                                          int64_t n, double *__restrict__ st) {
  __shared__ double red[kWaves * 3];
  double s[3] = {0.0, 0.0, 0.0};
  Joint m;
  const int64_t stride = (int64_t)gridDim.x * kTile;
  int64_t i = (int64_t)blockIdx.x * kTile + (int64_t)threadIdx.x * kPair;
  for (; i + stride + 1 < n; i += 2 * stride) {
    const Pair x0 = load_pair(x + i), x1 = load_pair(x + i + stride);
    const Pair z0 = load_pair(z + i), z1 = load_pair(z + i + stride);
    s[0] += (x0[0] + x0[1]) + (x1[0] + x1[1]);
    s[1] += (z0[0] + z0[1]) + (z1[0] + z1[1]);
    m.pair(x0, z0);
    m.pair(x1, z1);
  }
  for (; i < n; i += stride) {
    const bool two = i + 1 < n;
    for (int e = 0; e < (two ? 2 : 1); ++e) {
      const double xv = x[i + e], zv = z[i + e];
      s[0] += xv;
      s[1] += zv;
      m.one(xv, zv);
    }
  }
  s[2] = m.n;
  block_sums<3>(s, red);
  double c[3] = {m.xx, m.xz, m.zz};
  if (m.n > 0.0) {
    const double dx = m.mx - s[0] / s[2], dz = m.mz - s[1] / s[2];
    c[0] += m.n * (dx * dx);
    c[1] += m.n * (dx * dz);
    c[2] += m.n * (dz * dz);
  }
  block_sums<3>(c, red);
  if (threadIdx.x != 0) return;
  double *p = st + kPartOff + blockIdx.x * kPart;
  p[0] = s[0], p[1] = s[1], p[2] = s[2], p[3] = c[0], p[4] = c[1], p[5] = c[2];
}

// pass 1: the first pass's results from its partials (every workgroup, the
// same sums), then per workgroup of xt = x - (slope z + intercept): sum,
// count, centred square; of the slice |z| < 0.1 sigma_z: count, sum x,
// centred square
__global__ __launch_bounds__(kThreads) void moments_second(const double *__restrict__ x,
                                                           const double *__restrict__ z,
                                                           int64_t n, double *__restrict__ st) {
  __shared__ double red[kWaves * 4];
  static_assert(kMaxBlocks <= kThreads, "one partial a thread");
  const bool has = threadIdx.x < gridDim.x;
  const double *p = st + kPartOff + threadIdx.x * kPart;
  double t[2] = {has ? p[0] : 0.0, has ? p[1] : 0.0};
  const double cnt = has ? p[2] : 1.0;
  const double bx = t[0] / cnt, bz = t[1] / cnt;
  double c[3] = {0.0, 0.0, 0.0};
  if (has) c[0] = p[3], c[1] = p[4], c[2] = p[5];
  block_sums<2>(t, red);
  const double dn = (double)n, mx = t[0] / dn, mz = t[1] / dn;
  if (has) {
    const double dx = bx - mx, dz = bz - mz;
    c[0] += cnt * (dx * dx);
    c[1] += cnt * (dx * dz);
    c[2] += cnt * (dz * dz);
  }
  block_sums<3>(c, red);
  const double sz = sqrt(c[2] / dn), p0 = c[1] / c[2], p1 = mx - p0 * mz;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st[S_MX] = mx, st[S_MZ] = mz, st[S_SX] = sqrt(c[0] / dn), st[S_SZ] = sz;
    st[S_P0] = p0, st[S_P1] = p1;
  }
  const double cut = 0.1 * sz;

  // the slice's centred square is taken about the thread's first slice
  // particle, a sample of the slice, so little cancels
  double s[4] = {0.0, 0.0, 0.0, 0.0};   // sum xt, count, slice count, slice sum x
  Joint m;
  double from = 0.0, e1 = 0.0, e2 = 0.0;
  auto slice = [&](double xv, double zv) {
    const bool in = fabs(zv) < cut;
    from = in && s[2] == 0.0 ? xv : from;
    const double e = in ? xv - from : 0.0;
    s[2] += in ? 1.0 : 0.0;
    s[3] += in ? xv : 0.0;
    e1 += e;
    e2 += e * e;
  };
  const int64_t stride = (int64_t)gridDim.x * kTile;
  int64_t i = (int64_t)blockIdx.x * kTile + (int64_t)threadIdx.x * kPair;
  for (; i + stride + 1 < n; i += 2 * stride) {
    const Pair x0 = load_pair(x + i), x1 = load_pair(x + i + stride);
    const Pair z0 = load_pair(z + i), z1 = load_pair(z + i + stride);
    const Pair t0 = x0 - (p0 * z0 + p1), t1 = x1 - (p0 * z1 + p1);
    s[0] += (t0[0] + t0[1]) + (t1[0] + t1[1]);
    m.pair(t0, t0);
    m.pair(t1, t1);
    slice(x0[0], z0[0]);
    slice(x0[1], z0[1]);
    slice(x1[0], z1[0]);
    slice(x1[1], z1[1]);
  }
  for (; i < n; i += stride) {
    const bool two = i + 1 < n;
    for (int e = 0; e < (two ? 2 : 1); ++e) {
      const double xv = x[i + e], zv = z[i + e], xt = xv - (p0 * zv + p1);
      s[0] += xt;
      m.one(xt, xt);
      slice(xv, zv);
    }
  }
  s[1] = m.n;
  const double ns = s[2];
  block_sums<4>(s, red);
  double q[2] = {m.xx, 0.0};
  if (m.n > 0.0) {
    const double d = m.mx - s[0] / s[1];
    q[0] += m.n * (d * d);
  }
  if (ns > 0.0) {
    const double v = e2 - e1 * (e1 / ns), d = (from + e1 / ns) - s[3] / s[2];
    q[1] = (v < 0.0 ? 0.0 : v) + ns * (d * d);
  }
  block_sums<2>(q, red);
  if (threadIdx.x != 0) return;
  double *o = st + kPartOff + (kMaxBlocks + blockIdx.x) * kPart;
  o[0] = s[0], o[1] = s[1], o[2] = q[0], o[3] = s[2], o[4] = s[3], o[5] = q[1];
}

__global__ __launch_bounds__(kThreads) void moments_final(int64_t n, int nblk,
                                                          const double *__restrict__ st,
                                                          double *__restrict__ out) {
  __shared__ double red[kWaves * 3];
  const bool has = (int)threadIdx.x < nblk;
  const double *p = st + kPartOff + (kMaxBlocks + threadIdx.x) * kPart;
  double v[kPart];
#pragma unroll
  for (int k = 0; k < kPart; ++k) v[k] = has ? p[k] : 0.0;
  double t[3] = {v[0], v[3], v[4]};
  block_sums<3>(t, red);
  const double dn = (double)n, mxt = t[0] / dn;
  const double msl = t[2] / t[1];   // NaN for an empty slice, as np.std([])
  double q[2] = {v[2], v[5]};
  if (has) {
    const double d = v[0] / v[1] - mxt;
    q[0] += v[1] * (d * d);
  }
  if (v[3] > 0.0) {
    const double d = v[4] / v[3] - msl;
    q[1] += v[3] * (d * d);
  }
  block_sums<2>(q, red);
  if (threadIdx.x != 0) return;
  for (int k = 0; k <= S_P1; ++k) out[k] = st[k];
  out[S_MXT] = mxt;
  out[S_SXT] = sqrt(q[0] / dn);
  out[S_SSL] = sqrt(q[1] / t[1]);
  out[S_NSL] = t[1];
}

// ---- per-step beam statistics (CSR.py:837-859, twiss.py:2-70) -------------
//
// Means and the sample covariance (np.cov, ddof = 1) of the six coordinates
// (x, px, y, py, z, pz) in one pass over the particles: sums of d = v - c
// and of the products d_p d_q, each a fixed reduction tree, with c the mean
// of the first (up to) 256 particles -- within a small fraction of a sigma
// of the bunch's mean, so the shifted sums lose nothing to cancellation
// beyond a few ulps.  The final single-workgroup pass forms
// mean = c + S_d / n and cov = (S_pq - S_p S_q / n) / (n - 1), then the
// Twiss and dispersion parameters of (x, px, pz) and (y, py, pz) and the
// energy statistics.
constexpr int kNCov = 27;          // 6 shifted sums, then the 21 products (upper triangle)
constexpr int kShift = 256;        // particles whose mean is the shift
constexpr int kStatOff = 32;       // partials start here (doubles): kNCov rows of kMaxBlocks

__device__ inline int tri_index(int i, int j) {   // i <= j < 6, row-major upper triangle
  return i * 6 - i * (i - 1) / 2 + (j - i);
}

struct CovSums {
  double a[kNCov] = {};

  __device__ void add(const double (&v)[6]) {
#pragma unroll
    for (int k = 0; k < 6; ++k) a[k] += v[k];
#pragma unroll
    for (int p = 0; p < 6; ++p)
#pragma unroll
      for (int q = p; q < 6; ++q) a[6 + tri_index(p, q)] += v[p] * v[q];
  }
};

__global__ __launch_bounds__(kThreads) void stats_partial(
    const double *__restrict__ x, const double *__restrict__ px, const double *__restrict__ y,
    const double *__restrict__ py, const double *__restrict__ z, const double *__restrict__ pz,
    int64_t n, double *__restrict__ st) {
  __shared__ double red[kWaves * kNCov];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const double *c[6] = {x, px, y, py, z, pz};
  // the shift: every workgroup forms the same sums in the same order, one
  // coordinate a wave
  const int shifted = n < kShift ? (int)n : kShift;
#pragma unroll
  for (int k = 0; k < 6; ++k)
    if (wid == k) {
      double v = 0.0;
#pragma unroll
      for (int j = 0; j < kShift / 64; ++j) v += lane + 64 * j < shifted ? c[k][lane + 64 * j] : 0.0;
      v = wave_sum(v) / (double)shifted;
      if (lane == 0) red[k] = v;
    }
  __syncthreads();
  double m[6];
#pragma unroll
  for (int k = 0; k < 6; ++k) m[k] = red[k];
  if (blockIdx.x == 0 && threadIdx.x < 6) st[threadIdx.x] = red[threadIdx.x];
  CovSums s;
  const int64_t stride = (int64_t)gridDim.x * kTile;
  int64_t i = (int64_t)blockIdx.x * kTile + (int64_t)threadIdx.x * kPair;
  for (; i + 1 < n; i += stride) {
    Pair w[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) w[k] = load_pair(c[k] + i);
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      double v[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) v[k] = w[k][e] - m[k];
      s.add(v);
    }
  }
  if (i < n) {
    double v[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = c[k][i] - m[k];
    s.add(v);
  }
  __syncthreads();
  wave_sums<kNCov>(s.a, red);
  __syncthreads();
  if (threadIdx.x < kNCov) {
    double v = 0.0;
    for (int w = 0; w < kWaves; ++w) v += red[w * kNCov + threadIdx.x];
    st[kStatOff + threadIdx.x * kMaxBlocks + blockIdx.x] = v;
  }
}

// Twiss and dispersion of one plane from its 3 x 3 covariance of (u, pu,
// delta) (twiss.py:30-70): out = alpha, beta, gamma, emit, eta, etap, norm_emit.
__device__ inline void twiss_plane(double s00, double s01, double s02, double s11, double s12,
                                   double s22, double p0c, double mc2, double *out) {
  const double delta2 = s22;
  const double eb = s00 - s02 * s02 / delta2;
  const double eg = s11 - s12 * s12 / delta2;
  const double ea = -s01 + s02 * s12 / delta2;
  const double emit = sqrt(eb * eg - ea * ea);
  out[0] = ea / emit;
  out[1] = eb / emit;
  out[2] = eg / emit;
  out[3] = emit;
  out[4] = s02 / delta2;
  out[5] = s12 / delta2;
  out[6] = emit * p0c / mc2;
}

__global__ __launch_bounds__(kThreads) void stats_final(int64_t n, int nblk, double p0c,
                                                        double mc2, const double *__restrict__ st,
                                                        double *__restrict__ out) {
  __shared__ double tot[kNCov], cov[21];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const double dn = (double)n;
  for (int k = wid; k < kNCov; k += kWaves) {   // one sum a wave
    double v = 0.0;
#pragma unroll
    for (int j = 0; j < kMaxBlocks / 64; ++j) {
      const int b = lane + 64 * j;
      v += b < nblk ? st[kStatOff + k * kMaxBlocks + b] : 0.0;
    }
    v = wave_sum(v);
    if (lane == 0) tot[k] = v;
  }
  __syncthreads();
  if (wid == 0) {
    if (lane < 6) out[DFCSR_STAT_MEAN + lane] = st[lane] + tot[lane] / dn;
    int p = 0;
    while (p < 5 && lane >= tri_index(p + 1, p + 1)) ++p;
    const int q = p + lane - tri_index(p, p);
    if (lane < 21) {
      const double v = (tot[6 + lane] - tot[p] * tot[q] / dn) / (dn - 1.0);
      cov[lane] = v;
      out[DFCSR_STAT_COV + lane] = v;
    }
  }
  __syncthreads();
  // planes (x, px, pz) and (y, py, pz): coordinates 0, 1, 5 and 2, 3, 5; a
  // wave each, and the energy = (pz + 1) p0c (beams.py:166-181), its mean and
  // population std
  if (lane != 0) return;
  if (wid < 2) {
    const int u = 2 * wid;
    twiss_plane(cov[tri_index(u, u)], cov[tri_index(u, u + 1)], cov[tri_index(u, 5)],
                cov[tri_index(u + 1, u + 1)], cov[tri_index(u + 1, 5)], cov[tri_index(5, 5)], p0c,
                mc2, out + (wid ? DFCSR_STAT_TWISS_Y : DFCSR_STAT_TWISS_X));
  } else if (wid == 2) {
    out[DFCSR_STAT_MEAN_ENERGY] = ((st[5] + tot[5] / dn) + 1.0) * p0c;
    out[DFCSR_STAT_SIGMA_ENERGY] = p0c * sqrt(cov[tri_index(5, 5)] * ((dn - 1.0) / dn));
  }
}

}  // namespace
}  // namespace dfcsr

using namespace dfcsr;

extern "C" int64_t dfcsr_beam_statistics_workspace_bytes(int64_t n) {
  (void)n;
  return (int64_t)(kStatOff + 1024 * kNCov) * (int64_t)sizeof(double);
}

extern "C" int dfcsr_beam_statistics(const double *x, const double *px, const double *y,
                                     const double *py, const double *z, const double *pz,
                                     int64_t n, double p0c, double mc2, void *ws,
                                     int64_t ws_bytes, double *out, void *stream) {
  if (!x || !px || !y || !py || !z || !pz || !out || !ws)
    return set_error(DFCSR_EINVAL, "beam_statistics: NULL pointer");
  if (n < 2)
    return set_error(DFCSR_EINVAL, "beam_statistics: need n >= 2 particles (n=%lld)",
                     (long long)n);
  if (ws_bytes < dfcsr_beam_statistics_workspace_bytes(n))
    return set_error(DFCSR_ENOWS, "beam_statistics: workspace %lld < %lld bytes",
                     (long long)ws_bytes, (long long)dfcsr_beam_statistics_workspace_bytes(n));
  hipStream_t s = as_stream(stream);
  double *st = static_cast<double *>(ws);
  const int nb = nblocks_for(n);
  hipLaunchKernelGGL(stats_partial, dim3(nb), dim3(kThreads), 0, s, x, px, y, py, z, pz, n, st);
  hipLaunchKernelGGL(stats_final, dim3(1), dim3(kThreads), 0, s, n, nb, p0c, mc2,
                     (const double *)st, out);
  DFCSR_LAUNCH_CHECK("beam_statistics");
  return DFCSR_OK;
}

extern "C" int64_t dfcsr_moments_workspace_bytes(int64_t n) {
  (void)n;
  return (int64_t)(kPartOff + kWsPartials) * (int64_t)sizeof(double);
}

extern "C" int dfcsr_beam_moments(const double *x, const double *z, int64_t n, void *ws,
                                  int64_t ws_bytes, double *out, void *stream) {
  if (!x || !z || !out || !ws) return set_error(DFCSR_EINVAL, "beam_moments: NULL pointer");
  if (n < 2) return set_error(DFCSR_EINVAL, "beam_moments: need n >= 2 particles (n=%lld)",
                              (long long)n);
  if (ws_bytes < dfcsr_moments_workspace_bytes(n))
    return set_error(DFCSR_ENOWS, "beam_moments: workspace %lld < %lld bytes",
                     (long long)ws_bytes, (long long)dfcsr_moments_workspace_bytes(n));
  hipStream_t s = as_stream(stream);
  double *st = static_cast<double *>(ws);
  int nb = nblocks_for(n);
  hipLaunchKernelGGL(moments_first, dim3(nb), dim3(kThreads), 0, s, x, z, n, st);
  hipLaunchKernelGGL(moments_second, dim3(nb), dim3(kThreads), 0, s, x, z, n, st);
  hipLaunchKernelGGL(moments_final, dim3(1), dim3(kThreads), 0, s, n, nb, (const double *)st, out);
  DFCSR_LAUNCH_CHECK("beam_moments");
  return DFCSR_OK;
}
