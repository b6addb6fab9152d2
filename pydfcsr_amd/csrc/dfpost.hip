// a4-a6: density-function post-processing of one deposited slice.
//
// Replaces deposit.py:183-235 as four launches on one stream: the maximum of
// the raw density; the velocity division and the smoothing of density and
// vx; their normalisation, gradients and the smoothing of those; the fill of
// vx_x.  The grids are small (100 x 100 to 256 x 256 in use), so launches and
// serial passes bound it, not bytes: what a step needs of the whole grid
// (maxima, the trapezoid normalisation, the masked mean of vx_x) is left as
// one partial a workgroup by the step before and added by each workgroup of
// the next in the same fixed order, so results are the same every launch.
// The four kernels with a window of 9 take 24 us at 100 x 100 and 25 us at
// 256 x 256 (MI355X; as eight launches, two of them one workgroup over the
// whole grid, 256 x 256 took 160 us).
// A tile's inputs, gradients and first smoothing stay in LDS.  The velocity
// division and the normalisation are applied where their inputs are read, in
// the reference's operation order.
//
// Savitzky-Golay: scipy.signal.savgol_filter(mode='interp') is linear: the
// interior is the symmetric smoothing stencil c[] (the centre row of the
// least-squares hat matrix H = V (V^T V)^-1 V^T of the window) and the
// first/last window//2 outputs are rows of the same H applied to the first/
// last `window` samples (scipy fits and evaluates a polynomial there,
// scipy/signal/_savitzky_golay.py _fit_edge).  H is computed on the host in
// extended precision and passed by value.
#include <string.h>

#include "common.h"

namespace dfcsr {

struct SGOp {
  int W, h;
  double c[DFCSR_MAX_SG_WINDOW];
  double E[DFCSR_MAX_SG_WINDOW / 2][DFCSR_MAX_SG_WINDOW];   // left-edge rows of H
};

// Hat matrix rows of a degree-`order` least-squares fit over `W` points,
// by Gauss-Jordan on the normal equations of the centred monomial basis
// (long double; the matrices are integer valued).
static int make_sg(int W, int order, SGOp *op) {
  if (W < 1 || (W % 2) == 0 || W > DFCSR_MAX_SG_WINDOW)
    return set_error(DFCSR_EINVAL, "savgol: window %d must be odd and <= %d", W,
                     DFCSR_MAX_SG_WINDOW);
  if (order < 0 || order >= W)
    return set_error(DFCSR_EINVAL, "savgol: polyorder %d must be < window %d", order, W);
  const int m = order + 1, h = W / 2;
  long double V[DFCSR_MAX_SG_WINDOW][DFCSR_MAX_SG_WINDOW];
  for (int j = 0; j < W; ++j) {
    long double t = (long double)(j - h), p = 1.0L;
    for (int k = 0; k < m; ++k) {
      V[j][k] = p;
      p *= t;
    }
  }
  // A = V^T V (m x m), B = V^T (m x W); solve A X = B in place.
  long double A[DFCSR_MAX_SG_WINDOW][DFCSR_MAX_SG_WINDOW];
  long double B[DFCSR_MAX_SG_WINDOW][DFCSR_MAX_SG_WINDOW];
  for (int a = 0; a < m; ++a) {
    for (int b = 0; b < m; ++b) {
      long double s = 0.0L;
      for (int j = 0; j < W; ++j) s += V[j][a] * V[j][b];
      A[a][b] = s;
    }
    for (int j = 0; j < W; ++j) B[a][j] = V[j][a];
  }
  for (int col = 0; col < m; ++col) {
    int piv = col;
    for (int r = col + 1; r < m; ++r)
      if (fabsl(A[r][col]) > fabsl(A[piv][col])) piv = r;
    if (A[piv][col] == 0.0L) return set_error(DFCSR_EINVAL, "savgol: singular fit");
    if (piv != col) {
      for (int k = 0; k < m; ++k) { long double t = A[col][k]; A[col][k] = A[piv][k]; A[piv][k] = t; }
      for (int k = 0; k < W; ++k) { long double t = B[col][k]; B[col][k] = B[piv][k]; B[piv][k] = t; }
    }
    long double d = A[col][col];
    for (int k = 0; k < m; ++k) A[col][k] /= d;
    for (int k = 0; k < W; ++k) B[col][k] /= d;
    for (int r = 0; r < m; ++r) {
      if (r == col) continue;
      long double f = A[r][col];
      if (f == 0.0L) continue;
      for (int k = 0; k < m; ++k) A[r][k] -= f * A[col][k];
      for (int k = 0; k < W; ++k) B[r][k] -= f * B[col][k];
    }
  }
  memset(op, 0, sizeof(*op));
  op->W = W;
  op->h = h;
  // H[i][j] = sum_k V[i][k] X[k][j]
  for (int i = 0; i <= h; ++i)
    for (int j = 0; j < W; ++j) {
      long double s = 0.0L;
      for (int k = 0; k < m; ++k) s += V[i][k] * B[k][j];
      if (i == h) op->c[j] = (double)s;
      else op->E[i][j] = (double)s;
    }
  return DFCSR_OK;
}

namespace {

// Threads of a workgroup.  There is at most one workgroup a CU at the grids in
// use, so a launch lasts as long as one chain: 512 threads pass over a tile
// with its margins (640 inputs at a window of 9) in two rounds where 256 take
// three, the inputs are on their way while the partials are added, and the
// fields of a tile are summed side by side.  The second and third kernel at
// 256 x 256: 7.9 and 13.0 us before, 5.9 and 9.5 with 512 (6.2 and 10.9 with
// 256, 6.9 and 10.8 with 1024).
constexpr int kT = 512;
constexpr int kMaxGrid = 512;     // workgroups (and partials) of a pass
constexpr int kMaxPerBlock = 1024;   // cells a workgroup of the maximum reads, at least

// Rows of partials, one value a workgroup, np values apart.
enum { P_RAW = 0, P_SUM, P_MAX, P_MIN, P_FILL, P_COUNT, P_ROWS };

// np.linspace(start, stop, n) with its step formed once.
struct Axis {
  double start, stop, step;
  int n, uniform;
  __device__ double at(int i) const {
#pragma clang fp contract(off)
    if (n <= 1) return start;
    return i == n - 1 ? stop : (double)i * step + start;
  }
  // spacing i -> i + 1; 0 outside the axis
  __device__ double width(int i) const {
#pragma clang fp contract(off)
    return i < 0 || i + 1 >= n ? 0.0 : at(i + 1) - at(i);
  }
};

// The operator's rows in LDS (a lane's row is its own, and kernel arguments
// are slow to load by lane): h edge rows, then the interior stencil.
struct SGRows {
  const double *c;
  int W, h;
};

__host__ __device__ inline int sg_rows_size(int W) { return (W / 2 + 1) * W; }

__device__ inline SGRows sg_rows(const SGOp &op, double *lds) {
  for (int e = threadIdx.x; e < (op.h + 1) * op.W; e += kT) {
    const int r = e / op.W, k = e - r * op.W;
    lds[e] = r == op.h ? op.c[k] : op.E[r][k];
  }
  return {lds, op.W, op.h};
}

// Savitzky-Golay sums of output i of NF lines of n inputs; in(f, k) gives
// input k of line f.  The last h rows mirror the left edge's.  The lines go
// on side by side, so that their reads are in flight together.
template <int NF, typename In>
__device__ inline void sg_at(const SGRows &op, const In &in, int n, int i, double (&acc)[NF]) {
#pragma clang fp contract(off)
  const int W = op.W, h = op.h;
  const bool left = i < h, right = !left && i >= n - h;
  const int from = left ? 0 : right ? n - W : i - h, step = right ? -1 : 1;
  const double *c = op.c + (left ? i : right ? n - 1 - i : h) * W + (right ? W - 1 : 0);
#pragma unroll
  for (int f = 0; f < NF; ++f) acc[f] = 0.0;
#pragma unroll 4
  for (int k = 0; k < W; ++k, c += step) {
#pragma unroll
    for (int f = 0; f < NF; ++f) acc[f] += *c * in(f, from + k);
  }
}

// np.gradient spacing test: the coordinate diffs all equal the first one
// (then numpy uses the scalar-spacing formula).  Evaluated on the host.
bool axis_uniform(double g0, double g1, int n) {
#pragma clang fp contract(off)
  if (n < 2) return true;
  const double d0 = linspace_at(g0, g1, n, 1) - linspace_at(g0, g1, n, 0);
  for (int i = 1; i < n - 1; ++i)
    if (linspace_at(g0, g1, n, i + 1) - linspace_at(g0, g1, n, i) != d0) return false;
  return true;
}

Axis make_axis(double g0, double g1, int n) {
#pragma clang fp contract(off)
  return {g0, g1, n > 1 ? (g1 - g0) / (double)(n - 1) : 0.0, n, axis_uniform(g0, g1, n)};
}

// np.gradient(f, g) at position i of an axis (edge_order 1),
// numpy/lib/_function_base_impl.py: the weights a, b, c of f(i - 1), f(i),
// f(i + 1) inside a non-uniform axis, else the divisor in a.
struct GradAt {
  double a, b, c;
};

__device__ inline GradAt grad_weights(const Axis &g, int i) {
#pragma clang fp contract(off)
  if (g.n < 2) return {0.0, 0.0, 0.0};
  const double dxu = g.width(0);
  if (i == 0) return {dxu, 0.0, 0.0};
  if (i == g.n - 1) return {g.uniform ? dxu : g.width(i - 1), 0.0, 0.0};
  if (g.uniform) return {2. * dxu, 0.0, 0.0};
  const double dx1 = g.width(i - 1), dx2 = g.width(i);
  return {-(dx2) / (dx1 * (dx1 + dx2)), (dx2 - dx1) / (dx1 * dx2), dx1 / (dx2 * (dx1 + dx2))};
}

// f: the value at i, st: the step between neighbours along the axis.
__device__ inline double grad_at(const double *f, int st, const Axis &g, int i, const GradAt &w) {
#pragma clang fp contract(off)
  if (g.n < 2) return 0.0;
  if (i == 0) return (f[st] - f[0]) / w.a;
  if (i == g.n - 1) return (f[0] - f[-st]) / w.a;
  if (g.uniform) return (f[st] - f[-st]) / w.a;
  return w.a * f[-st] + w.b * f[0] + w.c * f[st];
}

// A wave's values w, the same in its lanes, for every thread to add in the
// order of the waves.
template <int N>
__device__ inline void to_waves(const double (&w)[N], double (&each)[N][kT / 64]) {
#pragma unroll
  for (int f = 0; f < N; ++f)
    if ((threadIdx.x & 63) == 0) each[f][threadIdx.x >> 6] = w[f];
  __syncthreads();
}

// Maximum of a row of partials, in every thread (NaN ignored, as fmax).
__device__ inline double max_of(const double *part, int n, double *red) {
  double m = -INFINITY;
  for (int k = threadIdx.x; k < n; k += kT) m = fmax(m, part[k]);
  return block_max(m, red);
}

// 1. max of the raw density (deposit.py:183)
__global__ __launch_bounds__(kT) void df_max_kernel(const double *__restrict__ dens, int64_t N,
                                                    double *__restrict__ part) {
  __shared__ double red[kT / 64];
  double m = -INFINITY;
#pragma unroll 4
  for (int64_t e = (int64_t)blockIdx.x * kT + threadIdx.x; e < N; e += (int64_t)gridDim.x * kT)
    m = fmax(m, dens[e]);
  m = block_max(m, red);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// A tile of kTileX x kTileZ outputs and the inputs its smoothings read: rows
// [ra, rb) and columns [ca, cb), the outputs' windows or, at an edge, the
// first or last W of the line (the fit's rows there read them all); at most
// W + kTileX - 1 by W + kTileZ - 1 of them.
constexpr int kTileX = 8, kTileZ = 32;

struct Tile {
  int x0, z0, rows, cols, ra, rb, ca, cb;

  __device__ Tile(const SGRows &op, int nx, int nz, int t) {
    const int across = (nz + kTileZ - 1) / kTileZ;
    x0 = t / across * kTileX, z0 = t % across * kTileZ;
    rows = min(kTileX, nx - x0), cols = min(kTileZ, nz - z0);
    ra = max(0, min(x0 - op.h, nx - op.W)), rb = min(nx, max(x0 + kTileX + op.h, op.W));
    ca = max(0, min(z0 - op.h, nz - op.W)), cb = min(nz, max(z0 + kTileZ + op.h, op.W));
  }
};

int tiles_of(int nx, int nz) {
  return ((nx + kTileX - 1) / kTileX) * ((nz + kTileZ - 1) / kTileZ);
}

__host__ __device__ inline int tile_in(int W) { return (W + kTileX - 1) * (W + kTileZ - 1); }
__host__ __device__ inline int tile_mid(int W) { return kTileX * (W + kTileZ - 1); }
__host__ __device__ inline int tile_edge(int W) { return (W + kTileX + 1) * (W + kTileZ + 1); }

// Both smoothings of NF staged fields of a tile (in: rows of w values from
// (ra, ca)), axis 0 into mid, then axis 1; put(f, row, column, value).
template <int NF, typename Put>
__device__ void sg_tile(const SGRows &op, const Tile &t, int nx, int nz, const double *in,
                        double *mid, const Put &put) {
  const int w = t.cb - t.ca, nin = tile_in(op.W), nmid = tile_mid(op.W);
  double v[NF];
  for (int e = threadIdx.x; e < t.rows * w; e += kT) {
    const int r = e / w, c = e - r * w;
    const double *col = in + c;
    sg_at(op, [&](int f, int k) { return col[f * nin + (k - t.ra) * w]; }, nx, t.x0 + r, v);
#pragma unroll
    for (int f = 0; f < NF; ++f) mid[f * nmid + e] = v[f];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < t.rows * t.cols; e += kT) {
    const int r = e / t.cols, c = e - r * t.cols;
    const double *row = mid + r * w;
    sg_at(op, [&](int f, int k) { return row[f * nmid + k - t.ca]; }, nz, t.z0 + c, v);
#pragma unroll
    for (int f = 0; f < NF; ++f) put(f, t.x0 + r, t.z0 + c, v[f]);
  }
}

// 2. the velocity division and both smoothing axes of density and vx
// (deposit.py:183-184, 195-199), into S0 (density) and S1 (vx); partials of
// trapz(trapz(density, x_grids, axis=0), z_grids) (deposit.py:201), as the
// sum of each value times half its neighbouring spacings, and of the
// smoothed density's extremes
__global__ __launch_bounds__(kT) void df_sg_kernel(SGOp arg, const double *__restrict__ dens,
                                                   const double *__restrict__ vx, Axis gx, Axis gz,
                                                   double vt, double *__restrict__ part, int np, int nraw,
                                                   int ntiles, double *__restrict__ S0,
                                                   double *__restrict__ S1) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  __shared__ double red[kT / 64], each[3][kT / 64];
  const int nx = gx.n, nz = gz.n, nin = tile_in(arg.W), nmid = tile_mid(arg.W);
  const SGRows op = sg_rows(arg, lds + 2 * (nin + nmid));
  const auto stage = [&](const Tile &t) {
    const int w = t.cb - t.ca;
    for (int e = threadIdx.x; e < (t.rb - t.ra) * w; e += kT) {
      const int r = e / w, c = e - r * w;
      const int64_t g = (int64_t)(t.ra + r) * nz + (t.ca + c);
      lds[e] = dens[g];
      lds[nin + e] = vx[g];
    }
  };
  stage(Tile(op, nx, nz, blockIdx.x));
  const double thr = max_of(part + P_RAW * np, nraw, red) / vt;
  double sum = 0.0, hi = -INFINITY, lo = INFINITY;
  for (int i = blockIdx.x; i < ntiles; i += gridDim.x) {
    const Tile t(op, nx, nz, i);
    if (i != blockIdx.x) stage(t);
    // each thread divides what it staged
    for (int e = threadIdx.x; e < (t.rb - t.ra) * (t.cb - t.ca); e += kT) {
      const double d = lds[e], v = lds[nin + e];
      if (d > thr) lds[nin + e] = v / d;
    }
    __syncthreads();
    sg_tile<2>(op, t, nx, nz, lds, lds + 2 * nin, [&](int f, int r, int c, double v) {
      (f == 0 ? S0 : S1)[(int64_t)r * nz + c] = v;
      if (f != 0) return;
      const double wx = 0.5 * (gx.width(r - 1) + gx.width(r));
      const double wz = 0.5 * (gz.width(c - 1) + gz.width(c));
      if (nx > 1 && nz > 1) sum += v * wx * wz;
      hi = fmax(hi, v);
      lo = fmin(lo, v);
    });
    __syncthreads();
  }
  const double w[3] = {wave_sum(sum), wave_max(hi), wave_max(-lo)};
  to_waves(w, each);
  if (threadIdx.x != 0) return;
  sum = each[0][0], hi = each[1][0], lo = each[2][0];
#pragma unroll
  for (int k = 1; k < kT / 64; ++k) {
    sum += each[0][k];
    hi = fmax(hi, each[1][k]);
    lo = fmax(lo, each[2][k]);
  }
  part[P_SUM * np + blockIdx.x] = sum;
  part[P_MAX * np + blockIdx.x] = hi;
  part[P_MIN * np + blockIdx.x] = -lo;
}

// What the partials of the first two passes give: the raw density's maximum,
// dsum, and the normalised density's maximum, the extreme of the smoothed
// one that the division by dsum makes the largest (rounding is monotone, so
// it is that maximum bit for bit; -inf when every quotient is NaN).  One
// barrier for the four.
struct DensitySum {
  double raw, dsum, dmax;
  __device__ DensitySum(const double *part, int np, int nraw, int n) {
#pragma clang fp contract(off)
    __shared__ double red[4][kT / 64];
    double v = -INFINITY, s = 0.0, hi = -INFINITY, lo = INFINITY;
    for (int k = threadIdx.x; k < nraw; k += kT) v = fmax(v, part[P_RAW * np + k]);
    for (int k = threadIdx.x; k < n; k += kT) {
      s += part[P_SUM * np + k];
      hi = fmax(hi, part[P_MAX * np + k]);
      lo = fmin(lo, part[P_MIN * np + k]);
    }
    const double w[4] = {wave_max(v), wave_sum(s), wave_max(hi), wave_max(-lo)};
    to_waves(w, red);
    raw = red[0][0], dsum = red[1][0], hi = red[2][0], lo = red[3][0];
#pragma unroll
    for (int k = 1; k < kT / 64; ++k) {
      raw = fmax(raw, red[0][k]);
      dsum += red[1][k];
      hi = fmax(hi, red[2][k]);
      lo = fmax(lo, red[3][k]);
    }
    dmax = fmax(hi / dsum, -lo / dsum);
    if (dmax != dmax) dmax = -INFINITY;
  }
};

// 3. density and vx take their normalised and thresholded values
// (deposit.py:202, 204), their gradients (deposit.py:212-213) are smoothed
// along both axes (deposit.py:215-224), and the smoothed vx_x above
// 8 max / vt leaves partials of its mean (deposit.py:233-235)
__global__ __launch_bounds__(kT) void df_grad_kernel(
    SGOp arg, const double *__restrict__ S0, const double *__restrict__ S1, Axis gx, Axis gz,
    double vt, double *__restrict__ part, int np, int nraw, int nsum, int ntiles,
    double *__restrict__ dens, double *__restrict__ vx, double *__restrict__ o0,
    double *__restrict__ o1, double *__restrict__ o2) {
#pragma clang fp contract(off)
  extern __shared__ double lds[];
  __shared__ double each[2][kT / 64];
  const int nx = gx.n, nz = gz.n, nin = tile_in(arg.W), nedge = tile_edge(arg.W);
  double *const D = lds, *const V = D + nedge, *const G = V + nedge, *const mid = G + 3 * nin;
  double *const rows = mid + 3 * tile_mid(arg.W);
  GradAt *const wx = reinterpret_cast<GradAt *>(rows + sg_rows_size(arg.W));
  GradAt *const wz = wx + arg.W + kTileX;
  const SGRows op = sg_rows(arg, rows);
  // one more row and column on each side for the gradients
  struct Edge {
    int ea, fa, eh, ew;
    __device__ Edge(const Tile &t, int nx, int nz)
        : ea(max(0, t.ra - 1)), fa(max(0, t.ca - 1)), eh(min(nx, t.rb + 1) - ea),
          ew(min(nz, t.cb + 1) - fa) {}
  };
  const auto stage = [&](const Edge &m) {
    for (int e = threadIdx.x; e < m.eh * m.ew; e += kT) {
      const int r = e / m.ew, c = e - r * m.ew;
      const int64_t g = (int64_t)(m.ea + r) * nz + (m.fa + c);
      D[e] = S0[g];
      V[e] = S1[g];
    }
  };
  stage(Edge(Tile(op, nx, nz, blockIdx.x), nx, nz));
  const DensitySum q(part, np, nraw, nsum);
  const double thr = q.raw / vt, dsum = q.dsum, thr2 = q.dmax / vt * 8;
  double s = 0.0, c1 = 0.0;
  for (int i = blockIdx.x; i < ntiles; i += gridDim.x) {
    const Tile t(op, nx, nz, i);
    const Edge m(t, nx, nz);
    const int ea = m.ea, fa = m.fa, ew = m.ew;
    if (i != blockIdx.x) stage(m);
    // each thread normalises what it staged
    for (int e = threadIdx.x; e < m.eh * ew; e += kT) {
      const int r = e / ew, c = e - r * ew;
      const double d = D[e] / dsum, v = d <= thr ? 0.0 : V[e];
      D[e] = d;
      V[e] = v;
      const int x = ea + r - t.x0, z = fa + c - t.z0;
      if (x >= 0 && x < t.rows && z >= 0 && z < t.cols) {
        const int64_t g = (int64_t)(ea + r) * nz + (fa + c);
        dens[g] = d, vx[g] = v;
      }
    }
    const int w = t.cb - t.ca;
    for (int e = threadIdx.x; e < t.rb - t.ra + w; e += kT) {
      const int k = e - (t.rb - t.ra);
      if (k < 0) wx[e] = grad_weights(gx, t.ra + e);
      else wz[k] = grad_weights(gz, t.ca + k);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < (t.rb - t.ra) * w; e += kT) {
      const int r = e / w, c = e - r * w, x = t.ra + r, z = t.ca + c;
      const int at = (x - ea) * ew + (z - fa);
      G[e] = grad_at(D + at, ew, gx, x, wx[r]);
      G[nin + e] = grad_at(D + at, 1, gz, z, wz[c]);
      G[2 * nin + e] = grad_at(V + at, ew, gx, x, wx[r]);
    }
    __syncthreads();
    sg_tile<3>(op, t, nx, nz, G, mid, [&](int f, int r, int c, double v) {
      (f == 0 ? o0 : f == 1 ? o1 : o2)[(int64_t)r * nz + c] = v;
      if (f != 2) return;
      const bool in = D[(r - ea) * ew + (c - fa)] > thr2;
      s += in ? v : 0.0;
      c1 += in ? 1.0 : 0.0;
    });
    __syncthreads();
  }
  const double w[2] = {wave_sum(s), wave_sum(c1)};
  to_waves(w, each);
  if (threadIdx.x != 0) return;
  s = each[0][0], c1 = each[1][0];
#pragma unroll
  for (int k = 1; k < kT / 64; ++k) s += each[0][k], c1 += each[1][k];
  part[P_FILL * np + blockIdx.x] = s;
  part[P_COUNT * np + blockIdx.x] = c1;
}

// 4. vx_x below 8 max / vt takes the mean of vx_x above it
// (deposit.py:233-235); the record of the slice
__global__ __launch_bounds__(kT) void df_fill_kernel(const double *__restrict__ dens, int64_t N,
                                                     double vt, const double *__restrict__ part,
                                                     int np, int nraw, int nsum, double *__restrict__ vxx,
                                                     double *__restrict__ info) {
#pragma clang fp contract(off)
  __shared__ double red[2 * (kT / 64)];
  double sum = 0.0, cnt = 0.0;
  for (int k = threadIdx.x; k < nsum; k += kT) {
    sum += part[P_FILL * np + k];
    cnt += part[P_COUNT * np + k];
  }
  const DensitySum q(part, np, nraw, nsum);
  const double thr2 = q.dmax / vt * 8;
  sum = block_sum(sum, red);
  cnt = block_sum(cnt, red + kT / 64);
  const double fill = cnt > 0.0 ? sum / cnt : NAN;   // np.mean of an empty selection
  for (int64_t e = (int64_t)blockIdx.x * kT + threadIdx.x; e < N; e += (int64_t)gridDim.x * kT)
    if (dens[e] < thr2) vxx[e] = fill;
  if (info && blockIdx.x == 0 && threadIdx.x == 0) {
    info[0] = q.raw;
    info[1] = q.dsum;
    info[2] = q.dmax;
    info[3] = fill;
  }
}

}  // namespace
}  // namespace dfcsr

using namespace dfcsr;

extern "C" int64_t dfcsr_df_workspace_bytes(int nbins_x, int nbins_z) {
  if (nbins_x < 1 || nbins_z < 1) return 0;
  const int64_t N = (int64_t)nbins_x * nbins_z;
  // The smoothed density and vx (2 N), then the partials: P_ROWS for each
  // workgroup, min(tiles, kMaxGrid) of them.  Up to 344 workgroups fit the
  // fixed 2056 doubles, and the smallest grid of more (2745 x 1) leaves N more.
  static_assert(P_ROWS * kMaxGrid <= 2745 + 2056 && P_ROWS * 342 <= 2056, "partials fit");
  return (3 * N + nbins_z + 2 * 1024 + 8) * 8 + 64;
}

extern "C" int dfcsr_df_process(double *density, double *vx, double *density_x,
                                double *density_z, double *vx_x, int nbins_x, double x_start,
                                double x_end, int nbins_z, double z_start, double z_end,
                                double velocity_threshold, int window, int order, double *info,
                                void *ws, int64_t ws_bytes, void *stream) {
  if (!density || !vx || !density_x || !density_z || !vx_x || !ws)
    return set_error(DFCSR_EINVAL, "df_process: NULL pointer");
  if (nbins_x < 1 || nbins_z < 1) return set_error(DFCSR_EINVAL, "df_process: bad grid");
  if ((int64_t)nbins_x * nbins_z > (int64_t)1 << 22)
    return set_error(DFCSR_ERANGE, "df_process: grid %d x %d above 4M cells", nbins_x, nbins_z);
  if (window > nbins_x || window > nbins_z)
    return set_error(DFCSR_EINVAL,
                     "df_process: If mode is 'interp', window_length must be less than or "
                     "equal to the size of x (window %d, grid %d x %d)",
                     window, nbins_x, nbins_z);
  if (ws_bytes < dfcsr_df_workspace_bytes(nbins_x, nbins_z))
    return set_error(DFCSR_ENOWS, "df_process: workspace too small");
  SGOp op;
  int rc = make_sg(window, order, &op);
  if (rc) return rc;
  const int nx = nbins_x, nz = nbins_z;
  const int64_t N = (int64_t)nx * nz;
  double *S0 = static_cast<double *>(ws), *S1 = S0 + N, *part = S1 + N;
  const int ntiles = tiles_of(nx, nz), g = ntiles < kMaxGrid ? ntiles : kMaxGrid;
  const int64_t mb = (N + kMaxPerBlock - 1) / kMaxPerBlock;
  const int graw = (int)(mb < kMaxGrid ? mb : kMaxGrid);
  const int np = g > graw ? g : graw;
  const int64_t fb = (N + kT - 1) / kT;
  const int fill = (int)(fb < kMaxGrid ? fb : kMaxGrid);
  const Axis gx = make_axis(x_start, x_end, nx), gz = make_axis(z_start, z_end, nz);
  const int pass = tile_in(op.W) + tile_mid(op.W), rows = sg_rows_size(op.W);
  const size_t lds1 = 8 * (size_t)(2 * pass + rows);
  const size_t lds2 = 8 * (size_t)(2 * tile_edge(op.W) + 3 * pass + rows) +
                      sizeof(GradAt) * (size_t)(2 * op.W + kTileX + kTileZ);
  hipStream_t s = as_stream(stream);
  hipLaunchKernelGGL(df_max_kernel, dim3(graw), dim3(kT), 0, s, density, N, part);
  hipLaunchKernelGGL(df_sg_kernel, dim3(g), dim3(kT), lds1, s, op, density, vx, gx, gz,
                     velocity_threshold, part, np, graw, ntiles, S0, S1);
  hipLaunchKernelGGL(df_grad_kernel, dim3(g), dim3(kT), lds2, s, op, S0, S1, gx, gz,
                     velocity_threshold, part, np, graw, g, ntiles, density, vx, density_x,
                     density_z, vx_x);
  hipLaunchKernelGGL(df_fill_kernel, dim3(fill), dim3(kT), 0, s, density, N, velocity_threshold,
                     part, np, graw, g, vx_x, info);
  DFCSR_LAUNCH_CHECK("df_process");
  return DFCSR_OK;
}

extern "C" int dfcsr_savgol_operator(int window, int order, double *c, double *edge) {
  // Host-side helper (no device work): interior stencil c[window] and the
  // left-edge rows edge[(window/2) * window] of the smoothing operator.
  SGOp op;
  int rc = make_sg(window, order, &op);
  if (rc) return rc;
  for (int j = 0; j < window; ++j) c[j] = op.c[j];
  for (int i = 0; i < window / 2; ++i)
    for (int j = 0; j < window; ++j) edge[i * window + j] = op.E[i][j];
  return DFCSR_OK;
}
