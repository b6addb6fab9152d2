// The wake by z lines: region 0 and the near regions of meshes whose
// observers share them along a z line.  Included by wake.hip.
//
// Off the chirp branch every observer of a z line shares the regions' x' rows
// and s' columns, and so the history row pair and its x fraction.  Lanes are
// neighbouring observers of one line and evaluate the same source point
// together.  |r - r'| is convex along the line, so the plane and z' indices
// that a (row, column)'s lookups can reach follow from the two end observers
// and the perpendicular: that window of the history is staged in LDS -- in
// float64 already interpolated along x, so a lookup reads four cells (160
// bytes) there instead of eight (320 bytes) through the L1, which bounds the
// phase form.  A column's lattice data are wave-uniform: scalar registers.
//   near regions (line_block): a workgroup takes a z line, a region and some
//     of its rows; a row's window covers as many columns as fit.
//   region 0 (far_line_block): its columns lie a slice or more apart, so each
//     (row, column) has its own window (2 or 3 planes, tens of z cells); a
//     wave stages those of several rows of one column, the next ones' loads
//     in flight over the points of the current ones.
// z lines are dealt round the XCDs and rows round the workgroups, since those
// near the bunch have most of the work (contiguous ranges per XCD: 1.3x
// slower at 128 x 128).  The rule is by_lines.
// Bound: vector ALU issue, about 95 (float64) and 125 (mixed) instructions a
// point; float64 near regions at 128 x 128, 430 slices: 76 % busy.  Measured, the phase and
// observer-major forms and this one: float64 128 x 128 mesh, 355 slices (near
// 5661 and 1610 us, region 0 3386 and 1134 us); float64 32 x 32, 91 slices (436
// and 320, 343 and 188 us); mixed 64 x 57, 187 slices (868 and 478, 549 and 360
// us); three mixed simulations batched (1207 and 875, 1282 and 482 us).
#pragma once

// What one column (fixed s') gives every observer of a z line: r - r' =
// (ax, ay) + x n_s - x' n', the lattice at s', rho, the trapezoid weight, the
// z' index at R = 0, n_s . tau', n_s - n'; for the mixed form also n'.(n_s -
// n') and e = tau'.n', a = tau'.tau', b = n'.n', with float32 copies.
struct LineColumn64 {
  double ax, ay, nx, ny, tx, ty, rho, w, uz0, p2, mx, my;
};
struct LineColumn : LineColumn64 {
  double P1, e, a, b;
  float ef, af, bf, pad;
};
static_assert(sizeof(LineColumn64) == kColFp64 * sizeof(double), "column stride");
static_assert(sizeof(LineColumn) == kColMixed * sizeof(double), "column stride");

// The column at s' = sp of the line whose observers have lattice o.
__device__ inline LineColumn make_line_column(const WakeTask &T, const HistAxes &A, const Lat6 &o,
                                              double sp, double w, double inv_ds) {
  const Lat6 c = lattice_at<true>(T.L, sp, inv_ds);
  LineColumn v;
  v.ax = o.X0 - c.X0;
  v.ay = o.Y0 - c.Y0;
  v.nx = c.nx;
  v.ny = c.ny;
  v.tx = c.tx;
  v.ty = c.ty;
  v.rho = rho_at(T.L, sp);
  v.w = w;
  v.uz0 = ((sp - T.P.t) - A.min_z) * A.iz;
  v.p2 = o.nx * c.tx + o.ny * c.ty;
  v.mx = o.nx - c.nx;
  v.my = o.ny - c.ny;
  v.e = c.tx * c.nx + c.ty * c.ny;
  v.a = c.tx * c.tx + c.ty * c.ty;
  v.b = c.nx * c.nx + c.ny * c.ny;
  v.P1 = c.nx * v.mx + c.ny * v.my;
  v.ef = (float)v.e;
  v.af = (float)v.a;
  v.bf = (float)v.b;
  v.pad = 0.0f;
  return v;
}

// Column e of the table of a line-form wake: z line, region 1 or 2, column.
__device__ inline void line_column(const WakeTask &T, int e, double *__restrict__ ws) {
  const int Nz = T.P.Nz;
  const int zl = e / (2 * Nz), q = e - zl * 2 * Nz;
  const int r = 1 + q / Nz, k = q % Nz;
  double xm, zm;
  mesh_point(T.P, zl, xm, zm);   // the line's first mesh point
  const double t = T.P.t, s = t + zm;
  Regions rg = {};
  make_regions(T.P, s, xm, t, rg);
  const double inv_ds = 1.0 / T.L.ds;
  const HistAxes A = make_axes(T.H);
  const Lat6 o = lattice_at<true>(T.L, s, inv_ds);
  double *line = ws + line_at(T, zl);
  if (q == 0)
    for (int j = 0; j < 3; ++j) {
      store_axis(line + 4 * j, rg.xa[j]);
      store_axis(line + 12 + 4 * j, rg.sa[j]);
    }
  const LineColumn v = make_line_column(T, A, o, rg.sa[r].at(k), rg.sa[r].w(k), inv_ds);
  double *out = line + kLineHead + (int64_t)q * T.cstride;
  if (T.cstride == kColMixed) *reinterpret_cast<LineColumn *>(out) = v;
  else *reinterpret_cast<LineColumn64 *>(out) = v;
}

// A column at a wave-uniform address, by scalar loads.  The empty asm keeps
// them together ahead of the point: sunk into its branches they are waited
// for two or three times.
__device__ inline double pinned(double v) {
  asm volatile("" : "+s"(v));
  return v;
}
__device__ inline float pinned(float v) {
  asm volatile("" : "+s"(v));
  return v;
}

template <bool kMixed>
__device__ inline LineColumn load_column(const double *at) {
  const auto p = (const __attribute__((address_space(4))) LineColumn *)(uintptr_t)at;
  LineColumn c;
  c.ax = p->ax, c.ay = p->ay, c.nx = p->nx, c.ny = p->ny, c.tx = p->tx, c.ty = p->ty;
  c.rho = p->rho, c.w = p->w, c.uz0 = p->uz0, c.p2 = p->p2, c.mx = p->mx, c.my = p->my;
  if (kMixed) {
    c.P1 = p->P1, c.e = p->e, c.a = p->a, c.b = p->b;
    c.ef = p->ef, c.af = p->af, c.bf = p->bf;
  }
  c.ax = pinned(c.ax), c.ay = pinned(c.ay), c.nx = pinned(c.nx), c.ny = pinned(c.ny);
  c.tx = pinned(c.tx), c.ty = pinned(c.ty), c.w = pinned(c.w), c.uz0 = pinned(c.uz0);
  c.p2 = pinned(c.p2), c.mx = pinned(c.mx), c.my = pinned(c.my);
  if (kMixed) {
    c.P1 = pinned(c.P1), c.e = pinned(c.e), c.a = pinned(c.a), c.b = pinned(c.b);
    c.ef = pinned(c.ef), c.af = pinned(c.af), c.bf = pinned(c.bf);
  }
  return c;
}

// A column every lane holds the same values of, as scalars.
__device__ inline void uniform_column(LineColumn &c) {
  c.ax = uniform(c.ax), c.ay = uniform(c.ay), c.nx = uniform(c.nx), c.ny = uniform(c.ny);
  c.tx = uniform(c.tx), c.ty = uniform(c.ty), c.rho = uniform(c.rho), c.uz0 = uniform(c.uz0);
  c.p2 = uniform(c.p2), c.mx = uniform(c.mx), c.my = uniform(c.my), c.P1 = uniform(c.P1);
  c.e = uniform(c.e), c.a = uniform(c.a), c.b = uniform(c.b);
  c.ef = uniform(c.ef), c.af = uniform(c.af), c.bf = uniform(c.bf);
}

// First and last index in [0, n) that lookups at u in [lo, hi] truncate to;
// false when none is valid.  The margin covers the rounding of u.
__device__ inline bool index_range(double lo, double hi, int n, int &i0, int &i1) {
  constexpr double margin = 1e-3;
  lo -= margin;
  hi += margin;
  if (!(hi > -1.0 && lo < (double)n)) return false;   // also NaN
  i0 = lo > 0.0 ? (int)lo : 0;
  i1 = hi < (double)(n - 1) ? (hi > 0.0 ? (int)hi : 0) : n - 1;
  return true;
}

// 1/sqrt(a) for a normal a > 0: the hardware estimate (relative error below
// 2^-22) and one third-order step y (1 + h / 2 + 3 h^2 / 8), h = 1 - a y^2,
// whose error is below h^3: a few ulp, three operations fewer than two Newton
// steps.
__device__ inline double rsqrt_third(double a) {
  const double y = __builtin_amdgcn_rsq(a);
  const double h = fma(-(a * y), y, 1.0);
  return fma(y, h * fma(h, 0.375, 0.5), y);
}

// What a lane (one observer of a z line) keeps for all its points: x, the
// velocity tau + vx n, and the line's normal and index axes.
struct LineObserver {
  double x, vel_x, vel_y, nx, ny, ut0, it, iz;
};

// The lane's observer ix of z line zl, and the x range of observers ixa..ixb.
// s, the lattice and the axes are the line's; x and vx the observer's.
__device__ inline LineObserver line_observer(const WakeTask &T, const HistAxes &A,
                                             const double *__restrict__ ws, int zl, int ixa,
                                             int ixb, int ix, double &xlo, double &xhi) {
  const int zb = T.P.mesh_zbins;
  const double *od0 = ws + obs_at(T, ixa * zb + zl), *od = ws + obs_at(T, ix * zb + zl);
  const double xe0 = od0[1], xe1 = ws[obs_at(T, ixb * zb + zl) + 1];
  xlo = fmin(xe0, xe1);   // x is linear along the line
  xhi = fmax(xe0, xe1);
  const double vx = od[8];
  LineObserver o;
  o.x = od[1];
  o.nx = uniform(od0[4]);
  o.ny = uniform(od0[5]);
  o.vel_x = od0[6] + vx * o.nx;
  o.vel_y = od0[7] + vx * o.ny;
  o.ut0 = uniform((T.P.t - A.min_t) * A.it);
  o.it = uniform(A.it);
  o.iz = uniform(A.iz);
  return o;
}

// Range of R over the observers x in [xlo, xhi] of a line for a source whose
// r - r' is (ax, ay) + x n: R^2 is a convex quadratic of x.
__device__ inline void line_range(double ax, double ay, double nx, double ny, double xlo,
                                  double xhi, double &R0, double &R1) {
  const double ex = ax + xlo * nx, ey = ay + xlo * ny;
  const double fx = ax + xhi * nx, fy = ay + xhi * ny;
  const double e2 = ex * ex + ey * ey, f2 = fx * fx + fy * fy;
  const double nn = nx * nx + ny * ny, xv = -(ax * nx + ay * ny);
  double m2 = fmin(e2, f2);
  if (xv > xlo * nn && xv < xhi * nn) {
    const double cr = ax * ny - ay * nx;
    m2 = fmin(m2, cr * cr / nn);
  }
  R0 = sqrt(m2);
  R1 = sqrt(fmax(e2, f2));
}

// Window [t0, t1] x [z0, z1] of first corners that the line's lookups from
// row x' = xp (history row xi) and a column can take; false when none can
// contribute: outside the history, or outside the rows' z spans (every
// integrand exactly 0, zspan_holds).  A column that may hold R = 0, where
// the reference's formula is 0/0, is always kept.
__device__ inline bool line_window(const DfcsrHistory &H, const LineObserver &o,
                                   const LineColumn &c, double xp, int xi, double xlo, double xhi,
                                   int &t0, int &t1, int &z0, int &z1) {
  double R0, R1;
  line_range(c.ax - xp * c.nx, c.ay - xp * c.ny, o.nx, o.ny, xlo, xhi, R0, R1);
  const bool zero = !(R0 > 1e-9);
  bool in = index_range(o.ut0 - R1 * o.it, o.ut0 - R0 * o.it, H.nt, t0, t1);
  in = in && index_range(c.uz0 + R0 * o.iz, c.uz0 + R1 * o.iz, H.Zi, z0, z1);
  if (in && H.zspan && t1 - t0 < 8 && !zero) {
    bool any = false;
    for (int ti = t0; ti <= t1; ++ti) {
      const uint32_t e = H.zspan[(int64_t)xi * H.cap + hist_slot(H, ti)];
      any = any || (z1 + 1 >= (int)(e & 0xffffu) && z0 <= (int)(e >> 16));
    }
    in = any;
  }
  if (!in && zero) {
    t0 = t1 = H.nt - 1;
    z0 = z1 = 0;
    in = true;
  }
  return in;
}

// A window of the history in LDS for one x' row: cells [plane - ta][z - za],
// nz cells a plane, for first corners in [ta, ta + nT) x [za, za + nZ) (nT =
// 0: this lane has no row).
template <typename Cell>
struct LineWindow {
  const Cell *cells;
  int ta, za, nz;
  unsigned nT, nZ;
  // The cell (lt, lz), by full-rate 24-bit multiplies.
  __device__ const Cell *at(unsigned lt, unsigned lz) const {
    const unsigned o = __umul24(__umul24(lt, (unsigned)nz) + lz, (unsigned)sizeof(Cell));
    return reinterpret_cast<const Cell *>(reinterpret_cast<const char *>(cells) + o);
  }
};

// Cells of a window of nT x nZ (at most 2^24: times a group of rows it still
// fits an int).
__device__ inline int window_cells(int nT, int nZ) { return min(nT, 0xfff) * min(nZ, 0xfff); }

// e / d of indices below 2^20 by the reciprocal inv = 1 / d: (e + 1/2) / d is
// at least 1 / (2 d) from an integer, far more than the rounding.
__device__ inline int small_div(int e, float inv) { return (int)(((float)e + 0.5f) * inv); }

template <bool kMixed>
struct LineForm;

// ---- float64 -------------------------------------------------------------------
template <>
struct LineForm<false> {
  typedef double Real;
  struct Cell {          // the five fields, interpolated along x to the row
    double f[DFCSR_CELL];
  };
  struct Coefs {};       // nothing per (lane, column)
  static constexpr int kPlanesExtra = 1;   // a lookup reads planes t0 and t0 + 1

  __device__ static Coefs coefs(const LineObserver &, const LineColumn &) { return {}; }

  __device__ static double2 scales(double xp, double rho) {
    const double s = 1 + xp * rho;
    return make_double2(s, recip_newton(s));
  }

  // The window cell (plane ti, z) of a row between x cells i0 and i0 + di:
  // its loads, and what they give at the row's x fraction xf.
  struct Raw {
    double a[DFCSR_CELL], b[DFCSR_CELL];
  };
  __device__ static void load(const DfcsrHistory &H, int64_t rowD, int i0, int di, int ti, int z,
                              Raw &r) {
    const double *a = H.cells + ((int64_t)hist_slot(H, ti) * H.Xi + i0) * rowD +
                      (int64_t)z * DFCSR_CELL;
    const double *b = a + di * rowD;
#pragma unroll
    for (int f = 0; f < DFCSR_CELL; ++f) r.a[f] = a[f];
#pragma unroll
    for (int f = 0; f < DFCSR_CELL; ++f) r.b[f] = b[f];
  }
  __device__ static void store(const Raw &r, double xf, Cell &out) {
#pragma unroll
    for (int f = 0; f < DFCSR_CELL; ++f) out.f[f] = fma(xf, r.b[f], (1 - xf) * r.a[f]);
  }

  // One point: lane observer o, column c (scalar), row x' = xp; adds its
  // integrand (CSR.py:645-775, csr_point's formula) times w to cz, cx when its
  // lookup falls on the window.
  __device__ static void point(const LineObserver &o, const LineColumn &c, const Coefs &,
                               double xp, double, double w, double2 sc, const LineWindow<Cell> &W,
                               double &cz, double &cx, unsigned &evaluated) {
    const double rx = (c.ax + o.x * o.nx) - xp * c.nx;
    const double ry = (c.ay + o.x * o.ny) - xp * c.ny;
    const double R2 = rx * rx + ry * ry;
    double iR = rsqrt_third(R2), R = R2 * iR;
    if (__any(R2 == 0.0)) {   // the reference's 0/0 and x/0
      asm volatile("");       // a branch, not selects on every point
      iR = R2 == 0.0 ? INFINITY : iR;
      R = R2 == 0.0 ? 0.0 : R;
    }
    const double ut = o.ut0 - R * o.it, uz = c.uz0 + R * o.iz;
    const int it = (int)ut, iz = (int)uz;   // truncation: (-1, 0) is index 0
    const unsigned lt = (unsigned)(it - W.ta), lz = (unsigned)(iz - W.za);
    if ((lt < W.nT) & (lz < W.nZ)) {
      ++evaluated;
      const double td = ut - (double)it, zd = uz - (double)iz;
      const Cell *s0 = W.at(lt, lz), *s1 = s0 + W.nz;
      const double t_0 = 1.0 - td, z_0 = 1.0 - zd;
      const double w00 = t_0 * z_0, w01 = t_0 * zd, w10 = td * z_0, w11 = td * zd;
      double f[DFCSR_CELL];
#pragma unroll
      for (int v = 0; v < DFCSR_CELL; ++v)
        f[v] = fma(w11, s1[1].f[v], fma(w10, s1[0].f[v], fma(w01, s0[1].f[v], w00 * s0[0].f[v])));
      const double dens = f[DFCSR_F_DENSITY], dens_x = f[DFCSR_F_DENSITY_X];
      const double vx_ret = f[DFCSR_F_VX], div_v = f[DFCSR_F_VX_X];
      const double dzs = f[DFCSR_F_DENSITY_Z] * sc.y;
      const double vr_x = c.tx + vx_ret * c.nx, vr_y = c.ty + vx_ret * c.ny;
      const double nab_x = dens_x * c.nx + dzs * c.tx;
      const double nab_y = dens_x * c.ny + dzs * c.ty;
      const double part1 = o.vel_x * vr_x + o.vel_y * vr_y;
      const double ddv = dens * div_v;
      const double num1 = (o.vel_x - part1 * vr_x) * nab_x + (o.vel_y - part1 * vr_y) * nab_y;
      const double pd = -(vr_x * nab_x + vr_y * nab_y) - ddv;
      const double p1 = rx * c.mx + ry * c.my;
      const double siR = sc.x * iR;
      cz += w * ((num1 - part1 * ddv) * siR);
      cx += w * ((p1 * iR * (iR * dens + pd) - c.p2 * pd) * siR);
    } else if (R2 == 0.0 && W.nT) {
      cz = cx = NAN;
    }
  }
};

// ---- mixed precision -------------------------------------------------------------
// csr_point_mixed's arithmetic: the float32 operations are the same, in the
// same order (time, x, z lerps), so a window cell keeps the values and time
// differences of both x cells.
template <>
struct LineForm<true> {
  typedef float Real;
  struct alignas(16) Cell {
    float v0[DFCSR_CELL], v1[DFCSR_CELL], d0[DFCSR_CELL], d1[DFCSR_CELL];   // x0, x1
  };
  struct Coefs {
    float D0, D1, D2, G0, G1, G2, A, B;
    double P0;
  };
  static constexpr int kPlanesExtra = 0;   // the differences stand for plane t0 + 1

  __device__ static Coefs coefs(const LineObserver &o, const LineColumn &c) {
    const double A = o.vel_x * c.tx + o.vel_y * c.ty, B = o.vel_x * c.nx + o.vel_y * c.ny;
    Coefs m;
    m.P0 = (c.ax + o.x * o.nx) * c.mx + (c.ay + o.x * o.ny) * c.my;
    m.D0 = (float)(B - A * c.e);
    m.D1 = (float)(-(A * c.b + B * c.e));
    m.D2 = (float)(-B * c.b);
    m.G0 = (float)(A * (1.0 - c.a));
    m.G1 = (float)(-(A * c.e + B * c.a));
    m.G2 = (float)(-B * c.e);
    m.A = (float)A;
    m.B = (float)B;
    return m;
  }

  __device__ static float2 scales(double xp, double rho) {
    const float s = fmaf((float)xp, (float)rho, 1.0f);
    return make_float2(s, __builtin_amdgcn_rcpf(s));
  }

  typedef Cell Raw;
  __device__ static void load(const DfcsrHistory &H, int64_t rowD, int i0, int di, int ti, int z,
                              Raw &r) {
    const int64_t at = ((int64_t)hist_slot(H, ti) * H.Xi + i0) * rowD + (int64_t)z * DFCSR_CELL;
    const float *v = H.cells32 + at, *d = H.dcells32 + at;
    const int64_t dx = di * rowD;
#pragma unroll
    for (int f = 0; f < DFCSR_CELL; ++f) {
      r.v0[f] = v[f];
      r.v1[f] = v[dx + f];
      r.d0[f] = d[f];
      r.d1[f] = d[dx + f];
    }
  }
  __device__ static void store(const Raw &r, double, Cell &out) { out = r; }

  // xfrac, w: the row's x fraction and trapezoid weight.
  __device__ static void point(const LineObserver &o, const LineColumn &c, const Coefs &m,
                               double xp, double xfrac, double w, float2 sc,
                               const LineWindow<Cell> &W, double &cz, double &cx,
                               unsigned &evaluated) {
    const double rx = (c.ax + o.x * o.nx) - xp * c.nx;
    const double ry = (c.ay + o.x * o.ny) - xp * c.ny;
    const double R2 = rx * rx + ry * ry;
    if (__any(R2 == 0.0)) {   // the reference's 0/0 (or +-inf): not a finite contribution
      asm volatile("");       // a branch, not selects on every point
      if (R2 == 0.0 && W.nT) cz = cx = NAN;
    }
    double y = (double)__builtin_amdgcn_rsqf((float)R2);
    y = y * (1.5 - 0.5 * R2 * y * y);   // one Newton step: ~1e-14 relative
    const double R = R2 * y;
    const double ut = o.ut0 - R * o.it, uz = c.uz0 + R * o.iz;
    const int it = (int)ut, iz = (int)uz;
    const unsigned lt = (unsigned)(it - W.ta), lz = (unsigned)(iz - W.za);
    if ((lt < W.nT) & (lz < W.nZ)) {
      ++evaluated;
      const float td = (float)(ut - (double)it), zd = (float)(uz - (double)iz);
      const float xd = (float)xfrac;
      const Cell *s0 = W.at(lt, lz);
      const Cell a = s0[0], b = s0[1];
      float f[DFCSR_CELL];
#pragma unroll
      for (int k = 0; k < DFCSR_CELL; ++k) {
        const float c00 = fmaf(td, a.d0[k], a.v0[k]);
        const float c01 = fmaf(td, b.d0[k], b.v0[k]);
        const float c10 = fmaf(td, a.d1[k], a.v1[k]);
        const float c11 = fmaf(td, b.d1[k], b.v1[k]);
        const float c0 = fmaf(xd, c10 - c00, c00);
        const float c1 = fmaf(xd, c11 - c01, c01);
        f[k] = fmaf(zd, c1 - c0, c0);
      }
      const float dens = f[DFCSR_F_DENSITY], dx = f[DFCSR_F_DENSITY_X], dz = f[DFCSR_F_DENSITY_Z];
      const float vr = f[DFCSR_F_VX], dv = f[DFCSR_F_VX_X];
      const float ce = c.ef, ca = c.af, cb = c.bf;
      const float g = dz * sc.y;
      const float Cd = fmaf(vr, fmaf(vr, m.D2, m.D1), m.D0);
      const float Cg = fmaf(vr, fmaf(vr, m.G2, m.G1), m.G0);
      const float part1 = fmaf(vr, m.B, m.A);
      const float vgrad = fmaf(dx, fmaf(vr, cb, ce), g * fmaf(vr, ce, ca));
      const float ddv = dens * dv;
      const float pd = -vgrad - ddv;
      const double p1 = m.P0 - xp * c.P1;
      const double p1R = p1 * y;
      const float q = (float)(p1R - c.p2);
      const float ir = (float)y;
      const float sir = sc.x * ir;
      const float Iz = sir * (fmaf(dx, Cd, g * Cg) - part1 * ddv);
      const float Ix = sir * fmaf((float)p1R * ir, dens, pd * q);
      const float wx = (float)w;
      cz += c.w * (double)(wx * Iz);
      cx += c.w * (double)(wx * Ix);
    }
  }
};

template <bool kMixed>
using LineScale = std::conditional_t<kMixed, float2, double2>;

// Whether s and an end column of region axis sa both lie outside the lattice
// table: there the reference's integrand is 0/0 (as wake_phase).
__device__ inline bool line_nan(const WakeTask &T, const double *od0, const LinAxis &sa) {
  if (od0[9] == 0.0) return false;
  const double inv_ds = 1.0 / T.L.ds;
  return !trunc_index((sa.at(0) - T.L.min_s) * inv_ds, T.L.ns).ok ||
         !trunc_index((sa.at(sa.n - 1) - T.L.min_s) * inv_ds, T.L.ns).ok;
}

// Hull [v0, v1) of the rows of xa inside the history (x' is monotone in j);
// hull: two shared ints.
__device__ inline void line_hull(const DfcsrHistory &H, const HistAxes &A, const LinAxis &xa,
                                 int *hull, int &v0, int &v1) {
  if (threadIdx.x == 0) {
    hull[0] = xa.n;
    hull[1] = -1;
  }
  __syncthreads();
  int lo = xa.n, hi = -1;
  for (int j = threadIdx.x; j < xa.n; j += blockDim.x) {
    const double ux = (xa.at(j) - A.min_x) * A.ix;
    if (ux > -1.0 && ux < (double)H.Xi) {
      lo = min(lo, j);
      hi = max(hi, j);
    }
  }
  if (lo <= hi) {
    atomicMin(&hull[0], lo);
    atomicMax(&hull[1], hi);
  }
  __syncthreads();
  v0 = __builtin_amdgcn_readfirstlane(hull[0]);
  v1 = max(__builtin_amdgcn_readfirstlane(hull[1]) + 1, v0);
}

__device__ inline void count_points(const WakeTask &T, unsigned evaluated, bool valid) {
  if (!T.P.points_evaluated) return;   // uniform: a diagnostic call
  unsigned long long c = valid ? evaluated : 0u;
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) c += __shfl_xor(c, d, 64);
  if ((threadIdx.x & 63) == 0 && c) atomicAdd(T.P.points_evaluated, c);
}

// ---- near regions -----------------------------------------------------------------
constexpr int kLineCols = 256;        // columns bounded at a time, one per thread
constexpr int kLineMinCols = 8;       // columns a window is shrunk to before it is tiled

// S rows side by side in a wave (64 / S observers) and per pass; threads and
// window bytes of a workgroup.  Four waves a SIMD either way; 512 threads share
// the larger window that two rows need (float64 32 x 32: 326 us against 398 us
// with 256 threads and 29600 bytes, where windows are tiled more often; 64
// observers prefer 256 threads: 1580 against 1706 us at 128 x 128).
template <int S>
struct LineSize {
  static constexpr int kThreads = S == 1 ? 256 : 512;
  static constexpr int kBytes = S == 1 ? 29600 : 64000;
};

template <bool kMixed, int S>
struct LineLds {
  typedef typename LineForm<kMixed>::Cell Cell;
  static constexpr int kCells = LineSize<S>::kBytes / sizeof(Cell);
  Cell slab[kCells];                                            // [row][plane][z]
  LineScale<kMixed> scale[S][kLineCols];
  int t0[kLineCols], t1[kLineCols], z0[kLineCols], z1[kLineCols];   // t0 > t1: skipped
  int hull[2];
};

template <bool kMixed, int S>
__device__ void line_block(const WakeTask &T, int l, const double *__restrict__ lines,
                           double *__restrict__ partials, LineLds<kMixed, S> &sh) {
  typedef LineForm<kMixed> Form;
  typedef typename Form::Cell Cell;
  constexpr int W = 64 / S, kCells = LineLds<kMixed, S>::kCells;
  constexpr int kLineThreads = LineSize<S>::kThreads;
  const DfcsrHistory &H = T.H;
  const PhasePlan pl = make_plan(T.P, T.cstride);
  const int xb = T.P.mesh_xbins, zb = T.P.mesh_zbins, Nz = T.P.Nz;
  const int per_line = pl.nog * pl.nB;
  const int zl = __builtin_amdgcn_readfirstlane(l / per_line), rem = l - zl * per_line;
  // observer group; region and row group
  const int og = __builtin_amdgcn_readfirstlane(rem / pl.nB), ph = rem - og * pl.nB;
  const int r = 1 + __builtin_amdgcn_readfirstlane(ph / pl.ng), rg = ph - (r - 1) * pl.ng;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane / W, ol = lane - sub * W;
  const int cstep = (kLineThreads / 64) / pl.obg;   // waves that share an observer block
  const int wob = wave % pl.obg, wcol = wave / pl.obg;
  const int ix = (og * pl.obg + wob) * W + ol;
  const bool valid = ix < xb;
  const int ixa = og * pl.obg * W, ixb = min(ixa + pl.obg * W, xb) - 1;   // the group
  const HistAxes A = make_axes(H);
  const LinAxis xa = load_axis(partials + line_at(T, zl) + 4 * r);
  const LinAxis sa = load_axis(partials + line_at(T, zl) + 12 + 4 * r);
  const double *od0 = partials + obs_at(T, ixa * zb + zl);
  // the group's partial sums: thread e < obg * W writes observer ixa + e
  const int we = threadIdx.x;
  const bool writer = we < pl.obg * W && ixa + we < xb;
  double *out = partials + T.part +
                ((int64_t)((writer ? ixa + we : ixa) * zb + zl) * (pl.nA + pl.nB) + pl.nA + ph) * 2;
  const bool single = xa.n < 2 || sa.n < 2;   // trapz over a single sample is 0
  const bool nan = !single && line_nan(T, od0, sa);
  int v0, v1;
  line_hull(H, A, xa, sh.hull, v0, v1);
  // rows dealt round the row groups, S at a time: rows near the bunch have
  // more live columns than the outer ones
  const int j0 = v0 + rg * S, jstep = pl.ng * S;
  if (single || nan || j0 >= v1) {   // uniform over the workgroup
    if (writer) out[0] = out[1] = nan ? NAN : 0.0;
    return;
  }
  double xlo, xhi;
  const LineObserver o = line_observer(T, A, partials, zl, ixa, ixb, valid ? ix : ixa, xlo, xhi);
  const int64_t rowD = (int64_t)DFCSR_CELL_ROW(H.Zi) * DFCSR_CELL;
  const double *cols = lines + line_at(T, zl) + kLineHead + (int64_t)(r - 1) * Nz * T.cstride;
  double acc_z = 0.0, acc_x = 0.0;
  unsigned evaluated = 0;
  for (int j = j0; j < v1; j += jstep) {
    const int nrow = min(S, v1 - j);               // rows of this pass
    const int row = min(sub, nrow - 1);            // this lane's
    const double xp = xa.at(j + row), wr = xa.w(j + row);
    const double fr = trunc_index((xp - A.min_x) * A.ix, H.Xi).frac;
    double cz = 0.0, cx = 0.0;
    for (int kc = 0; kc < Nz; kc += kLineCols) {
      const int nc = min(kLineCols, Nz - kc);
      // the index ranges of column kc + thread over the pass's rows
      __syncthreads();
      if ((int)threadIdx.x < nc) {
        LineColumn c;
        static_cast<LineColumn64 &>(c) = *reinterpret_cast<const LineColumn64 *>(
            cols + (int64_t)(kc + threadIdx.x) * T.cstride);
        int t0 = 0x7fffffff, t1 = -1, z0 = 0x7fffffff, z1 = -1;
        for (int q = 0; q < nrow; ++q) {
          const double xq = xa.at(j + q);
          const int xi = trunc_index((xq - A.min_x) * A.ix, H.Xi).i0;
          int a0, a1, b0, b1;
          if (line_window(H, o, c, xq, xi, xlo, xhi, a0, a1, b0, b1)) {
            t0 = min(t0, a0);
            t1 = max(t1, a1);
            z0 = min(z0, b0);
            z1 = max(z1, b1);
          }
          sh.scale[q][threadIdx.x] = Form::scales(xq, c.rho);
        }
        sh.t0[threadIdx.x] = t0;
        sh.t1[threadIdx.x] = t1;
        sh.z0[threadIdx.x] = z0;
        sh.z1[threadIdx.x] = z1;
      }
      __syncthreads();
      // columns [ka, kb) whose joint window fits; every wave finds the same
      int len = nc;
      for (int ka = 0; ka < nc;) {
        int kb, t0, t1, z0, z1;
        while (true) {
          kb = min(ka + len, nc);
          t0 = z0 = 0x7fffffff;
          t1 = z1 = -1;
          for (int k = ka + lane; k < kb; k += 64) {
            t0 = min(t0, sh.t0[k]);
            t1 = max(t1, sh.t1[k]);
            z0 = min(z0, sh.z0[k]);
            z1 = max(z1, sh.z1[k]);
          }
#pragma unroll
          for (int d = 32; d >= 1; d >>= 1) {
            t0 = min(t0, __shfl_xor(t0, d, 64));
            t1 = max(t1, __shfl_xor(t1, d, 64));
            z0 = min(z0, __shfl_xor(z0, d, 64));
            z1 = max(z1, __shfl_xor(z1, d, 64));
          }
          t0 = __builtin_amdgcn_readfirstlane(t0);
          t1 = __builtin_amdgcn_readfirstlane(t1);
          z0 = __builtin_amdgcn_readfirstlane(z0);
          z1 = __builtin_amdgcn_readfirstlane(z1);
          if (t1 < 0 || kb - ka <= kLineMinCols ||
              window_cells(t1 - t0 + 1 + Form::kPlanesExtra, z1 - z0 + 2) * S <= kCells)
            break;
          len = (kb - ka + 1) / 2;
        }
        if (t1 < 0) {   // nothing to look up
          ka = kb;
          continue;
        }
        // windows of the joint range that fit (one, unless kLineMinCols
        // columns' range does not): nT x nZ first corners each
        constexpr int X = Form::kPlanesExtra, room = kCells / S;
        int nT = t1 - t0 + 1, nZ = z1 - z0 + 1;
        if (window_cells(nT + X, nZ + 1) > room) {
          nT = min(nT, max(1, room / min(nZ + 1, room / 2) - X));
          nZ = min(nZ, room / (nT + X) - 1);
        }
        for (int ta = t0; ta <= t1; ta += nT)
          for (int za = z0; za <= z1; za += nZ) {
            const int wz = nZ + 1, wcells = (nT + X) * wz;
            const float icells = __builtin_amdgcn_rcpf((float)wcells);
            const float iwz = __builtin_amdgcn_rcpf((float)wz);
            __syncthreads();
            for (int e = threadIdx.x; e < nrow * wcells; e += kLineThreads) {
              const int q = S == 1 ? 0 : small_div(e, icells), w = e - q * wcells;
              const int p = small_div(w, iwz), z = w - p * wz;
              const TruncIdx X0 = trunc_index((xa.at(j + q) - A.min_x) * A.ix, H.Xi);
              typename Form::Raw raw;
              Form::load(H, rowD, X0.i0, X0.i1 - X0.i0, min(ta + p, H.nt - 1),
                         min(za + z, H.Zi), raw);
              Form::store(raw, X0.frac, sh.slab[e]);
            }
            __syncthreads();
            LineWindow<Cell> win;
            win.cells = sh.slab + row * wcells;
            win.ta = ta;
            win.za = za;
            win.nz = wz;
            win.nT = sub < nrow ? min(nT, t1 + 1 - ta) : 0;
            win.nZ = min(nZ, z1 + 1 - za);
            // this wave's live columns, 64 at a time, as bits of a scalar
            const unsigned long long mine =
                (cstep == 8 ? 0x0101010101010101ull
                            : cstep == 4 ? 0x1111111111111111ull
                            : cstep == 2 ? 0x5555555555555555ull : ~0ull) << wcol;
            for (int kw = ka & ~63; kw < kb; kw += 64) {
              const int kl = kw + lane;
              unsigned long long live =
                  __ballot(kl >= ka && kl < kb && sh.t0[min(kl, nc - 1)] <= sh.t1[min(kl, nc - 1)]);
              for (live &= mine; live; live &= live - 1) {
                const int k = kw + __builtin_ctzll(live);
                const LineColumn c = load_column<kMixed>(cols + (int64_t)(kc + k) * T.cstride);
                const typename Form::Coefs m = Form::coefs(o, c);
                Form::point(o, c, m, xp, fr, kMixed ? wr : c.w, sh.scale[row][k], win, cz, cx,
                            evaluated);
              }
            }
          }
        ka = kb;
      }
    }
    if (kMixed || sub < nrow) {   // the mixed points carry their row's weight
      acc_z += kMixed ? cz : wr * cz;
      acc_x += kMixed ? cx : wr * cx;
    }
  }
  count_points(T, evaluated, valid);
  __syncthreads();
  double *sums = reinterpret_cast<double *>(sh.slab);   // [wave][lane] z, then x
  sums[threadIdx.x] = acc_z;
  sums[kLineThreads + threadIdx.x] = acc_x;
  __syncthreads();
  if (!writer) return;
  const int b = we / W, e = we - b * W;   // block, lane within it
  double tz = 0.0, tx = 0.0;
  for (int w = b; w < kLineThreads / 64; w += pl.obg)
    for (int q = 0; q < S; ++q) {
      tz += sums[w * 64 + q * W + e];
      tx += sums[kLineThreads + w * 64 + q * W + e];
    }
  out[0] = tz;
  out[1] = tx;
}

// ---- region 0 -----------------------------------------------------------------------
// A wave's window cells (one a lane) and the most rows staged together.  Two
// cells a lane spill: float64 128 x 128 1190 us against 1156 us, 32 x 32 315
// against 190 us.
constexpr int kFarCells = 64, kFarRows = 8;

// A tile of a wave's work: rows, the joint range of their windows, and the
// part of it in LDS.
struct FarTile {
  int ra, n, ta, tb, za, zt, nT, nZ, tw, zw;
};

template <bool kMixed, int S>
struct FarLineLds {
  typedef typename LineForm<kMixed>::Cell Cell;
  Cell slab[kThreads / 64][kFarCells];
  LineScale<kMixed> scale[kThreads / 64][kMaxRows];
  double xp[kMaxRows], w[kMaxRows], frac[kMaxRows];
  int i0[kMaxRows], di[kMaxRows];
  int hull[2];
};

template <bool kMixed, int S>
__device__ void far_line_block(const WakeTask &T, int l, double *__restrict__ partials,
                               FarLineLds<kMixed, S> &sh) {
  typedef LineForm<kMixed> Form;
  typedef typename Form::Cell Cell;
  constexpr int W = 64 / S, X = Form::kPlanesExtra;
  const DfcsrHistory &H = T.H;
  const PhasePlan pl = make_plan(T.P, T.cstride);
  const int xb = T.P.mesh_xbins, zb = T.P.mesh_zbins, Nz = T.P.Nz;
  const int per_line = pl.nob * pl.nA;
  const int zl = __builtin_amdgcn_readfirstlane(l / per_line), rem = l - zl * per_line;
  const int ob = __builtin_amdgcn_readfirstlane(rem / pl.nA), g = rem - ob * pl.nA;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane / W, ol = lane - sub * W;
  const int ix = ob * W + ol;
  const bool valid = ix < xb;
  const int ixa = ob * W, ixb = min(ixa + W, xb) - 1;
  const int ncb = 4 * pl.nA, cb = 4 * g + wave;
  const int k0 = (int)((int64_t)cb * Nz / ncb), k1 = (int)((int64_t)(cb + 1) * Nz / ncb);
  const HistAxes A = make_axes(H);
  const double inv_ds = 1.0 / T.L.ds;
  const LinAxis xa = load_axis(partials + line_at(T, zl));
  const LinAxis sa = load_axis(partials + line_at(T, zl) + 12);
  const double *od0 = partials + obs_at(T, ixa * zb + zl);
  const bool writer = wave == 0 && sub == 0 && valid;
  double *out = partials + T.part +
                ((int64_t)((valid ? ix : ixa) * zb + zl) * (pl.nA + pl.nB) + g) * 2;
  const bool single = xa.n < 2 || sa.n < 2;   // trapz over a single sample is 0
  const bool nan = !single && line_nan(T, od0, sa);
  int v0, v1;
  line_hull(H, A, xa, sh.hull, v0, v1);
  if (single || nan) {   // uniform over the workgroup
    if (writer) out[0] = out[1] = nan ? NAN : 0.0;
    return;
  }
  double xlo, xhi;
  const LineObserver o = line_observer(T, A, partials, zl, ixa, ixb, valid ? ix : ixa, xlo, xhi);
  const Lat6 oL = {uniform(od0[2]), uniform(od0[3]), uniform(od0[4]),
                   uniform(od0[5]), uniform(od0[6]), uniform(od0[7])};
  const int64_t rowD = (int64_t)DFCSR_CELL_ROW(H.Zi) * DFCSR_CELL;
  Cell *slab = sh.slab[wave];
  double acc_z = 0.0, acc_x = 0.0;
  unsigned evaluated = 0;
  for (int b0 = v0; b0 < v1; b0 += kMaxRows) {   // uniform over the workgroup
    const int nr = min(kMaxRows, v1 - b0);
    __syncthreads();   // before the next rows overwrite the table
    if ((int)threadIdx.x < nr) {
      const double xp = xa.at(b0 + threadIdx.x);
      const TruncIdx Xi = trunc_index((xp - A.min_x) * A.ix, H.Xi);
      sh.xp[threadIdx.x] = xp;
      sh.w[threadIdx.x] = xa.w(b0 + threadIdx.x);
      sh.frac[threadIdx.x] = Xi.frac;
      sh.i0[threadIdx.x] = Xi.i0;
      sh.di[threadIdx.x] = Xi.i1 - Xi.i0;
    }
    __syncthreads();
    for (int k = k0; k < k1; ++k) {
      LineColumn c = make_line_column(T, A, oL, sa.at(k), 1.0, inv_ds);
      uniform_column(c);
      const typename Form::Coefs m = Form::coefs(o, c);
      // lane j: row j's window
      int t0 = 0x7fffffff, t1 = -1, z0 = 0x7fffffff, z1 = -1;
      if (lane < nr) {
        const double xq = sh.xp[lane];
        if (!line_window(H, o, c, xq, sh.i0[lane], xlo, xhi, t0, t1, z0, z1)) {
          t0 = z0 = 0x7fffffff;
          t1 = z1 = -1;
        }
        sh.scale[wave][lane] = Form::scales(xq, c.rho);
      }
      const unsigned long long live = __ballot(t1 >= 0);
      // Groups of n neighbouring rows (a power of two, S or more), as many as
      // leave every group's joint window within the wave's LDS: lane j ends
      // up with the joint window of its row's group.
      int n = 1;
      while (2 * n <= kFarRows) {
        const int a0 = min(t0, __shfl_xor(t0, n, 64)), a1 = max(t1, __shfl_xor(t1, n, 64));
        const int b0 = min(z0, __shfl_xor(z0, n, 64)), b1 = max(z1, __shfl_xor(z1, n, 64));
        const bool fits =
            a1 < 0 || window_cells(a1 - a0 + 1 + X, b1 - b0 + 2) * 2 * n <= kFarCells;
        if (n >= S && !__all(fits)) break;
        t0 = a0;
        t1 = a1;
        z0 = b0;
        z1 = b1;
        n *= 2;
      }
      double cz = 0.0, cx = 0.0;
      // Tiles: the rows [ra, ra + n) of a group and first corners [tw, tw +
      // nT) x [zw, zw + nZ) of their joint window; one per group, unless S
      // rows' window does not fit.
      const auto rows_from = [&](FarTile &t, int ra) {
        if (ra >= nr || !(live >> ra)) {   // no live row left
          t.ra = nr;
          return;
        }
        ra = (ra + __builtin_ctzll(live >> ra)) & ~(n - 1);   // its group: ta <= tb, za <= zt
        t.ra = ra;
        t.n = min(n, nr - ra);
        t.ta = t.tw = __builtin_amdgcn_readlane(t0, ra);
        t.tb = __builtin_amdgcn_readlane(t1, ra);
        t.za = t.zw = __builtin_amdgcn_readlane(z0, ra);
        t.zt = __builtin_amdgcn_readlane(z1, ra);
        t.nT = t.tb - t.ta + 1;
        t.nZ = t.zt - t.za + 1;
        if (window_cells(t.nT + X, t.nZ + 1) * t.n > kFarCells) {
          const int room = kFarCells / t.n;
          t.nT = min(t.nT, max(1, room / min(t.nZ + 1, room / 2) - X));
          t.nZ = min(t.nZ, room / (t.nT + X) - 1);
        }
      };
      const auto advance = [&](FarTile &t) {
        t.zw += t.nZ;
        if (t.zw <= t.zt) return;
        t.zw = t.za;
        t.tw += t.nT;
        if (t.tw <= t.tb) return;
        rows_from(t, t.ra + n);
      };
      // the tile's cells, one a lane: loads into registers, then to LDS
      typename Form::Raw raw;
      double raw_frac = 0.0;
      const auto issue = [&](const FarTile &t) {
        const int wz = t.nZ + 1, wcells = (t.nT + X) * wz;
        if (lane >= t.n * wcells) return;
        const int q = small_div(lane, __builtin_amdgcn_rcpf((float)wcells)), w = lane - q * wcells;
        const int p = small_div(w, __builtin_amdgcn_rcpf((float)wz)), z = w - p * wz;
        raw_frac = sh.frac[t.ra + q];
        Form::load(H, rowD, sh.i0[t.ra + q], sh.di[t.ra + q], min(t.tw + p, H.nt - 1),
                   min(t.zw + z, H.Zi), raw);
      };
      const auto commit = [&](const FarTile &t) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (lane < t.n * (t.nT + X) * (t.nZ + 1)) Form::store(raw, raw_frac, slab[lane]);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      };
      FarTile cur, next;
      rows_from(cur, 0);
      if (cur.ra < nr) issue(cur);
      while (cur.ra < nr) {
        commit(cur);
        next = cur;
        advance(next);
        if (next.ra < nr) issue(next);   // in flight over this tile's points
        const int wz = cur.nZ + 1, wcells = (cur.nT + X) * wz;
        for (int q = 0; q < cur.n; q += S) {
          if (!((live >> (cur.ra + q)) & (S == 2 ? 3 : 1))) continue;
          const int r = cur.ra + min(q + sub, cur.n - 1);
          LineWindow<Cell> win;
          win.cells = slab + (r - cur.ra) * wcells;
          win.ta = cur.tw;
          win.za = cur.zw;
          win.nz = wz;
          win.nT = q + sub < cur.n ? min(cur.nT, cur.tb + 1 - cur.tw) : 0;
          win.nZ = min(cur.nZ, cur.zt + 1 - cur.zw);
          Form::point(o, c, m, sh.xp[r], sh.frac[r], sh.w[r], sh.scale[wave][r], win, cz, cx,
                      evaluated);
        }
        cur = next;
      }
      const double wk = sa.w(k);
      acc_z += wk * cz;
      acc_x += wk * cx;
    }
  }
  count_points(T, evaluated, valid);
  __syncthreads();
  double *sums = reinterpret_cast<double *>(sh.slab[0]);   // [wave][lane] z, then x
  sums[threadIdx.x] = acc_z;
  sums[kThreads + threadIdx.x] = acc_x;
  __syncthreads();
  if (!writer) return;
  double tz = 0.0, tx = 0.0;
  for (int b = ol; b < kThreads; b += W) {
    tz += sums[b];
    tx += sums[kThreads + b];
  }
  out[0] = tz;
  out[1] = tx;
}

// Logical workgroup of a line-form launch: whole z lines dealt round the
// XCDs, since the lines near the bunch carry most of the work.
__device__ inline int line_group(const WakeTask &T, int b, int nb) {
  return xcd_group<false>(b, nb, nb / T.P.mesh_zbins);
}

template <bool kMixed, int S>
__global__ __launch_bounds__(kThreads, 4) void wake_far_line_kernel(
    WakeTask T, double *__restrict__ partials) {
  __shared__ FarLineLds<kMixed, S> sh;
  far_line_block<kMixed, S>(T, line_group(T, blockIdx.x, gridDim.x), partials, sh);
}

template <bool kMixed, int S>
__global__ __launch_bounds__((LineSize<S>::kThreads), 4) void wake_line_kernel(
    WakeTask T, const double *__restrict__ lines, double *__restrict__ partials) {
  __shared__ LineLds<kMixed, S> sh;
  line_block<kMixed, S>(T, line_group(T, blockIdx.x, gridDim.x), lines, partials, sh);
}
