// a3: cloud-in-cell deposition with two-word fixed-point sums.
//
// Replaces histogram_cic_2d (deposit.py:42-87) and the pair of calls in
// DF_tracker.get_DF (deposit.py:172-182).  Cell indices use the reference's
// FP64 expression cell = (q - start) * (1 / ((end - start) / nbins)),
// i = floor(cell), S = 1 - (cell - i), evaluated without fused multiply-add
// so they are bit-identical to the reference.  Each corner weight w*S1*S2 is
// split into two signed integers, its multiple of 2^-k and the remainder's
// multiple of 2^-(k + d), and both are summed as 64-bit integers.  Integer
// addition is associative, so the grid is the same for every launch order;
// k and d are chosen from n and max|w| so that no word can overflow, and the
// quantum 2^-(k + d) is 1e-22 or less of the largest weight (1e7 particles):
// the sums are exact to far below float64 rounding.
#include "common.h"

namespace dfcsr {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxBlocks = 512;

// ws layout: [0..3] k and d of grid A, then of grid B (as doubles),
//            [8 .. 8+kMaxBlocks) block max|w| partials,
//            then the words: per workgroup of the LDS form its tile's high
//            and low words, or (direct form) per grid nb1*nb2 of each.
constexpr int kHdr = 8 + kMaxBlocks;

int nblocks_for(int64_t n) {
  int64_t b = (n + kThreads * 4 - 1) / (kThreads * 4);
  if (b < 1) b = 1;
  if (b > kMaxBlocks) b = kMaxBlocks;
  return (int)b;
}

// max|w| over the finite weights (a weight that is not finite deposits
// nothing).  Four loads in flight per thread: 80 MB in 13 us.
__global__ __launch_bounds__(kThreads) void absmax_partial(const double *__restrict__ w, int64_t n,
                                                           double *__restrict__ part) {
  __shared__ double red[kThreads / 64];
  double m = 0.0;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  for (; i + 3 * stride < n; i += 4 * stride) {
    double v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) v[k] = fabs(w[i + k * stride]);
#pragma unroll
    for (int k = 0; k < 4; ++k) m = v[k] < INFINITY ? fmax(m, v[k]) : m;
  }
  for (; i < n; i += stride) {
    const double v = fabs(w[i]);
    m = v < INFINITY ? fmax(m, v) : m;
  }
  m = block_max(m, red);
  if (threadIdx.x == 0) part[blockIdx.x] = m;
}

// Fixed-point format of one grid.  A weight v is s = v 2^k = hi + r with
// hi = rint(s), |r| <= 1/2, and lo = rint(r 2^d).  n max|w| 2^k < 2^62 keeps
// the sum of n high words in 63 bits, n 2^(d-1) < 2^63 that of the low ones in
// 64 (one bit less of d would be a coarser quantum from 2^30 particles on than
// one word of 94 bits has); |s| < 2^50 and d <= 50 let the conversions add 1.5 2^52 and read the
// integer from the mantissa (4 operations a word, against about 15 for a
// float64 -> int64 conversion).
struct FxScale {
  int k, d;
  double up, up_lo;   // 2^k, 2^d
};

__device__ inline FxScale fx_scale(double max_w, int64_t n) {
  FxScale f;
  int e = 0, en = 0;
  frexp((double)(n < 1 ? 1 : n), &en);   // n < 2^en
  if (max_w > 0.0) frexp(max_w, &e);     // max|w| < 2^e
  f.k = min(62 - e - en, 50 - e);
  f.k = max_w > 0.0 ? min(f.k, 900) : 0;
  f.d = min(64 - en, 50);
  f.up = ldexp(1.0, f.k);
  f.up_lo = ldexp(1.0, f.d);
  return f;
}

struct FxWords {
  long long hi, lo;
};

__device__ inline FxWords fx_words(double v, const FxScale &f) {
#pragma clang fp contract(off)
  constexpr double M = 0x1.8p52;
  const double s = v * f.up;      // exact: a power of two
  const double h = s + M;
  const double r = s - (h - M);   // exact
  const double l = r * f.up_lo + M;
  FxWords w;
  w.hi = __double_as_longlong(h) - __double_as_longlong(M);
  w.lo = __double_as_longlong(l) - __double_as_longlong(M);
  return w;
}

// (hi + lo 2^-d) 2^-k.  The low word's whole units are carried into the high
// one, so what is left of it is half a unit or less and nothing cancels: below
// 2^53 units hi is exact and the sum is rounded once, past that it is within
// 1.5 times that rounding.
__device__ inline double fx_value(long long hi, long long lo, const FxScale &f) {
  long long carry = lo >> f.d;
  long long rest = lo - (carry << f.d);   // in [0, 2^d)
  if (rest >> (f.d - 1)) {
    ++carry;
    rest -= 1ll << f.d;
  }
  return ((double)(hi + carry) + (double)rest * (1.0 / f.up_lo)) * (1.0 / f.up);
}

// The format that a deposition kernel left in hdr (k and d as doubles).
__device__ inline FxScale fx_stored(const double *hdr) {
  FxScale f;
  f.k = (int)hdr[0];
  f.d = (int)hdr[1];
  f.up = ldexp(1.0, f.k);
  f.up_lo = ldexp(1.0, f.d);
  return f;
}

// Block reduction of the max|w| partials (0 without a weight).
__device__ inline double max_weight(const double *part, int npart, double *red) {
  double m = 0.0;
  for (int b = threadIdx.x; b < npart; b += blockDim.x) m = fmax(m, part[b]);
  return block_max(m, red);
}

__global__ __launch_bounds__(kThreads) void zero_i64(int64_t *__restrict__ a, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) a[i] = 0;
}

// Cell of one particle along an axis: floor index (or -8 when far off the
// grid: only to fail the range tests) and the lower corner's weight.
struct CicAxis {
  int i;
  double S;
};

__device__ inline CicAxis cic_axis(double q, double start, double inv, int nb) {
#pragma clang fp contract(off)
  const double c = (q - start) * inv;
  const double f = floor(c);
  CicAxis a;
  a.i = (f > -4.0 && f < (double)nb + 4.0) ? (int)f : -8;
  a.S = 1.0 - (c - f);
  return a;
}

// A weight that is not finite deposits nothing.
__device__ inline double fx_weight(double w) { return fabs(w) < INFINITY ? w : 0.0; }

// ---- particles' cells (parity outputs) --------------------------------------
// cell_index[2 p + {0, 1}] = floor of the exact cell coordinates, saturated
// to int32; cell_count += 1 at the lower cell when it lies on the grid.
__global__ __launch_bounds__(kThreads) void cic_cells_kernel(
    const double *__restrict__ q1, const double *__restrict__ q2, int64_t n, int nb1,
    double start1, double inv1, int nb2, double start2, double inv2,
    int32_t *__restrict__ cell_index, int32_t *__restrict__ cell_count) {
#pragma clang fp contract(off)
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  for (int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x; p < n; p += stride) {
    const double f1 = floor((q1[p] - start1) * inv1), f2 = floor((q2[p] - start2) * inv2);
    if (cell_index) {
      const double g1 = fmin(fmax(f1, -2147483648.0), 2147483647.0);
      const double g2 = fmin(fmax(f2, -2147483648.0), 2147483647.0);
      cell_index[2 * p] = isnan(f1) ? INT32_MIN : (int32_t)g1;
      cell_index[2 * p + 1] = isnan(f2) ? INT32_MIN : (int32_t)g2;
    }
    if (cell_count && f1 >= 0.0 && f1 < (double)nb1 && f2 >= 0.0 && f2 < (double)nb2)
      atomicAdd(cell_count + (int64_t)f1 * nb2 + (int64_t)f2, 1);
  }
}

__global__ __launch_bounds__(kThreads) void zero_i32(int32_t *__restrict__ a, int64_t n) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) a[i] = 0;
}

// ---- direct form: global atomics ---------------------------------------------
// For grids whose row tiles do not suit LDS (tile_plan), and few particles on
// many tiles (few_on_many).  blockIdx.y: the
// grid (0: weights wA, 1: weights wB; null: unit weights).
__global__ __launch_bounds__(kThreads) void cic_kernel(
    const double *__restrict__ q1, const double *__restrict__ q2,
    const double *__restrict__ wA, const double *__restrict__ wB, int64_t n, int nb1,
    double start1, double inv1, int nb2, double start2, double inv2, double *__restrict__ hdr,
    int npart, int64_t *__restrict__ acc) {
#pragma clang fp contract(off)
  __shared__ double red[kThreads / 64];
  const double *w = blockIdx.y ? wB : wA;
  const FxScale f = fx_scale(w ? max_weight(hdr + 8, npart, red) : 1.0, n);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    hdr[2 * blockIdx.y] = f.k;
    hdr[2 * blockIdx.y + 1] = f.d;
  }
  const int64_t nc = (int64_t)nb1 * nb2;
  unsigned long long *hi = reinterpret_cast<unsigned long long *>(acc) + blockIdx.y * 2 * nc;
  unsigned long long *lo = hi + nc;
  const int64_t stride = (int64_t)gridDim.x * kThreads;
  for (int64_t p = (int64_t)blockIdx.x * kThreads + threadIdx.x; p < n; p += stride) {
    const CicAxis A = cic_axis(q1[p], start1, inv1, nb1), B = cic_axis(q2[p], start2, inv2, nb2);
    const double wa = w ? fx_weight(w[p]) : 1.0;
    const bool a[2] = {A.i >= 0 && A.i < nb1, A.i + 1 >= 0 && A.i + 1 < nb1};
    const bool b[2] = {B.i >= 0 && B.i < nb2, B.i + 1 >= 0 && B.i + 1 < nb2};
    // Corner weights in the reference's association: (w*S1)*S2.
    const double t0 = wa * A.S, t1 = wa * (1.0 - A.S);
    const double t[4] = {t0 * B.S, t0 * (1.0 - B.S), t1 * B.S, t1 * (1.0 - B.S)};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      if (!(a[c >> 1] && b[c & 1])) continue;
      const FxWords v = fx_words(t[c], f);
      const int64_t cell = (int64_t)(A.i + (c >> 1)) * nb2 + B.i + (c & 1);
      if (v.hi) atomicAdd(hi + cell, (unsigned long long)v.hi);
      if (v.lo) atomicAdd(lo + cell, (unsigned long long)v.lo);
    }
  }
}

__global__ __launch_bounds__(kThreads) void fx_to_double(const int64_t *__restrict__ acc,
                                                         const double *__restrict__ hdr, int64_t n,
                                                         double *__restrict__ outA,
                                                         double *__restrict__ outB) {
  double *out = blockIdx.y ? outB : outA;
  const int64_t *hi = acc + blockIdx.y * 2 * n, *lo = hi + n;
  const FxScale f = fx_stored(hdr + 2 * blockIdx.y);
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    out[i] = fx_value(hi[i], lo[i], f);
}

// ---- LDS form -----------------------------------------------------------------
// A workgroup of 1024 threads owns one tile of one grid (density or vx) in
// LDS, 16 bytes a cell, and a chunk of the particles; it adds the corners
// that fall on its tile with 64-bit LDS atomics and stores the tile's words
// once, without atomics, for tile_sum_kernel to add up.  Tiles: groups of G
// rows dealt round the T tiles (row i in tile (i / G) % T), so a bunch whose
// rows carry very different numbers of particles still loads the tiles alike.
// Each grid has workgroups of its own: at 100 x 100 cells a whole grid is one
// tile, every lane works on every particle, and a particle's cell (25 of
// about 120 operations) is all that is computed twice.
// Bound: LDS atomics (8 per particle and grid, spread over the banks).
// kQueue (T > 2, where most of a wave's particles miss its tile): the wave
// scans x alone and queues the hits in LDS; every 64 of them are deposited by
// a full wave.
// Measured (both grids, whole call): 1e7 particles on 100 x 100 114 us (544 us
// with 48 KB row tiles, which left most lanes idle, and a flush by global
// atomics), 5e6 on 128 x 128 95 us; 3e6 on 256 x 256 98 us (2157 us with 16
// global atomics a particle, about 17 G atomics/s); 1e5 on 64 x 64 18 us (32).
constexpr int kTileThreads = 1024;
constexpr int kLdsBytes = 160 * 1024 - 256;   // a CU's LDS, less the static part
constexpr int kQueueLen = 128;                                   // per wave
constexpr int kQueueBytes = (kTileThreads / 64) * kQueueLen * 4;
constexpr int kMaxTiles = 64;
constexpr int kMaxWg = 256;                                      // one per CU
constexpr int kMinPer = 4096;                                    // particles per workgroup

struct TilePlan {
  int T, G, rows;    // tiles, rows per group, rows per tile (T = 0: direct form)
  int cells;         // rows * nb2
  size_t lds;        // bytes
};

// Fewest tiles that fit; larger row groups first (a particle's two rows are
// then in one tile more often).  Every tile scans all particles, so the gain
// over the direct form falls with the number of tiles: 52 tiles (600 x 600)
// take 1.6 ms at 1e7 particles and 33 us at 2e4, the direct form's atomics
// 8.0 ms and 39 us; kMaxTiles keeps to that range.
TilePlan tile_plan(int nb1, int nb2) {
  TilePlan p = {0, 0, 0, 0, 0};
  const int64_t map = (int64_t)(nb1 + 2) * 4 + 16;   // rows -2 to nb1, rounded up
  for (int G = 4; G >= 1; G >>= 1) {
    const int groups = (nb1 + G - 1) / G;
    for (int T = 1; T <= kMaxTiles && T <= groups; ++T) {
      const int64_t rows = (int64_t)((groups + T - 1) / T) * G;
      const int64_t lds = rows * nb2 * 16 + map + (T > 2 ? kQueueBytes : 0);
      if (lds > kLdsBytes) continue;
      p.T = T;
      p.G = G;
      p.rows = (int)rows;
      p.cells = (int)rows * nb2;
      p.lds = (size_t)lds;
      return p;
    }
  }
  return p;
}

// Few particles on a grid of many tiles, or of many rows (each workgroup makes a
// map of them): zeroing and storing the tiles' LDS takes longer than the direct
// form's atomics.  Measured, both grids, tiles / direct, us: 640 x 640 (45
// tiles a grid) at 100 particles 27 / 16, at 1e4 33 / 21, at 3e4 34 / 35; 400 x
// 400 (17) 19 / 16, 25 / 20, 30 / 37; 20000 x 3 25 / 16, 28 / 20, 34 / 31; 300 x
// 300 (10) 16 / 17, 21 / 20, 28 / 40; one grid of 400 x 400 16 / 18, 20 / 19.
// Either way the sums, and so the grids, are the same.
constexpr int64_t kFewParticles = 10240;
constexpr int kManyTiles = 24, kManyRows = 8192;

bool few_on_many(const TilePlan &p, int ngrid, int nb1, int64_t n) {
  return n <= kFewParticles && (p.T * ngrid >= kManyTiles || nb1 >= kManyRows);
}

// Chunks of the particles per tile and grid: at most kMaxWg workgroups.
int tile_chunks(const TilePlan &t, int ngrid, int64_t n) {
  int64_t c = kMaxWg / (t.T * ngrid);
  const int64_t most = (n + kMinPer - 1) / kMinPer;
  if (c > most) c = most;
  return (int)(c < 1 ? 1 : c);
}

template <bool kQueue>
__global__ __launch_bounds__(kTileThreads) void cic_tile_kernel(
    const double *__restrict__ q1, const double *__restrict__ q2,
    const double *__restrict__ wA, const double *__restrict__ wB, int64_t n, int64_t per,
    int nb1, double start1, double inv1, int nb2, double start2, double inv2, int T, int G,
    int cells, double *__restrict__ hdr, int npart, unsigned long long *__restrict__ words) {
#pragma clang fp contract(off)
  extern __shared__ __align__(16) unsigned long long lds[];
  __shared__ double red[kTileThreads / 64];
  unsigned long long *hi = lds, *lo = lds + cells;
  // first cell of grid row i in the tile, at [i + 2]; -1 when the row is in
  // another tile or off the grid (i = -2, -1 and nb1), -2 when the next row is
  // in the tile
  int *rowmap = reinterpret_cast<int *>(lds + 2 * (size_t)cells);
  const int grid = blockIdx.y / T, tile = blockIdx.y - grid * T;
  const double *w = grid ? wB : wA;
  for (int e = threadIdx.x; e < 2 * cells; e += kTileThreads) lds[e] = 0ull;
  for (int i = (int)threadIdx.x - 2; i <= nb1; i += kTileThreads) {
    const int g = i / G, h = (i + 1) / G;
    const bool in = i >= 0 && i < nb1 && g % T == tile,
               after = i >= -1 && i + 1 < nb1 && h % T == tile;
    rowmap[i + 2] = in ? ((g / T) * G + (i - g * G)) * nb2 : after ? -2 : -1;
  }
  const FxScale f = fx_scale(w ? max_weight(hdr + 8, npart, red) : 1.0, n);
  if (blockIdx.x == 0 && tile == 0 && threadIdx.x == 0) {
    hdr[2 * grid] = f.k;
    hdr[2 * grid + 1] = f.d;
  }
  __syncthreads();

  const auto add = [&](int cell, double t) {
    const FxWords v = fx_words(t, f);
    atomicAdd(hi + cell, (unsigned long long)v.hi);
    atomicAdd(lo + cell, (unsigned long long)v.lo);
  };
  const auto deposit = [&](double x, double z, double wt) {
    const CicAxis A = cic_axis(x, start1, inv1, nb1), B = cic_axis(z, start2, inv2, nb2);
    if (A.i < -1 || A.i >= nb1) return;
    const int ra = rowmap[A.i + 2], rb = rowmap[A.i + 3];
    const bool b0 = B.i >= 0 && B.i < nb2, b1 = B.i + 1 >= 0 && B.i + 1 < nb2;
    // Corner weights in the reference's association: (w*S1)*S2.
    const double t0 = wt * A.S, t1 = wt * (1.0 - A.S);
    if (ra >= 0) {
      if (b0) add(ra + B.i, t0 * B.S);
      if (b1) add(ra + B.i + 1, t0 * (1.0 - B.S));
    }
    if (rb >= 0) {
      if (b0) add(rb + B.i, t1 * B.S);
      if (b1) add(rb + B.i + 1, t1 * (1.0 - B.S));
    }
  };
  const int64_t p0 = (int64_t)blockIdx.x * per, p1 = min(p0 + per, n);
  if (!kQueue) {
    // kAhead particles a lane at once, the next kAhead's loads in flight over
    // their sums (one: 1e7 on 100 x 100 119 us, 5e6 on 128 x 128 102; four: 114
    // and 95)
    constexpr int kAhead = 4;
    struct Batch {
      double x[kAhead], z[kAhead], w[kAhead];
    };
    const auto load = [&](int64_t p, Batch &b) {
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        const int64_t q = p + k * kTileThreads;
        const bool in = q < p1;
        b.x[k] = in ? q1[q] : NAN;   // off the grid
        b.z[k] = in ? q2[q] : 0.0;
        b.w[k] = in && w ? w[q] : 1.0;
      }
    };
    Batch cur, next;
    int64_t p = p0 + threadIdx.x;
    load(p, cur);
    while (p < p1) {
      p += kAhead * kTileThreads;
      load(p, next);
#pragma unroll
      for (int k = 0; k < kAhead; ++k) deposit(cur.x[k], cur.z[k], fx_weight(cur.w[k]));
      cur = next;
    }
  } else {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int *queue = rowmap + nb1 + 3 + wave * kQueueLen;
    int count = 0;   // wave-uniform
    // the last particles taken off the queue: their loads are in flight while
    // the scan goes on, their sums are made when the next ones are taken
    double hx = NAN, hz = 0.0, hw = 1.0;
    const auto drain = [&](int take) {
      deposit(hx, hz, fx_weight(hw));
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      hx = NAN;   // off the grid
      if (lane < take) {
        const int64_t p = p0 + queue[count - take + lane];
        hx = q1[p];
        hz = q2[p];
        if (w) hw = w[p];
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      count -= take;
    };
    // kScan groups of 64 particles a time, the next kScan in flight.  Every
    // tile of either grid scans all particles, so the scan's instructions bound
    // the kernel (3e6 on 256 x 256: 91 us with the hits' loads waited for and
    // the row tested against both ends, 88.3 with those loads in flight, 86
    // with two sets of scanned positions in turn, 81 with the clamped row; one
    // XCD for a chunk's tiles, so that they share its L2, made no difference)
    constexpr int kScan = 4;
    const auto load = [&](int64_t b, double (&x)[kScan]) {
#pragma unroll
      for (int k = 0; k < kScan; ++k) {
        const int64_t p = b + k * 64 + lane;
        x[k] = p < p1 ? q1[p] : NAN;   // misses every tile
      }
    };
    const auto scan = [&](int64_t b, const double (&x)[kScan]) {
      const int at = (int)(b - p0) + lane;
#pragma unroll
      for (int k = 0; k < kScan; ++k) {
        // off the grid (or NaN): rows -2 and nb1, which no tile holds
        const double u = fmin(fmax((x[k] - start1) * inv1, -2.0), (double)nb1);
        const bool hit = rowmap[(int)floor(u) + 2] != -1;
        const unsigned long long m = __ballot(hit);
        if (hit)
          queue[count + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32),
                                                  __builtin_amdgcn_mbcnt_lo((unsigned)m, 0))] =
              at + k * 64;
        count += __popcll(m);
        if (count >= 64) drain(64);
      }
    };
    constexpr int kStep = kTileThreads * kScan;
    double xa[kScan], xb[kScan];
    int64_t b = p0 + wave * (64 * kScan);
    load(b, xa);
    while (b < p1) {
      load(b + kStep, xb);
      scan(b, xa);
      load(b + 2 * kStep, xa);
      scan(b + kStep, xb);
      b += 2 * kStep;
    }
    if (count) drain(count);
    deposit(hx, hz, fx_weight(hw));
  }
  __syncthreads();
  unsigned long long *out = words + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 2 * cells;
  for (int e = threadIdx.x; e < 2 * cells; e += kTileThreads) out[e] = lds[e];
}

// Adds the chunks' words of each cell and converts the sums: 64 cells per
// workgroup, its four waves each a quarter of the chunks.
__global__ __launch_bounds__(kThreads) void tile_sum_kernel(
    const unsigned long long *__restrict__ words, const double *__restrict__ hdr, int chunks,
    int nb1, int nb2, int T, int G, int cells, double *__restrict__ outA,
    double *__restrict__ outB) {
  __shared__ unsigned long long part[2][kThreads];
  const int grid = blockIdx.y / T, tile = blockIdx.y - grid * T;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int cell = blockIdx.x * 64 + lane;
  const unsigned long long *base = words + (int64_t)blockIdx.y * chunks * 2 * cells;
  unsigned long long h = 0, l = 0;
  if (cell < cells) {
    const int c1 = (wave + 1) * chunks / 4;
#pragma unroll 8
    for (int c = wave * chunks / 4; c < c1; ++c) {
      h += base[(int64_t)c * 2 * cells + cell];
      l += base[(int64_t)c * 2 * cells + cells + cell];
    }
  }
  part[0][threadIdx.x] = h;
  part[1][threadIdx.x] = l;
  __syncthreads();
  if (wave || cell >= cells) return;
#pragma unroll
  for (int k = 1; k < 4; ++k) {
    h += part[0][k * 64 + lane];
    l += part[1][k * 64 + lane];
  }
  const int lr = cell / nb2, col = cell - lr * nb2;
  const int row = ((lr / G) * T + tile) * G + lr % G;
  if (row >= nb1) return;
  const FxScale f = fx_stored(hdr + 2 * grid);
  (grid ? outB : outA)[(int64_t)row * nb2 + col] = fx_value((long long)h, (long long)l, f);
}

int grid_for(int64_t n) {
  int64_t b = (n + kThreads - 1) / kThreads;
  if (b < 1) b = 1;
  if (b > 4096) b = 4096;
  return (int)b;
}

int deposit_impl(const char *who, const double *q1, const double *q2, const double *wA,
                 const double *wB, int64_t n, int nb1, double s1, double e1, int nb2, double s2,
                 double e2, double *outA, double *outB, int32_t *cell_index,
                 int32_t *cell_count, void *ws, int64_t ws_bytes, void *stream) {
#pragma clang fp contract(off)
  // particle arrays may be NULL when there are no particles
  if ((n > 0 && (!q1 || !q2)) || !outA || !ws)
    return set_error(DFCSR_EINVAL, "%s: NULL pointer", who);
  if (n < 0 || nb1 < 1 || nb2 < 1) return set_error(DFCSR_EINVAL, "%s: bad sizes", who);
  if (n >= ((int64_t)1 << 31))
    return set_error(DFCSR_ERANGE, "%s: %lld particles >= 2^31", who, (long long)n);
  if ((int64_t)nb1 * nb2 > (int64_t)1 << 28)
    return set_error(DFCSR_ERANGE, "%s: grid %d x %d too large", who, nb1, nb2);
  if (ws_bytes < dfcsr_histogram_workspace_bytes(nb1, nb2))
    return set_error(DFCSR_ENOWS, "%s: workspace too small", who);
  hipStream_t s = as_stream(stream);
  double *hdr = static_cast<double *>(ws);
  const int64_t ncell = (int64_t)nb1 * nb2;
  // bins: inv_spacing = 1 / ((end - start) / nbins), deposit.py:55-58
  const double inv1 = 1.0 / ((e1 - s1) / (double)nb1);
  const double inv2 = 1.0 / ((e2 - s2) / (double)nb2);
  const int nb = nblocks_for(n);
  const int ngrid = outB ? 2 : 1;
  if (cell_count)
    hipLaunchKernelGGL(zero_i32, dim3(grid_for(ncell)), dim3(kThreads), 0, s, cell_count, ncell);
  if ((cell_index || cell_count) && n > 0)
    hipLaunchKernelGGL(cic_cells_kernel, dim3(grid_for(n)), dim3(kThreads), 0, s, q1, q2, n, nb1,
                       s1, inv1, nb2, s2, inv2, cell_index, cell_count);
  const double *wmax = wB ? wB : wA;   // the non-unit weight, if any
  if (wmax) hipLaunchKernelGGL(absmax_partial, dim3(nb), dim3(kThreads), 0, s, wmax, n, hdr + 8);
  const TilePlan t = tile_plan(nb1, nb2);
  if (t.T && !few_on_many(t, ngrid, nb1, n)) {
    int chunks = tile_chunks(t, ngrid, n);
    const int64_t per = n > 0 ? (n + chunks - 1) / chunks : 1;
    auto kernel = t.T > 2 ? cic_tile_kernel<true> : cic_tile_kernel<false>;
    unsigned long long *words = reinterpret_cast<unsigned long long *>(hdr + kHdr);
    hipLaunchKernelGGL(kernel, dim3(chunks, t.T * ngrid), dim3(kTileThreads), t.lds, s, q1, q2, wA,
                       wB, n, per, nb1, s1, inv1, nb2, s2, inv2, t.T, t.G, t.cells, hdr, nb,
                       words);
    hipLaunchKernelGGL(tile_sum_kernel, dim3((t.cells + 63) / 64, t.T * ngrid), dim3(kThreads), 0,
                       s, (const unsigned long long *)words, (const double *)hdr, chunks, nb1,
                       nb2, t.T, t.G, t.cells, outA, outB);
  } else {
    int64_t *acc = reinterpret_cast<int64_t *>(hdr + kHdr);
    hipLaunchKernelGGL(zero_i64, dim3(grid_for(2 * ngrid * ncell)), dim3(kThreads), 0, s, acc,
                       2 * ngrid * ncell);
    hipLaunchKernelGGL(cic_kernel, dim3(grid_for(n), ngrid), dim3(kThreads), 0, s, q1, q2, wA, wB,
                       n, nb1, s1, inv1, nb2, s2, inv2, hdr, nb, acc);
    hipLaunchKernelGGL(fx_to_double, dim3(grid_for(ncell), ngrid), dim3(kThreads), 0, s,
                       (const int64_t *)acc, (const double *)hdr, ncell, outA, outB);
  }
  DFCSR_LAUNCH_CHECK(who);
  return DFCSR_OK;
}

}  // namespace
}  // namespace dfcsr

using namespace dfcsr;

extern "C" int64_t dfcsr_histogram_workspace_bytes(int nbins_1, int nbins_2) {
  if (nbins_1 < 1 || nbins_2 < 1) return 0;
  // the tiles' words of every workgroup (LDS form), or both grids' (direct)
  const TilePlan t = tile_plan(nbins_1, nbins_2);
  int64_t words = 4 * (int64_t)nbins_1 * nbins_2;
  if (t.T) {
    words = 0;
    for (int g = 1; g <= 2; ++g) {
      const int64_t w =
          (int64_t)tile_chunks(t, g, (int64_t)1 << 31) * t.T * g * 2 * (int64_t)t.cells;
      words = w > words ? w : words;
    }
  }
  return ((int64_t)kHdr + words) * 8;
}

extern "C" int dfcsr_histogram_cic_2d(const double *q1, const double *q2, const double *w,
                                      int64_t n, int nbins_1, double bins_start_1,
                                      double bins_end_1, int nbins_2, double bins_start_2,
                                      double bins_end_2, double *hist, int32_t *cell_index,
                                      int32_t *cell_count, void *ws, int64_t ws_bytes,
                                      void *stream) {
  return deposit_impl("histogram_cic_2d", q1, q2, w, nullptr, n, nbins_1, bins_start_1,
                      bins_end_1, nbins_2, bins_start_2, bins_end_2, hist, nullptr, cell_index,
                      cell_count, ws, ws_bytes, stream);
}

extern "C" int dfcsr_deposit_density_vx(const double *x, const double *z, const double *px,
                                        int64_t n, int nbins_x, double x_start, double x_end,
                                        int nbins_z, double z_start, double z_end,
                                        double *density, double *vx, int32_t *cell_index,
                                        int32_t *cell_count, void *ws, int64_t ws_bytes,
                                        void *stream) {
  if ((n > 0 && !px) || !vx) return set_error(DFCSR_EINVAL, "deposit_density_vx: NULL pointer");
  return deposit_impl("deposit_density_vx", x, z, nullptr, px, n, nbins_x, x_start, x_end,
                      nbins_z, z_start, z_end, density, vx, cell_index, cell_count, ws,
                      ws_bytes, stream);
}
