"""GPU parity of the forms a kernel takes by size: tile edges, remainders and
the smallest and largest of each form's range, against the oracle."""
import numpy as np
import pytest
import torch

from oracle import cpu_ref as O
from tests.gpu_util import rel_max

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _t(a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to(DEV)


@pytest.fixture(scope="module")
def K():
    from pydfcsr_amd import kernels
    return kernels


@pytest.fixture(scope="module")
def ws():
    from pydfcsr_amd import _lib
    return _lib.Workspace(DEV)


# one LDS tile (the last one cell short of full), two, many (ragged row
# groups of 4, 2 and 1 rows), and grids past the tiles (direct form)
@pytest.mark.parametrize("bins", [(1, 1), (3, 5), (100, 101), (97, 104), (128, 128), (131, 77),
                                  (256, 256), (37, 2411), (13, 4200), (5, 9500), (4, 10300),
                                  (1500, 1300)])
@pytest.mark.parametrize("n", [1, 4097, 40001])
def test_deposit_forms(K, ws, bins, n):
    """Density and vx sums of the LDS tiles and of the direct form: exact
    fixed-point sums against the oracle's float64 ones, within 1e-13 of the
    largest; particles off the grid on every side; repeated bit for bit; a
    weight that is NaN or infinite leaves the other particles' sums exact."""
    rng = np.random.default_rng(n + bins[0])
    x = rng.normal(0.0, 1.0, n)
    z = rng.normal(0.0, 1.0, n) + 0.3 * x
    px = rng.normal(0.0, 1e-3, n) * np.exp(rng.normal(0.0, 3.0, n))
    if n > 100:
        x[:8] = [-9.0, 9.0, 2.5, -2.5, np.nan, 0.0, 1e300, -1e300]
    a = (bins[0], -2.5, 2.5, bins[1], -2.0, 2.25)
    d, v = K.deposit_density_vx(_t(x), _t(z), _t(px), *a, ws)
    ok = np.isfinite(x) & (np.abs(x) < 1e9)
    d0, v0 = (O.histogram_cic_2d(x[ok], z[ok], w[ok], *a) for w in (np.ones(n), px))
    assert rel_max(d.cpu(), d0) <= 1e-13
    assert rel_max(v.cpu(), v0) <= 1e-13
    d, v = d.clone(), v.clone()
    d2, v2 = K.deposit_density_vx(_t(x), _t(z), _t(px), *a, ws)
    assert torch.equal(d, d2) and torch.equal(v, v2)
    h = K.histogram_cic_2d(_t(x), _t(z), _t(px), *a, ws)
    assert torch.equal(h, v)
    if n > 100:
        bad = px.copy()
        bad[50:60] = np.nan
        bad[60:64] = np.inf
        _, v3 = K.deposit_density_vx(_t(x), _t(z), _t(bad), *a, ws)
        bad[50:64] = 0.0
        assert rel_max(v3.cpu(), O.histogram_cic_2d(x[ok], z[ok], bad[ok], *a)) <= 1e-13


# grids of many tiles or rows at either side of the line between few particles
# (direct) and more (tiles)
@pytest.mark.parametrize("bins", [(400, 401), (700, 690), (9000, 5), (41, 4001)])
@pytest.mark.parametrize("n", [1, 10240, 10241])
def test_deposit_few_on_many(K, ws, bins, n):
    """As test_deposit_forms; and the same sums bit for bit with particles off
    the grid beside them, up to a count that takes the tiles (8192 to 16383
    particles share one scale)."""
    test_deposit_forms(K, ws, bins, n)
    n = max(n, 8192)
    rng = np.random.default_rng(n)
    x, z, px = rng.normal(0.0, 1.0, n), rng.normal(0.0, 1.0, n), rng.normal(0.0, 1e-3, n)
    a, off = (bins[0], -2.5, 2.5, bins[1], -2.0, 2.25), 16383 - n
    d, v = (t.clone() for t in K.deposit_density_vx(_t(x), _t(z), _t(px), *a, ws))
    e, w = K.deposit_density_vx(*(_t(np.append(t, np.full(off, c)))
                                  for t, c in ((x, 9.0), (z, 9.0), (px, 0.0))), *a, ws)
    assert torch.equal(d, e) and torch.equal(v, w)


# whole grid in one tile, row tiles, and the direct form; few particles and
# counts either side of a power of two
@pytest.mark.parametrize("bins", [(16, 16), (256, 256), (1500, 1300)])
@pytest.mark.parametrize("n", [200, 4096, 65535, 1 << 20])
def test_deposit_relative(K, ws, bins, n):
    """Each cell's own relative error, for weights of both signs over 2^-42 to 1
    of the largest: every term (w S1) S2 is exact here (30 bits of weight, lower
    corners at multiples of 1/8), so math.fsum of a cell's terms is its sum
    rounded once.  The deposition may be off by two roundings, 2^-52 of the
    value, and by half a quantum a term; the quantum is 2^-k with n max|w| 2^k <
    2^94 or finer."""
    import math
    rng = np.random.default_rng(n + bins[0])
    w = np.ldexp(rng.integers(1 << 29, 1 << 30, n) / 2.0 ** 30, rng.integers(-42, 1, n))
    w *= rng.choice([-1.0, 1.0], n)
    w[0] = 1.0
    i, j = rng.integers(0, bins[0], n), rng.integers(0, bins[1], n)
    i[n // 2:] %= 12   # half of them on few cells, half spread over the grid
    j[n // 2:] %= 12
    a, b = rng.integers(0, 8, n) / 8, rng.integers(0, 8, n) / 8
    got = K.histogram_cic_2d(_t(i + a), _t(j + b), _t(w), bins[0], 0.0, float(bins[0]), bins[1],
                             0.0, float(bins[1]), ws).cpu().numpy()
    terms = {}
    for di in (0, 1):
        for dj in (0, 1):
            t = w * ((1 - a) if di == 0 else a) * ((1 - b) if dj == 0 else b)
            for c, r, v in zip(i + di, j + dj, t):
                if c < bins[0] and r < bins[1]:
                    terms.setdefault((c, r), []).append(v)
    quantum = 2.0 ** -(94 - math.frexp(float(n))[1])
    assert np.count_nonzero(got) <= len(terms)
    for (c, r), v in terms.items():
        ref = math.fsum(v)
        assert abs(got[c, r] - ref) <= 2.0 ** -52 * abs(ref) + len(v) * quantum / 2, (c, r, ref)


@pytest.mark.parametrize("n", [3, 10 ** 6, (1 << 29) + 1, (1 << 30) + 1])
def test_deposit_quantum(K, ws, n):
    """Weights far below the largest, each alone in a cell (the other particles
    lie off the grid): the value to half a quantum of n max|w| 2^k < 2^94, and
    two roundings, at the largest particle counts too."""
    import math
    x = torch.full((n,), -9.0, dtype=torch.float64, device=DEV)
    w = torch.ones(n, dtype=torch.float64, device=DEV)
    small = -(1 + 2.0 ** -20) * 2.0 ** -44
    x[0], x[1], x[2] = 1.0, 3.0, 5.0
    w[1], w[2] = small, -small / 64
    h = K.histogram_cic_2d(x, x, w, 8, 0.0, 8.0, 8, 0.0, 8.0, ws).cpu()
    quantum = 2.0 ** -(94 - math.frexp(float(n))[1])
    for at, ref in ((1, 1.0), (3, small), (5, -small / 64)):
        assert abs(float(h[at, at]) - ref) <= 2.0 ** -52 * abs(ref) + quantum / 2, (at, float(h[at, at]))
    assert np.count_nonzero(h) == 3


# one workgroup's pair tile (2048) less and more one, its last workgroup
# holding one particle, and past one tile and two a workgroup of the full grid
@pytest.mark.parametrize("n", [2, 3, 5, 2047, 2048, 2049, 4097, 524287, 524289, 1048577, 1572865])
@pytest.mark.parametrize("offset", [0, 1])
def test_moments_forms(K, ws, n, offset):
    """Moments and statistics against the oracle's numpy ones: rows on and off
    16 bytes, a tilted bunch.  Both sides sum n float64 terms in trees of some
    20 levels, and x_transform takes 10 sigma_z from x: 1e-12 of the largest
    value summed (1e-11 for sigma_energy and the slope, squares and quotients
    of such sums).  Counts equal, repeated bit for bit, NaN kept."""
    rng = np.random.default_rng(n)
    X = rng.standard_normal((6, n)) * (10.0 ** -np.arange(6))[:, None] + 0.3
    X[4] = rng.normal(2e-5, 1e-3, n)
    X[0] = 10.0 * X[4] + rng.normal(1e-3, 1e-3, n)
    X[5] = rng.normal(2e-3, 1e-3, n)
    coords = torch.empty(6 * n + 1, dtype=torch.float64, device=DEV)[offset:6 * n + offset].view(6, n)
    coords.copy_(_t(X))
    m, ref = K.beam_moments(coords[0], coords[4], ws), O.beam_moments(X[0], X[4])
    big = np.abs(X[0]).max()
    for k in ("mean_x", "mean_z", "sigma_x", "sigma_z", "mean_xt", "sigma_xt", "slice_sigma_x"):
        near = abs(m[k] - ref[k]) <= 1e-12 * max(abs(ref[k]), big)
        assert near or (np.isnan(m[k]) and np.isnan(ref[k])), (k, m[k], ref[k])
    assert np.allclose(m["slope"], ref["slope"], rtol=1e-11, atol=1e-12 * big)
    assert m["n_slice"] == ref["n_slice"]
    m2 = K.beam_moments(coords[0], coords[4], ws)
    assert all(np.array_equal(m2[k], m[k], equal_nan=True) for k in m)
    v = K.beam_statistics(coords, 1e8, 510998.95, ws)
    d, ref = K.statistics_dict(v), O.beam_statistics(*X, 1e8, 510998.95)
    sd = np.abs(X).max(axis=1)
    assert (np.abs(d["mean"] - X.mean(axis=1)) <= 1e-12 * sd).all()
    assert (np.abs(d["cov"] - ref["cov"]) <= 1e-12 * np.outer(sd, sd)).all()
    for k in ("mean_energy", "sigma_energy"):
        assert abs(d[k] - ref[k]) <= 1e-11 * abs(ref[k]), k
    assert torch.equal(v.nan_to_num(), K.beam_statistics(coords, 1e8, 510998.95, ws).nan_to_num())
    coords[0, n - 1] = float("nan")
    m = K.beam_moments(coords[0], coords[4], ws)
    assert np.isnan([m[k] for k in ("mean_x", "sigma_x", "sigma_xt")]).all()
    assert m["sigma_z"] == m2["sigma_z"]


# a grid of one window, one and two tiles (8 x 32 outputs) and one output past
# them, thin grids, windows 1 to 21, more tiles than workgroups (512)
@pytest.mark.parametrize("nx,nz,window,order", [
    (1, 1, 1, 0), (1, 40, 1, 0), (40, 1, 1, 0), (3, 3, 3, 1), (21, 21, 21, 3), (8, 32, 5, 2),
    (9, 33, 7, 2), (100, 100, 5, 3), (13, 300, 13, 2), (300, 15, 15, 3), (256, 256, 9, 2),
    (515, 263, 5, 1), (37, 2049, 21, 4)])
def test_df_forms(K, ws, nx, nz, window, order):
    """Post-processing of a slice (deposit.py:183-235) by tiles against the
    same steps in numpy: each value is a sum of at most 441 products and two
    quotients of float64, so 1e-12 of the field's largest; repeated bit for
    bit."""
    rng = np.random.default_rng(nx * nz + window)
    X = [(-1.3e-3, 1.7e-3, nx), (2e-5, 9e-4, nz)]
    xg, zg = np.linspace(*X[0]), np.linspace(*X[1])
    x, z = np.linspace(-3, 3, nx)[:, None], np.linspace(-3, 3, nz)[None, :]
    dens = 1e4 * np.exp(-0.5 * ((x - z) ** 2 + z ** 2)) * (1 + 0.1 * rng.random((nx, nz)))
    vx = dens * (0.3 * x + 0.1 * z + 0.01 * rng.random((nx, nz)))
    vt = 40.0
    d, v = _t(dens), _t(vx)
    out, info = [torch.empty_like(d) for _ in range(3)], torch.zeros(4, dtype=torch.float64, device=DEV)
    a = (*X[0][:2], *X[1][:2], vt, window, order, ws)
    K.df_process(d, v, *a, out=out, info=info)
    thr = dens.max() / vt
    r = {"vx": np.where(dens > thr, vx / dens, vx)}
    r["density"], r["vx"] = O._sg2(dens, window, order), O._sg2(r["vx"], window, order)
    with np.errstate(invalid="ignore", divide="ignore"):
        dsum = O._trapz(O._trapz(r["density"], xg, axis=0), zg)
        r["density"] = r["density"] / dsum
        r["vx"][r["density"] <= thr] = 0
        grad = [np.gradient(f, g, axis=k) if g.size > 1 else np.zeros_like(f)
                for f, g, k in ((r["density"], xg, 0), (r["density"], zg, 1), (r["vx"], xg, 0))]
    for k, g in zip(("density_x", "density_z", "vx_x"), grad):
        r[k] = O._sg2(g, window, order)
    got = dict(density=d, vx=v, density_x=out[0], density_z=out[1], vx_x=out[2])
    if min(nx, nz) > 1:
        top = r["density"].max()
        fill = r["vx_x"][r["density"] > top / vt * 8].mean()
        r["vx_x"][r["density"] < top / vt * 8] = fill
        assert np.allclose(info.cpu(), [dens.max(), dsum, top, fill], rtol=1e-12, atol=0)
        for k, g in got.items():
            assert rel_max(g.cpu(), r[k]) <= 1e-12, k
    else:
        assert info[1] == 0.0 and not np.isfinite(d.cpu()).any()   # no area: density / 0
    d2, v2, out2 = _t(dens), _t(vx), [torch.empty_like(d) for _ in range(3)]
    K.df_process(d2, v2, *a, out=out2)
    for g, h in zip([d, v, *out], [d2, v2, *out2]):
        assert np.array_equal(g.cpu().numpy(), h.cpu().numpy(), equal_nan=True)


@pytest.mark.parametrize("jobs", [16, 17, 64, 65, 131])
def test_regrid_many_jobs(K, ws, jobs):
    """Slices re-gridded in one call, whose jobs go 16 or 64 a launch, against
    the same slices in calls of one: every ring bit for bit."""
    rng = np.random.default_rng(jobs)
    nb, Xi, Zi, cap = (7, 9), 11, 35, jobs + 2
    src = _t(rng.normal(0.0, 1.0, (jobs, 5, *nb)))
    J = [(j, (3 * j) % cap if cap % 3 else j, *nb, -1.0 - 0.01 * j, 1.2, -1.0, 1.0 + 0.02 * j)
         for j in range(jobs)]

    def rings(calls):
        f64, f32 = (dict(dtype=d, device=DEV) for d in (torch.float64, torch.float32))
        h64, h32t = torch.zeros((Xi, Zi, cap, 20), **f64), torch.zeros((Xi, Zi, cap, 20), **f32)
        h32 = torch.zeros((Xi, cap, 5, Zi, 4), **f32)
        c, c32 = torch.zeros((cap, Xi, Zi + 1, 5), **f64), torch.zeros((cap, Xi, Zi + 1, 5), **f32)
        for k in calls:
            K.regrid(src, 5 * nb[0] * nb[1], k, h64, h32, Xi, Zi, -1.1, 1.1, -1.05, 1.5, ws, h32t,
                     c, c32)
        return h64, h32, h32t, c, c32

    for a, b in zip(rings([J]), rings([[j] for j in J])):
        assert a.any() and torch.equal(a, b)


def test_grids_of_many_launches(K, ws):
    """An interp grid of more tiles (re-grid) and rows (span table) than one
    launch's threads can hold: a slice of two by two points, whose fields are
    bilinear, on 140 million x rows, within three float32 roundings; spans of
    rows at either end, and none between."""
    from pydfcsr_amd import _lib
    lib, Xi, Zi = _lib.load(), 140_000_000, 2
    f = np.random.default_rng(0).normal(0.0, 1.0, (5, 2, 2))
    cells = torch.zeros((1, Xi, Zi + 1, 5), dtype=torch.float32, device=DEV)
    K.regrid(_t(f), 20, [(0, 0, 2, 2, -1.0, 1.0, -1.0, 1.0)], None, None, Xi, Zi, -1.0, 1.0, -1.0,
             1.0, ws, cells32=cells)
    for a in (0, 5_000_001, 5_782_280, 69_999_999, 134_217_728, Xi - 9):   # nine rows from a
        y = (np.arange(a, a + 9) / (Xi - 1))[:, None]
        for z in range(3):
            ref = (1 - y) * f[:, 0, min(z, 1)] + y * f[:, 1, min(z, 1)]
            got = cells[0, a:a + 9, z].cpu().numpy()
            assert np.abs(got - ref).max() <= 3 * 2.0 ** -24 * np.abs(f).max(), (a, z)
    Xi = 20_000_000
    cells = cells.view(-1)[:Xi * 15].view(1, Xi, 3, 5).zero_()
    hot = [0, 7, 3_222_784, 16_777_215, Xi - 1]
    for k, x in enumerate(hot):
        cells[0, x, k % 2, 0] = 1.0
    span = torch.full((Xi, 1), 7, dtype=torch.int32, device=DEV)
    _lib.check(lib.dfcsr_history_zspan(None, cells.data_ptr(), span.data_ptr(), Xi, Zi, 1, 0, 1, 0,
                                       torch.cuda.current_stream().cuda_stream), "zspan")
    ref = torch.full((Xi, 1), 0xFFFF, dtype=torch.int32, device=DEV)
    for k, x in enumerate(hot):   # an entry joins rows x and x + 1
        ref[max(x - 1, 0):x + 1] = (k % 2) | (k % 2) << 16
    assert torch.equal(span, ref)


# the smallest mesh, one that is no mesh, odd ones, the largest two wakes and
# the largest one wake that fit the LDS whole, and meshes of which the middle is
# held: one row too many, thin ones
@pytest.mark.parametrize("nx,nz,two", [(2, 2, 1), (1, 5, 1), (31, 33, 1), (103, 99, 1),
                                       (142, 144, 0), (103, 100, 1), (256, 300, 1), (2, 9000, 1),
                                       (30000, 2, 0)])
def test_kick_forms(K, nx, nz, two):
    """The kick with the wakes in LDS (1.25e6 particles or more, 4e6 for dE
    alone) against the same particles in smaller calls, bit for bit, and against
    scipy's interpolator within 1e-12 of the largest kick (four products and
    their sum); particles on and off the mesh's edges, NaN positions."""
    from scipy.interpolate import RegularGridInterpolator
    n, few = 1250000 if two else 4000001, 500000
    rng = np.random.default_rng(nx)
    x, z = rng.normal(0, 1e-4, n), rng.normal(1e-5, 5e-5, n)
    xr, zr, slope = (-2e-4, 2.5e-4), (-1e-4, 1.1e-4), (0.7, 1e-6)
    x[:4] = np.array([*xr, *xr]) + slope[0] * np.array([*zr, 0, 0]) + slope[1]
    z[:4] = [*zr, 0, 0]
    x[4:6], z[6:8] = np.nan, [np.nan, np.inf]
    px, pz = rng.normal(0, 1e-6, n), rng.normal(0, 1e-6, n)
    w = [rng.normal(0, 1e3, (nx, nz)) for _ in range(2)]
    d = [_t(w[0]), _t(w[1]) if two else None]
    whole, parts = [_t(px), _t(pz)], [_t(px), _t(pz)]
    X, Z, a = _t(x), _t(z), (*xr, *zr, *slope, 0.013, 2e9, two, nx, nz)
    K.apply_wakes(*whole, X, Z, *d, *a)
    for k in range(0, n, few):
        K.apply_wakes(*(v[k:k + few] for v in parts), X[k:k + few], Z[k:k + few], *d, *a)
    for u, v in zip(whole, parts):
        assert torch.equal(u, v)
    xt = x[:few] - (slope[0] * z[:few] + slope[1])
    for u, v, k in ((whole[1], pz, 0), (whole[0], px, 1)):
        got = u[:few].cpu().numpy() - v[:few]
        if min(nx, nz) < 2 or (k and not two):
            assert (got == 0).all()
            continue
        f = RegularGridInterpolator((np.linspace(*xr, nx), np.linspace(*zr, nz)),
                                    0.013 * w[k] * 1e6 / 2e9, fill_value=0.0, bounds_error=False)
        ok = np.isfinite(x[:few] + z[:few])
        ref = f(np.array([xt[ok], z[:few][ok]]).T)
        # the kick is what is left of px + kick - px: an ulp of px beside it
        assert np.abs(got[ok] - ref).max() <= 1e-12 * np.abs(ref).max() + 2e-21
        assert (got[~ok] == 0).all()


# meshes whose middle would be less than one cell wide if its sides were only in
# proportion, and meshes without a cell
@pytest.mark.parametrize("nx,nz,two", [(30000, 2, 1), (2, 9000, 1), (3, 50000, 1), (50000, 2, 0),
                                       (2, 30000, 0), (12000, 1, 1), (25000, 1, 0), (1, 12000, 1)])
def test_kick_thin_meshes(K, nx, nz, two):
    """As test_kick_forms: few particles a call and many, and scipy's."""
    test_kick_forms(K, nx, nz, two)


# the largest meshes of which the middle is held, and the next
@pytest.mark.parametrize("nx,nz,two", [(1024, 640, 1), (1024, 641, 1), (2048, 640, 0),
                                       (2048, 641, 0)])
def test_kick_large_meshes(K, nx, nz, two):
    """As test_kick_forms."""
    test_kick_forms(K, nx, nz, two)


LAT_ELEMENTS = [dict(type="drift", L=0.1, nsep=1), dict(type="dipole", L=0.3, angle=0.05, nsep=1),
                dict(type="drift", L=0.4, nsep=2), dict(type="dipole", L=0.3, angle=-0.05, nsep=1)]


class _History:
    """A smooth synthetic history (nt slices on Xi x Zi) with the attributes
    DeviceHistory and the oracle's C integral read."""

    def __init__(self, t, sx, sz, nt=9, Xi=37, Zi=700):
        x, z = np.linspace(-5, 5, Xi), np.linspace(-5, 5, Zi)
        k = np.arange(nt)[:, None, None]
        g = np.exp(-0.5 * (x[None, :, None] ** 2 + z[None, None, :] ** 2))
        g = np.where(g > 1e-4, g, 0.0) * (1 + 0.1 * np.sin(k + z[None, None, :]))
        one = np.ones_like(g)
        self.data = dict(density=g / (sx * sz), density_x=-x[None, :, None] * g / sx ** 2 / sz,
                         density_z=-z[None, None, :] * g / sz ** 2 / sx,
                         vx=(1e-3 * x[None, :, None] + 1e-4 * k) * one,
                         vx_x=1e-3 / sx * one * (1 + 0.05 * z[None, None, :]))
        self._axes = dict(min_t=t - 0.03 * (nt - 1), min_x=-5 * sx, min_z=-5 * sz, dt=0.03,
                          dx=10 * sx / (Xi - 1), dz=10 * sz / (Zi - 1))

    def axes(self):
        return self._axes


# mesh bins about a quarter, half and whole wave and several observer blocks;
# odd rows and columns; sigma_x / sigma_z thin, round and wide (windows of a
# few z cells, of the whole grid, and tiled); the mesh past the lattice's end
@pytest.mark.parametrize("mesh,nxz,sx,sz,t", [
    ((17, 3), (13, 9), 20e-6, 80e-6, 0.33), ((32, 4), (24, 31), 50e-6, 50e-6, 0.33),
    ((33, 3), (21, 40), 300e-6, 30e-6, 0.33), ((64, 2), (40, 33), 20e-6, 80e-6, 0.5),
    ((65, 2), (9, 17), 50e-6, 50e-6, 0.33), ((129, 2), (16, 16), 300e-6, 30e-6, 0.5),
    ((300, 1), (11, 12), 50e-6, 50e-6, 0.33), ((20, 5), (10, 300), 20e-6, 80e-6, 0.33),
    ((24, 6), (12, 15), 50e-6, 50e-6, 1.1)])
def test_wake_line_form(K, ws, mesh, nxz, sx, sz, t):
    """The wake by z lines (cell-major rings, |slope| <= 1) against the same
    wake by phases (explicit observers) and the oracle's C integral, float64
    within 1e-10 of max|W| and mixed within 1e-8 of the phases' (the same
    float32 operations, float64 sums in another order); batched bit for bit;
    the span table changes no bit and evaluates no more points."""
    from oracle import csr_ref_c as C
    from pydfcsr_amd import _lib
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    beam = dict(sigma_x=sx, sigma_z=sz, slope=np.array([0.3, 1e-6]), mean_x=0.0)
    xa, za = (-5 * sx, 5 * sx, mesh[0]), (-5 * sz, 5 * sz, mesh[1])
    L = DeviceLattice(lat, DEV)
    args = (t, beam, 0.05, 4.0, *nxz, 9.0, xa, za)
    P = wake_params(*args)
    rings = ("fp64", "fp32t", "cells", "cells32")
    H = DeviceHistory(T, DEV, wrap=2, rings=rings)
    Hz = DeviceHistory(T, DEV, wrap=2, rings=rings + ("zspan",))
    M = mesh[0] * mesh[1]
    out = {p: {k: v.cpu().numpy() for k, v in K.wake_mesh(H.desc, L.desc, P, p, DEV, ws).items()}
           for p in (0, 1)}
    obs_np = np.stack([out[0]["zmesh"], out[0]["xmesh"]], axis=1)
    obs = _t(obs_np)
    Po = wake_params(*args[:-2], (0.0, 0.0, 1), (0.0, 0.0, M), observers=obs)
    keep = C._Keep()
    ref = C.wake(C.hist_from_tracker(T, keep), C.lat_from_tables(lat, keep), t, beam, 0.05, 4.0,
                 *nxz, 9.0, obs_np)
    for p, tol, oracle in ((0, 1e-10, 1e-10), (1, 1e-8, 1e-4)):
        ph = K.wake_mesh(H.desc, L.desc, Po, p, DEV, ws)
        for k, r in zip(("dE_dct", "x_kick"), ref):
            a, b = out[p][k], ph[k].cpu().numpy()
            assert np.array_equal(np.isnan(a), np.isnan(b)), (p, k)
            assert np.array_equal(np.isnan(a), np.isnan(r)), (p, k)
            ok = np.isfinite(r)
            assert ok.any() and np.abs(r[ok]).max() > 0
            # observers whose sources all lie on one straight (t = 0.5) have
            # no x kick: what each form holds there is rounding of terms as
            # large as dE_dct's (the oracle's own is 1e-13 to 1e-12 of it)
            straight = k == "x_kick" and np.nanmax(np.abs(r)) < 1e-9 * np.nanmax(np.abs(ref[0]))
            scale = np.nanmax(np.abs(ref[0])) / np.nanmax(np.abs(r)) if straight else 1.0
            assert rel_max(a[ok], b[ok]) <= tol * scale, (p, k)
            assert rel_max(a[ok], r[ok]) <= oracle * scale, (p, k)
        z = K.wake_mesh(Hz.desc, L.desc, P, p, DEV, ws)
        o = [{k: torch.empty(M, dtype=torch.float64, device=DEV) for k in ("dE_dct", "x_kick")}
             for _ in range(2)]
        K.wake_mesh_batched([H.desc, Hz.desc], [L.desc] * 2, [P] * 2, p, o, DEV, ws)
        for k in ("dE_dct", "x_kick"):
            for v in (z[k], o[0][k], o[1][k]):
                assert np.array_equal(out[p][k], v.cpu().numpy(), equal_nan=True), (p, k)
        n = [K.wake_points_evaluated(h.desc, L.desc, P, p, DEV, ws) for h in (H, Hz)]
        assert 0 < n[1] <= n[0]


# the same edges with z lines and rows enough that the line form is taken: one
# and two observers past a quarter, half and whole wave, several blocks, an odd
# last pass of rows, tiled windows, columns past 256, the mesh past the lattice
@pytest.mark.parametrize("mesh,nxz,sx,sz,t", [
    ((17, 46), (13, 9), 20e-6, 80e-6, 0.33), ((32, 24), (24, 31), 50e-6, 50e-6, 0.33),
    ((33, 34), (22, 40), 300e-6, 30e-6, 0.33), ((64, 10), (41, 33), 20e-6, 80e-6, 0.5),
    ((65, 76), (9, 17), 50e-6, 50e-6, 0.33), ((129, 48), (16, 16), 300e-6, 30e-6, 0.5),
    ((300, 28), (11, 12), 50e-6, 50e-6, 0.33), ((20, 52), (10, 300), 20e-6, 80e-6, 0.33),
    ((35, 9), (79, 257), 20e-6, 80e-6, 0.33), ((34, 61), (12, 15), 50e-6, 50e-6, 1.1)])
def test_wake_line_form_taken(K, ws, mesh, nxz, sx, sz, t):
    """The wake by z lines on meshes that the rule of sizes gives to them (in
    mixed precision from 33 x bins on) against the same wake by phases (explicit
    observers), float64 within 1e-10 of max|W| and mixed within 1e-8; the oracle's
    C integral within 1e-10 (mixed 1e-4) of max|dE_dct|, the size of the terms
    that x_kick's sums cancel; batched bit for bit; the span table changes no bit
    and evaluates no more points."""
    from oracle import csr_ref_c as C
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    from tests.test_abi import _forms
    assert _forms(*mesh, *nxz, 0) == (4 if mesh[0] < 33 else 2)
    assert _forms(*mesh, *nxz, 1) == (1 if mesh[0] < 33 else 2)
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    beam = dict(sigma_x=sx, sigma_z=sz, slope=np.array([0.3, 1e-6]), mean_x=0.0)
    xa, za = (-5 * sx, 5 * sx, mesh[0]), (-5 * sz, 5 * sz, mesh[1])
    L, args, M = DeviceLattice(lat, DEV), (t, beam, 0.05, 4.0, *nxz, 9.0), mesh[0] * mesh[1]
    P = wake_params(*args, xa, za)
    rings = ("fp64", "fp32t", "cells", "cells32")
    H, Hz = (DeviceHistory(T, DEV, wrap=2, rings=r) for r in (rings, rings + ("zspan",)))
    keep, ref = C._Keep(), None
    for p, tol, oracle in ((0, 1e-10, 1e-10), (1, 1e-8, 1e-4)):
        line = K.wake_mesh(H.desc, L.desc, P, p, DEV, ws)
        obs = torch.stack([line["zmesh"].flatten(), line["xmesh"].flatten()], dim=1).contiguous()
        Po = wake_params(*args, (0.0, 0.0, 1), (0.0, 0.0, M), observers=obs)
        ph = K.wake_mesh(H.desc, L.desc, Po, p, DEV, ws)
        if ref is None:
            ref = C.wake(C.hist_from_tracker(T, keep), C.lat_from_tables(lat, keep), t, beam, 0.05,
                         4.0, *nxz, 9.0, obs.cpu().numpy())
        top = np.nanmax(np.abs(ref[0]))
        for k, r in zip(("dE_dct", "x_kick"), ref):
            a, b = line[k].cpu().numpy().ravel(), ph[k].cpu().numpy().ravel()
            assert np.array_equal(np.isnan(a), np.isnan(b)), (p, k)
            assert np.array_equal(np.isnan(a), np.isnan(r)), (p, k)
            ok = np.isfinite(r)
            assert ok.any() and np.abs(r[ok]).max() > 0
            straight = k == "x_kick" and np.abs(r[ok]).max() < 1e-9 * top
            assert np.abs(a - b)[ok].max() <= tol * (top if straight else np.abs(r[ok]).max()), (p, k)
            assert np.abs(a - r)[ok].max() <= oracle * top, (p, k)
        z = K.wake_mesh(Hz.desc, L.desc, P, p, DEV, ws)
        o = [{k: torch.empty(M, dtype=torch.float64, device=DEV) for k in ("dE_dct", "x_kick")}
             for _ in range(2)]
        K.wake_mesh_batched([H.desc, Hz.desc], [L.desc] * 2, [P] * 2, p, o, DEV, ws)
        for k in ("dE_dct", "x_kick"):
            for v in (z[k], o[0][k], o[1][k]):
                assert np.array_equal(line[k].cpu().numpy().ravel(), v.cpu().numpy().ravel(),
                                      equal_nan=True), (p, k)
        n = [K.wake_points_evaluated(h.desc, L.desc, P, p, DEV, ws) for h in (H, Hz)]
        assert 0 < n[1] <= n[0]


# s' columns in one to five groups of 64, dealt a wave each, shared by two or
# four waves, or each to all waves; the chirp branch (four regions) and not
@pytest.mark.parametrize("nz", [5, 64, 65, 128, 150, 200, 256, 257])
@pytest.mark.parametrize("slope", [0.3, -1.7])
def test_wake_phase_groups(K, ws, nz, slope):
    """The wake by phases (a mesh of 5 x bins) against the oracle's C integral,
    as test_wake_line_form's, and batched bit for bit."""
    from oracle import csr_ref_c as C
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    sx, sz, t = 50e-6, 50e-6, 0.33
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    beam = dict(sigma_x=sx, sigma_z=sz, slope=np.array([slope, 1e-6]), mean_x=0.0)
    args = (t, beam, 0.05, 4.0, 70, nz, 9.0, (-sx, sx, 5), (-sz, sz, 3))
    H = DeviceHistory(T, DEV, wrap=2, rings=("fp64", "fp32t", "cells", "cells32", "zspan"))
    L, P = DeviceLattice(lat, DEV), wake_params(*args)
    keep, ref = C._Keep(), None
    for p, tol in ((0, 1e-10), (1, 1e-4)):
        out = K.wake_mesh(H.desc, L.desc, P, p, DEV, ws)
        if ref is None:
            obs = np.stack([out["zmesh"].cpu().numpy(), out["xmesh"].cpu().numpy()], axis=1)
            ref = C.wake(C.hist_from_tracker(T, keep), C.lat_from_tables(lat, keep), t, beam, 0.05,
                         4.0, 70, nz, 9.0, obs)
        o = [{k: torch.empty_like(out["dE_dct"]) for k in ("dE_dct", "x_kick")} for _ in range(2)]
        K.wake_mesh_batched([H.desc] * 2, [L.desc] * 2, [P] * 2, p, o, DEV, ws)
        for k, r in zip(("dE_dct", "x_kick"), ref):
            a, ok = out[k].cpu().numpy(), np.isfinite(r)
            assert np.array_equal(np.isnan(a), np.isnan(r)) and ok.any()
            assert rel_max(a[ok], r[ok]) <= tol, (p, k)
            for v in o:
                assert np.array_equal(a, v[k].cpu().numpy(), equal_nan=True), (p, k)


@pytest.mark.parametrize("forms", [0, -1, 8])
def test_wake_batch_forms_unset(K, ws, forms):
    """A batch shape that tells no valid form launches them all: tasks of every
    form (5, 20 and 33 x bins) equal the single launches bit for bit."""
    import ctypes
    from pydfcsr_amd import _lib
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    sx, sz, t = 50e-6, 50e-6, 0.33
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    beam = dict(sigma_x=sx, sigma_z=sz, slope=np.array([0.3, 1e-6]), mean_x=0.0)
    H = DeviceHistory(T, DEV, wrap=2, rings=("fp64", "fp32t", "cells", "cells32", "zspan"))
    L, lib = DeviceLattice(lat, DEV), _lib.load()
    Ps = [wake_params(t, beam, 0.05, 4.0, 70, 65, 9.0, (-sx, sx, m), (-sz, sz, 3))
          for m in (5, 20, 33)]
    k = len(Ps)
    for p in (0, 1):
        one = [K.wake_mesh(H.desc, L.desc, P, p, DEV, ws) for P in Ps]
        o = [{n: torch.full_like(w[n], 7.0) for n in ("dE_dct", "x_kick")} for w in one]
        host = torch.empty(lib.dfcsr_wake_task_table_bytes(k), dtype=torch.uint8)
        batch = _lib.WakeBatch()
        _lib.check(lib.dfcsr_wake_tasks_pack(
            k, (_lib.History * k)(*[H.desc] * k), (_lib.Lattice * k)(*[L.desc] * k),
            (_lib.WakeParams * k)(*Ps), p, (_lib.c_dp * k)(*[v["dE_dct"].data_ptr() for v in o]),
            (_lib.c_dp * k)(*[v["x_kick"].data_ptr() for v in o]), host.data_ptr(), host.numel(),
            ctypes.byref(batch)), "pack")
        batch.forms = forms
        dev = host.to(DEV)
        part = torch.empty(int(batch.partial_bytes), dtype=torch.uint8, device=DEV)
        _lib.check(lib.dfcsr_wake_batched_launch(
            dev.data_ptr(), ctypes.byref(batch), p, part.data_ptr(), part.numel(),
            torch.cuda.current_stream().cuda_stream), "launch")
        for w, v in zip(one, o):
            for n in v:
                assert np.array_equal(w[n].cpu().numpy(), v[n].cpu().numpy(), equal_nan=True), (p, n)


@pytest.mark.parametrize("forms", [0, -1, 8])
def test_wake_batch_all_forms_unset(K, ws, forms):
    """As test_wake_batch_forms_unset, with z lines enough for every form."""
    import ctypes
    from pydfcsr_amd import _lib
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    sx, sz, t = 50e-6, 50e-6, 0.33
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    beam = dict(sigma_x=sx, sigma_z=sz, slope=np.array([0.3, 1e-6]), mean_x=0.0)
    H = DeviceHistory(T, DEV, wrap=2, rings=("fp64", "fp32t", "cells", "cells32", "zspan"))
    L, lib = DeviceLattice(lat, DEV), _lib.load()
    Ps = [wake_params(t, beam, 0.05, 4.0, 70, 65, 9.0, (-sx, sx, m), (-sz, sz, 16))
          for m in (5, 20, 33)]
    k = len(Ps)
    for p in (0, 1):
        one = [K.wake_mesh(H.desc, L.desc, P, p, DEV, ws) for P in Ps]
        o = [{n: torch.full_like(w[n], 7.0) for n in ("dE_dct", "x_kick")} for w in one]
        host = torch.empty(lib.dfcsr_wake_task_table_bytes(k), dtype=torch.uint8)
        batch = _lib.WakeBatch()
        _lib.check(lib.dfcsr_wake_tasks_pack(
            k, (_lib.History * k)(*[H.desc] * k), (_lib.Lattice * k)(*[L.desc] * k),
            (_lib.WakeParams * k)(*Ps), p, (_lib.c_dp * k)(*[v["dE_dct"].data_ptr() for v in o]),
            (_lib.c_dp * k)(*[v["x_kick"].data_ptr() for v in o]), host.data_ptr(), host.numel(),
            ctypes.byref(batch)), "pack")
        batch.forms = forms
        dev = host.to(DEV)
        part = torch.empty(int(batch.partial_bytes), dtype=torch.uint8, device=DEV)
        _lib.check(lib.dfcsr_wake_batched_launch(
            dev.data_ptr(), ctypes.byref(batch), p, part.data_ptr(), part.numel(),
            torch.cuda.current_stream().cuda_stream), "launch")
        for w, v in zip(one, o):
            for n in v:
                assert np.array_equal(w[n].cpu().numpy(), v[n].cpu().numpy(), equal_nan=True), (p, n)


def test_wake_batch_of_many_launches(K, ws):
    """A batch whose region 0 takes more workgroups than a launch holds (4096
    tasks of 17 x 17 points, 1500 columns by z lines, a chirp-branch task among
    them): each task equals its single launch bit for bit."""
    from pydfcsr_amd import _lib
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    sx, sz, t, k = 50e-6, 50e-6, 0.33, 4096
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    H = DeviceHistory(T, DEV, wrap=2, rings=("fp64", "cells", "zspan"))
    L = DeviceLattice(lat, DEV)
    P = [wake_params(t, dict(sigma_x=sx, sigma_z=sz, slope=np.array([s, 1e-6]), mean_x=0.0), 0.05,
                     4.0, 48, 1500, 9.0, (-sx, sx, 17), (-sz, sz, 17)) for s in (0.3, -0.4, -1.7)]
    one = [K.wake_mesh(H.desc, L.desc, p, 0, DEV, ws) for p in P]
    which = [2 if j == 2000 else j % 2 for j in range(k)]
    out = {n: torch.full((k, 17 * 17), 7.0, dtype=torch.float64, device=DEV)
           for n in ("dE_dct", "x_kick")}
    o = [{n: v[j] for n, v in out.items()} for j in range(k)]
    # (its 29 GB go with this workspace)
    K.wake_mesh_batched([H.desc] * k, [L.desc] * k, [P[w] for w in which], 0, o, DEV,
                        _lib.Workspace(DEV))
    for n in out:
        ref = torch.stack([w[n].flatten() for w in one])[torch.tensor(which, device=DEV)]
        assert torch.isfinite(ref).any()
        assert torch.equal(out[n].nan_to_num(nan=1e300), ref.nan_to_num(nan=1e300)), n


@pytest.mark.parametrize("precision,tol", [(0, 1e-10), (1, 1e-8)])
def test_wake_of_many_launches(K, ws, precision, tol):
    """A mesh whose near regions by phases take more workgroups than a launch
    holds (1200 x 1200 points, the chirp branch, 12 phases) against the same
    points as explicit observers in small calls, float64 within 1e-10 of max|W|
    and mixed within 1e-8 (the same float32 operations, float64 sums in another
    order)."""
    from pydfcsr_amd import _lib
    from tests.gpu_util import DeviceHistory, DeviceLattice, wake_params
    sx, sz, t, m, own = 50e-6, 50e-6, 0.33, 1200, _lib.Workspace(DEV)
    T, lat = _History(t, sx, sz), O.LatticeTables(LAT_ELEMENTS)
    beam = dict(sigma_x=sx, sigma_z=sz, slope=np.array([-1.7, 1e-6]), mean_x=0.0)
    H = DeviceHistory(T, DEV, wrap=2, rings=("fp64", "fp32t", "cells", "cells32", "zspan"))
    L, args = DeviceLattice(lat, DEV), (t, beam, 0.05, 4.0, 200, 3, 9.0)
    P = wake_params(*args, (-sx, sx, m), (-sz, sz, m))
    got = {k: v.flatten() for k, v in K.wake_mesh(H.desc, L.desc, P, precision, DEV, own).items()}
    obs = torch.stack([got["zmesh"], got["xmesh"]], dim=1)
    ref = {k: torch.empty_like(got[k]) for k in ("dE_dct", "x_kick")}
    for a in range(0, m * m, m * m // 16):
        o = obs[a:a + m * m // 16].contiguous()
        Po = wake_params(*args, (0.0, 0.0, 1), (0.0, 0.0, len(o)), observers=o)
        for k, v in K.wake_mesh(H.desc, L.desc, Po, precision, DEV, ws).items():
            if k in ref:
                ref[k][a:a + len(o)] = v.flatten()
    for k, r in ref.items():
        ok = torch.isfinite(r)
        assert torch.equal(ok, torch.isfinite(got[k])) and ok.any()
        assert (got[k] - r)[ok].abs().max() <= tol * r[ok].abs().max(), k
