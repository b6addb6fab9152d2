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
