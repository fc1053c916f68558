"""Sets that the default method leaves: GMRES starts over and solves what it solves where it
is asked for by name, in the precision asked for."""
import numpy as np
import pytest

from paraexastolog_amd import cu_context
from paraexastolog_amd.surrogate import DeviceArray
from tests.test_gpu_reduced import NETS, WIDE, kept

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cu_context(0)
    yield c
    c.close()


# 49,116 states undecided between four attractors, some sets holding their mass so long that a
# residual of 1e-12 is near what rounding leaves: FP32 cycles with FP64 residuals get there
@pytest.mark.parametrize("seed", [2, 5])
def test_absorption_near_the_rounding(ctx, seed):
    p, _, n = kept(ctx, 0, 16, 6, 5, 12)
    assert p.info()["unknowns"] == 49116
    rates = np.exp(np.random.default_rng(seed).uniform(np.log(0.1), np.log(10.0), (12, 32)))
    dr, x, y = DeviceArray.from_host(ctx, rates), DeviceArray(ctx, (12, n), np.float64), DeviceArray(ctx, (12, n), np.float64)
    opts = {"precision": 1, "tol": 1e-12}
    p.solve(12, dr.ptr, y.ptr, restart=32, **opts)
    rep = p.solve(12, dr.ptr, x.ptr, **opts)
    assert rep["residual"] <= 1e-12
    # masses of four attractors that sum to one, each with the error that the conditioning leaves
    # of two solves to that residual: the vectors differ by no more than the methods' tests allow
    assert np.abs(x.download() - y.download()).sum(axis=1).max() <= 1e-10


# the default method stopped where GMRES alone is done, which is before it is done on any set
@pytest.mark.parametrize("unknowns", [296, 32636])
def test_every_set_left(ctx, unknowns):
    B = 5
    p, dr, n = kept(ctx, *{**NETS, **WIDE}[unknowns], B)
    assert p.info()["terminal_segments"] == 0
    x, y = DeviceArray(ctx, (B, n), np.float64), DeviceArray(ctx, (B, n), np.float64)
    opts = {"precision": 0, "tol": 1e-12, "exact_fallback": 0}
    its = p.solve(B, dr.ptr, y.ptr, restart=32, **opts)["iterations"]
    p.solve(B, dr.ptr, x.ptr, max_iters=its, **opts)
    assert (p.set_results(B)[1] > its).all()
    # no anchors to differ: the same iteration, so the same bits
    np.testing.assert_array_equal(x.download(), y.download())
