"""Rate sets on which the default method's shadow vector loses the residual: the cycle ends
there and another one finishes, instead of running out of its 500 products."""
import numpy as np
import pytest

from paraexastolog_amd import cu_context
from paraexastolog_amd.surrogate import DeviceArray
from tests.test_gpu_reduced import kept

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cu_context(0)
    yield c
    c.close()


# per set (1,695 unknowns) and device-wide (11,772): with cycles of 500 products the slowest set takes
# 1,004 and 1,060 on the CPU, with cycles that end 132 and 108
@pytest.mark.parametrize("net,unknowns,seed,B", [((0, 11, 64, 5), 1695, 5128, 40), ((0, 14, 1, 3), 11772, 2571, 257)])
@pytest.mark.parametrize("precision", [0, 1])
def test_slowest_set(ctx, net, unknowns, seed, B, precision):
    p, _, n = kept(ctx, *net, B)
    assert p.info()["unknowns"] == unknowns
    rates = np.exp(np.random.default_rng(seed).uniform(-2.302585, 2.302585, (B, 2 * net[1])))
    if unknowns == 11772:
        rates = np.exp(np.random.default_rng(seed).uniform(-2.3, 2.3, (B, 2 * net[1])))
    dr, x, y = DeviceArray.from_host(ctx, rates), DeviceArray(ctx, (B, n), np.float64), DeviceArray(ctx, (B, n), np.float64)
    rep = p.solve(B, dr.ptr, x.ptr, precision=precision, tol=1e-12)
    assert rep["residual"] <= 1e-12 and rep["exact_solves"] == 0 and rep["fp64_fallback"] == 0
    assert rep["iterations"] < 500  # no cycle ran to its end
    p.solve(B, dr.ptr, y.ptr, precision=0, tol=1e-13, restart=32)
    assert np.abs(x.download() - y.download()).sum(axis=1).max() <= 1e-10  # as the methods' other tests
