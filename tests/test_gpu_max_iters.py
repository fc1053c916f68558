"""The iteration bound: what GMRES alone solves within it, the default method and the
GMRES behind it solve too, although the default method takes twice as many products."""
import numpy as np
import pytest

from tests.test_gpu_reduced import NETS, WIDE, kept
from paraexastolog_amd import cu_context
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cu_context(0)
    yield c
    c.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("unknowns", [256, 936, 2048, 3944, 32636, 32768])
def test_bound_that_gmres_meets(ctx, unknowns, precision):
    p, dr, n = kept(ctx, *{**NETS, **WIDE}[unknowns], 3)
    x = DeviceArray(ctx, (3, n), np.float64)
    opts = {"precision": precision, "tol": 1e-12, "exact_fallback": 0}
    its = p.solve(3, dr.ptr, x.ptr, restart=32, **opts)["iterations"]
    # half as many more: the two may start from different anchors
    bound = its + its // 2
    p.solve(3, dr.ptr, x.ptr, restart=32, max_iters=bound, **opts)
    rep = p.solve(3, dr.ptr, x.ptr, max_iters=bound, **opts)
    # both methods' iterations, a step of the first being two products
    assert rep["residual"] <= 1e-12 and rep["iterations"] <= 2 * bound + 1
    assert np.abs(x.download().sum(axis=1) - 1.0).max() <= 1e-11
