"""The per-set solver's kernels for up to one set per compute unit, with several sets:
what a set reads and writes lies at its own place.  And the kernel for the largest
systems, whose rows are those of the larger parity class."""
import numpy as np
import pytest

from paraexastolog_amd import cu_context
from paraexastolog_amd.surrogate import DeviceArray
from paraexastolog_amd import initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from tests.test_gpu_reduced import NETS, kept

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cu_context(0)
    yield c
    c.close()


def compare(p, ctx, dr, B, n, precision):
    red, ref = DeviceArray(ctx, (B, n), np.float64), DeviceArray(ctx, (B, n), np.float64)
    # as in the tests of one set and of 257: 1e-10 in L1 between solvers that stop at 1e-12
    rep = p.solve(B, dr.ptr, red.ptr, precision=precision, tol=1e-12)
    assert rep["residual"] <= 1e-12 and (p.set_results(B)[2] >= 0).all()
    x = red.download()
    p.solve(B, dr.ptr, ref.ptr, precision=precision, tol=1e-12, restart=32)
    assert np.abs(x - ref.download()).sum(axis=1).max() <= 1e-10
    assert np.abs(x.sum(axis=1) - 1.0).max() <= 1e-11
    return x


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("unknowns", [60, 296, 936, 2048, 2908])
@pytest.mark.parametrize("B", [2, 97, 250, 256])
def test_several_sets(ctx, unknowns, B, precision):
    p, dr, n = kept(ctx, *NETS[unknowns], B)
    x = compare(p, ctx, dr, B, n, precision)
    # the sets in another order: the same vectors in that order
    order = np.random.default_rng(B).permutation(B)
    dr2, out = DeviceArray.from_host(ctx, dr.download()[order]), DeviceArray(ctx, (B, n), np.float64)
    p.solve(B, dr2.ptr, out.ptr, precision=precision, tol=1e-12)
    np.testing.assert_array_equal(out.download(), x[order])


def stars(copies):
    """Triples of nodes, each switched on only while all three are off: a triple's states
    are 000 and the three neighbours of it, 1 even and 3 odd ones; 4^copies states, of
    which 2^(copies - 1) more than half have one parity."""
    net = synth.Network(3 * copies)
    for i in range(net.N):
        a = i - i % 3
        net.inputs.append([a, a + 1, a + 2])
        net.tables.append([1 if k == 0 else 0 for k in range(8)])
    return net


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("B", [1, 3, 257])
def test_unbalanced_parities(ctx, B, precision):
    net = stars(6)  # 4,096 unknowns, 2,080 of one parity
    rates = np.exp(np.random.default_rng(7).uniform(np.log(0.1), np.log(10.0), (B, 2 * net.N)))
    m = model_builder().parse_model(net.bnet())
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes).state)
    p = solve_plan(ctx, t, x0.ptr)
    assert p.info()["unknowns"] == 4096
    x = compare(p, ctx, DeviceArray.from_host(ctx, rates), B, 1 << net.N, precision)
    # the triples are independent: products of their stationary vectors, node k on with
    # weight up_k / down_k
    b = B - 1
    q = np.ones(1)
    for a in range(0, net.N, 3):
        w = np.zeros(8)
        w[0] = 1.0
        for k in range(3):
            w[1 << k] = rates[b, 2 * (a + k)] / rates[b, 2 * (a + k) + 1]
        q = np.multiply.outer(w / w.sum(), q).ravel()
    assert np.abs(x[b] - q).sum() <= 1e-10
