"""The per-set solver on the parity-reduced system (the default method) against
restarted GMRES with ILU(0) on the full one, which an explicit restart length
asks for: systems of 8 to 3,944 unknowns, so that every workgroup size and the
rows past a workgroup's last full one are met; one set per compute unit and
more; both precisions.  And the same method device-wide on larger systems, for odd
and even batches within and beyond one block's sets, from a warm start too."""
import numpy as np
import pytest

from paraexastolog_amd import cu_context, initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cu_context(0)
    yield c
    c.close()


def kept(ctx, K, N, seed, n_fixed, B):
    net, rng = synth.generate(N, K, seed, n_fixed)
    rates = synth.rate_sets(rng, N, B)
    m = model_builder().parse_model(net.bnet())
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    fixed, vals = net.fixed_spec()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes, fixed, vals).state)
    p = solve_plan(ctx, t, x0.ptr)
    p._keep = (m, t, g, x0)
    return p, DeviceArray.from_host(ctx, rates), 1 << N


# unknowns of the network: (K, N, seed, fixed nodes)
NETS = {8: (2, 10, 1, 0), 60: (2, 10, 2, 0), 256: (2, 12, 0, 0), 296: (2, 9, 0, 0), 696: (0, 10, 2, 5),
        936: (2, 10, 6, 0), 2048: (2, 16, 11, 0), 2908: (0, 12, 1, 5), 3944: (2, 12, 7, 0)}


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("unknowns", sorted(NETS))
@pytest.mark.parametrize("B", [1, 257])
def test_reduced_matches_gmres(ctx, unknowns, B, precision):
    p, dr, n = kept(ctx, *NETS[unknowns], B)
    assert p.info()["unknowns"] == unknowns
    red, ref = DeviceArray(ctx, (B, n), np.float64), DeviceArray(ctx, (B, n), np.float64)
    # both stop at a relative residual of 1e-12; 1e-10 in L1 is what the batch
    # tests allow between solvers at that tolerance
    rep = p.solve(B, dr.ptr, red.ptr, precision=precision, tol=1e-12)
    assert rep["residual"] <= 1e-12
    res, its, meth = p.set_results(B)
    assert (meth >= 0).all()
    p.solve(B, dr.ptr, ref.ptr, precision=precision, tol=1e-12, restart=32)
    x, y = red.download(), ref.download()
    assert np.abs(x - y).sum(axis=1).max() <= 1e-10
    assert np.abs(x.sum(axis=1) - 1.0).max() <= 1e-11
    # a replayed graph and a pinned schedule give the same bits
    p.set_schedule(5)
    for graph in (0, 1, 1):
        red2 = DeviceArray(ctx, (B, n), np.float64)
        p.solve(B, dr.ptr, red2.ptr, precision=precision, tol=1e-12, graph=graph)
        np.testing.assert_array_equal(red2.download(), x)


# terminal segment of 12 states and 12,256 undecided ones (its first cycle breaks down
# for some rate sets); 32,768 terminal states; 32,636 undecided between four attractors
WIDE = {12268: (2, 14, 5, 0), 32768: (0, 15, 0, 5), 32636: (0, 15, 1, 5)}


@pytest.mark.parametrize("unknowns", sorted(WIDE))
@pytest.mark.parametrize("B", [1, 2, 3, 70, 131])
def test_device_wide_reduced_matches_gmres(ctx, unknowns, B):
    p, dr, n = kept(ctx, *WIDE[unknowns], B)
    assert p.info()["unknowns"] == unknowns
    red, ref = DeviceArray(ctx, (B, n), np.float64), DeviceArray(ctx, (B, n), np.float64)
    p.set_schedule(2, 32)  # device-wide GMRES, to 1e-13: at 1e-12 it is itself 1.5e-10 off on one of these
    p.solve(B, dr.ptr, ref.ptr, precision=0, tol=1e-13)
    p.set_schedule(-1)
    y = ref.download()
    for precision in (0, 1):
        rep = p.solve(B, dr.ptr, red.ptr, precision=precision, tol=1e-12)
        assert rep["residual"] <= 1e-12 and rep["exact_solves"] == 0
        x = red.download()
        assert np.abs(x - y).sum(axis=1).max() <= 1e-10
        assert np.abs(x.sum(axis=1) - 1.0).max() <= 1e-11
    # a warm start from the answer converges at once and to the same vectors
    nt = p.info()["n_t"]
    warm = DeviceArray(ctx, (B, nt), np.float64)
    p.gather_terminal(B, red.ptr, warm.ptr)
    rep = p.solve(B, dr.ptr, ref.ptr, precision=0, tol=1e-12, warm=warm.ptr)
    assert np.abs(ref.download() - x).sum(axis=1).max() <= 1e-10
