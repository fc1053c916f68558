"""A captured solve holds the addresses of its plan's buffers: a call between two replays
that makes the plan allocate one of them anew, with sets that are finished by GMRES,
must not leave the old address in use."""
import numpy as np
import pytest

from paraexastolog_amd import initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from paraexastolog_amd._lib import EslError
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("many", [False, True])
def test_basis_grown_between_replays(ctx, many):
    net, rng = synth.generate(10, 2, 6, 0)
    B, n = 5, 1 << net.N
    rates = synth.rate_sets(rng, net.N, B)
    m = model_builder().parse_model(net.bnet())
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes, *net.fixed_spec()).state)
    p = solve_plan(ctx, t, x0.ptr)
    dr, out = DeviceArray.from_host(ctx, rates), DeviceArray(ctx, (B, n), np.float64)

    def gmres(**opts):
        opts = {"precision": 0, "tol": 1e-12, "restart": 16, "preconditioner": 2, **opts}
        if many:
            solve_plan.solve_many(ctx, [p], [B], [dr.ptr], [out.ptr], **opts)
        else:
            p.solve(B, dr.ptr, out.ptr, **opts)
        return out.download()

    want = gmres(graph=0)
    np.testing.assert_array_equal(gmres(graph=1), want)  # 17 basis vectors a set
    # the default method, stopped after two products: GMRES takes over with 33
    with pytest.raises(EslError):
        if many:
            solve_plan.solve_many(ctx, [p], [B], [dr.ptr], [out.ptr], precision=0, tol=1e-12, max_iters=2,
                                  exact_fallback=0)
        else:
            p.solve(B, dr.ptr, out.ptr, precision=0, tol=1e-12, max_iters=2, exact_fallback=0)
    # takes what the smaller basis has left, where it is kept for reuse, and fills it
    other = [DeviceArray(ctx, (B, n), np.float64) for _ in range(3)]
    q = solve_plan(ctx, t, x0.ptr)
    for o in other:
        q.solve(B, dr.ptr, o.ptr, precision=0, tol=1e-12, restart=16)
    for _ in range(3):
        np.testing.assert_array_equal(gmres(graph=1), want)
        q.solve(B, dr.ptr, other[0].ptr, precision=0, tol=1e-12, restart=16)
        np.testing.assert_array_equal(other[0].download(), want)
