"""What device-wide solves keep between calls: a plan its own three vectors, the context
at most the bound of its pool, and nothing of it once an allocation has failed."""
import ctypes

import numpy as np
import pytest

from paraexastolog_amd import cu_context, initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from paraexastolog_amd._lib import EslError, check, lib
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu

N, B, UNKNOWNS = 15, 1024, 32768
VECTOR = 8 * UNKNOWNS * B
POOL, SLACK = 512 << 20, 128 << 20


def free_bytes():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def test_memory_kept_by_plans():
    ctx = cu_context(0)
    net, rng = synth.generate(N, 0, 0, 5)
    rates = synth.rate_sets(rng, N, B)
    m = model_builder().parse_model(net.bnet())
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes, *net.fixed_spec()).state)
    dr = DeviceArray.from_host(ctx, rates)
    outs = [DeviceArray(ctx, (B, 1 << N), np.float64) for _ in range(2)]
    opts = {"precision": 1, "tol": 1e-12}
    plans = [solve_plan(ctx, t, x0.ptr) for _ in range(4)]
    assert plans[0].info()["unknowns"] == UNKNOWNS
    plans[0].solve(B, dr.ptr, outs[0].ptr, **opts)  # code, the runtime's memory
    want = outs[0].download()
    free0 = free_bytes()
    for p in plans[1:3]:
        p.solve(B, dr.ptr, outs[0].ptr, **opts)
        np.testing.assert_array_equal(outs[0].download(), want)
    solve_plan.solve_many(ctx, plans[2:], [B, B], [dr.ptr] * 2, [o.ptr for o in outs], **opts)
    for o in outs:
        np.testing.assert_array_equal(o.download(), want)
    # right-hand side, 1 / D and iterate of three plans more; a solve needs nine such vectors
    # besides, and GMRES's anchor sweeps two
    assert free0 - free_bytes() <= 3 * 3 * VECTOR + POOL + SLACK
    p = ctypes.c_void_p()
    with pytest.raises(EslError):
        check(lib().esl_device_alloc(ctx.handle, ctypes.c_size_t(1 << 55), ctypes.byref(p)), ctx.handle)
    assert free0 - free_bytes() <= 3 * 3 * VECTOR + SLACK
    for p in plans:
        p.solve(B, dr.ptr, outs[0].ptr, **opts)
        np.testing.assert_array_equal(outs[0].download(), want)
    ctx.close()
