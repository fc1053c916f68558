"""Workspaces of device-wide solves between calls: reused ones give the results of fresh
ones, on host threads too, what is kept stays within its bound, and goes back when an
allocation fails and with the context."""
import ctypes
import gc

import numpy as np
import pytest

from paraexastolog_amd import cu_context, initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from paraexastolog_amd._lib import EslError, check, lib
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu

N, UNKNOWNS = 15, 32768
SIZES = [1024, 700, 400]  # workspaces of 2.4, 1.6 and 0.9 GB
VECTORS = 8 * UNKNOWNS * sum(SIZES)  # one per plan
WIDE, POOL, SLACK = 2 << 30, 512 << 20, 256 << 20


def free_bytes():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


def made(ctx):
    net, rng = synth.generate(N, 0, 0, 5)
    rates = synth.rate_sets(rng, N, SIZES[0])
    m = model_builder().parse_model(net.bnet())
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes, *net.fixed_spec()).state)
    outs = [DeviceArray(ctx, (b, 1 << N), np.float64) for b in SIZES]
    plans = [solve_plan(ctx, t, x0.ptr) for _ in SIZES]
    assert plans[0].info()["unknowns"] == UNKNOWNS
    return plans, DeviceArray.from_host(ctx, rates), outs, (m, t, g, x0)


def test_workspaces_between_calls():
    opts = {"precision": 1, "tol": 1e-12}
    want = []
    for i, b in enumerate(SIZES):  # each from a context of its own: nothing to reuse
        ctx = cu_context(0)
        plans, dr, outs, held = made(ctx)
        plans[i].solve(b, dr.ptr, outs[i].ptr, **opts)
        want.append(outs[i].download())
        del plans, dr, outs, held
        gc.collect()
        ctx.close()

    before = free_bytes()
    ctx = cu_context(0)
    plans, dr, outs, held = made(ctx)
    free0 = free_bytes()

    def same():
        for o, w in zip(outs, want):
            np.testing.assert_array_equal(o.download(), w)
            o.upload(np.zeros_like(w))

    plans[0].solve(SIZES[0], dr.ptr, outs[0].ptr, **opts)
    # a plan's three vectors, and five more of the solve's nine (blocks up to 512 MB are kept)
    assert free0 - free_bytes() >= 8 * 8 * UNKNOWNS * SIZES[0]
    for _ in range(2):
        for p, b, o in zip(plans, SIZES, outs):
            p.solve(b, dr.ptr, o.ptr, **opts)
        same()
        assert free0 - free_bytes() <= 3 * VECTORS + WIDE + POOL + SLACK
        solve_plan.solve_many(ctx, plans, SIZES, [dr.ptr] * len(SIZES), [o.ptr for o in outs], **opts)
        same()
        assert free0 - free_bytes() <= 3 * VECTORS + WIDE + POOL + SLACK
    p = ctypes.c_void_p()
    with pytest.raises(EslError):
        check(lib().esl_device_alloc(ctx.handle, ctypes.c_size_t(1 << 55), ctypes.byref(p)), ctx.handle)
    assert free0 - free_bytes() <= 3 * VECTORS + SLACK
    plans[0].solve(SIZES[0], dr.ptr, outs[0].ptr, **opts)
    np.testing.assert_array_equal(outs[0].download(), want[0])
    del plans, dr, outs, held, p
    gc.collect()  # a table and its exported arrays refer to each other
    ctx.close()
    assert before - free_bytes() <= SLACK
