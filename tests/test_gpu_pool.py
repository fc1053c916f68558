"""Device buffers that a context keeps between calls: the results on reused blocks
are those on fresh ones, what is kept stays within its bound and goes back with
the context, and objects that outlive their context can still be destroyed."""
import ctypes
import gc

import numpy as np
import pytest

from paraexastolog_amd import cu_context, initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from paraexastolog_amd._lib import lib
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu

BOUND = 512 << 20


def free_bytes():
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0  # of the runtime the library is linked to
    return f.value


def pass_over(ctx, N, seed):
    net, rng = synth.generate(N, 2, seed, 0)
    rates = synth.rate_sets(rng, N, 3)
    m = model_builder().parse_model(net.bnet())
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    fixed, vals = net.fixed_spec()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes, fixed, vals).state)
    p = solve_plan(ctx, t, x0.ptr)
    dr, out = DeviceArray.from_host(ctx, rates), DeviceArray(ctx, (3, 1 << N), np.float64)
    p.solve(3, dr.ptr, out.ptr)
    return (m, t, g, x0, p, dr, out), (out.download(), np.array(t.rows), np.array(g.reordered_vertices))


def test_reused_buffers_and_bound():
    sizes = [(18, 1), (16, 2), (20, 0), (17, 3), (18, 4)]
    ref = {}
    for N, seed in sizes:
        fresh = cu_context(0)
        held, ref[N, seed] = pass_over(fresh, N, seed)
        del held
        gc.collect()  # a table and its exported arrays refer to each other
        fresh.close()
    # from here on, code objects and the runtime's own memory are in place
    free0 = free_bytes()
    ctx = cu_context(0)
    for _ in range(2):
        for N, seed in sizes:
            held, got = pass_over(ctx, N, seed)
            for a, b in zip(got, ref[N, seed]):
                np.testing.assert_array_equal(a, b)
            del held
            gc.collect()
            # beside the pool: the context's own scratch, some words per state
            assert free0 - free_bytes() <= BOUND + (256 << 20)
    held, _ = pass_over(ctx, 18, 1)
    ctx.close()
    del held  # after their context
    gc.collect()
    assert free0 - free_bytes() <= 256 << 20
