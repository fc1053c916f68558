"""A call that failed on the device reports its error once: the next call is not failed by it."""
import ctypes

import numpy as np
import pytest

from paraexastolog_amd import initial_state, model_builder, solve_plan, synth, transition_graph, transition_table
from paraexastolog_amd._lib import EslError, check, lib
from paraexastolog_amd.surrogate import DeviceArray, Surrogate

pytestmark = pytest.mark.gpu


def fail_to_allocate(ctx):
    p = ctypes.c_void_p()
    with pytest.raises(EslError) as e:
        check(lib().esl_device_alloc(ctx.handle, ctypes.c_size_t(1 << 55), ctypes.byref(p)), ctx.handle)
    assert e.value.status == 6  # out of memory


def test_failed_allocation_leaves_no_error(ctx):
    net, rng = synth.generate(10, 2, 6, 0)
    rates = synth.rate_sets(rng, 10, 3)
    m = model_builder().parse_model(net.bnet())
    fail_to_allocate(ctx)
    t = transition_table(ctx, m, rates[0])
    t.construct_table()
    g = transition_graph(ctx, t)
    g.reorganize_vertices()
    x0 = DeviceArray.from_host(ctx, initial_state(m.nodes, *net.fixed_spec()).state)
    p = solve_plan(ctx, t, x0.ptr)
    dr, out = DeviceArray.from_host(ctx, rates), DeviceArray(ctx, (3, 1 << 10), np.float64)
    fail_to_allocate(ctx)
    p.solve(3, dr.ptr, out.ptr)
    assert np.abs(out.download().sum(axis=1) - 1.0).max() <= 1e-11
    s = Surrogate(ctx, 5, 7, hidden=16, hidden_layers=2)
    fail_to_allocate(ctx)
    probs = s.forward(np.zeros((3, 5), np.float32))
    assert np.abs(probs.sum(axis=1) - 1.0).max() <= 1e-5
