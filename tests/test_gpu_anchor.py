"""Rate sets whose mass has not settled when the anchors are picked: the picked row's
entry is a thousandth of the largest one or less, and rounding alone keeps the residual
above the tolerance until the anchor is moved there."""
import numpy as np
import pytest

from paraexastolog_amd import cu_context, initial_state, model_builder, solve_plan, solver, synth, transition_graph, transition_table
from paraexastolog_amd.surrogate import DeviceArray

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = cu_context(0)
    yield c
    c.close()


def batch(seed, sets, N):
    return np.exp(np.random.default_rng(seed).uniform(np.log(0.1), np.log(10.0), (sets, 2 * N)))


def flip_masks(net):
    s = np.arange(1 << net.N)
    mask = np.zeros_like(s)
    for i in range(net.N):
        idx = sum(((s >> j) & 1) << k for k, j in enumerate(net.inputs[i]))
        mask |= (np.asarray(net.tables[i])[idx] ^ ((s >> i) & 1)) << i
    return mask


def generator_times(mask, N, rates, x):
    """K x, column s of K being the rates out of state s."""
    y = np.zeros_like(x)
    s = np.arange(len(x))
    for i in range(N):
        f = np.where((mask >> i) & 1, rates[2 * i + ((s >> i) & 1)] * x, 0.0)
        y -= f
        y += f[s ^ (1 << i)]
    return y


class Kept:
    def __init__(self, ctx, net):
        self.net = net
        self.m = model_builder().parse_model(net.bnet())
        self.t = transition_table(ctx, self.m, np.ones(2 * net.N))
        self.t.construct_table()
        self.g = transition_graph(ctx, self.t)
        self.g.reorganize_vertices()
        self.x0 = initial_state(self.m.nodes, *net.fixed_spec())
        self.dx0 = DeviceArray.from_host(ctx, self.x0.state)
        self.p = solve_plan(ctx, self.t, self.dx0.ptr)
        self.ctx = ctx

    def solve(self, rates, call="solve", **opts):
        out = DeviceArray(self.ctx, (len(rates), 1 << self.net.N), np.float64)
        dr = DeviceArray.from_host(self.ctx, rates)
        getattr(self.p, call)(len(rates), dr.ptr, out.ptr, **opts)
        return out.download(), self.p.set_results(len(rates))


@pytest.fixture(scope="module")
def n16(ctx):
    """2,048 states in one terminal component."""
    return Kept(ctx, synth.generate(16, 2, 11, 0)[0])


def dense(mask, N, rates, states):
    """Stationary vector of a terminal component, the normalisation in place of one row."""
    n = len(states)
    pos = np.full(1 << N, -1)
    pos[states] = np.arange(n)
    A = np.zeros((n, n))
    for i in range(N):
        s = states[(mask[states] >> i) & 1 == 1]
        r = rates[2 * i + ((s >> i) & 1)]
        A[pos[s], pos[s]] -= r
        A[pos[s ^ (1 << i)], pos[s]] += r
    A[-1] = 1.0
    return np.linalg.solve(A, np.eye(n)[-1])


# batch seed, rate set in it: the largest entry is 4,500, 6,600 and 2,800 times that of the row picked first
BAD = [(1337, 77), (8820, 16), (10873, 197)]


@pytest.mark.parametrize("seed,row", BAD)
@pytest.mark.parametrize("B", [1, 3, 250, 257])
def test_per_set(n16, seed, row, B):
    rates = batch(seed, 250, 16)
    if B < 250:
        rates = rates[[row] + list(range(B - 1))]
        row = 0
    elif B > 250:
        rates = np.concatenate([rates, batch(5, B - 250, 16)])
    x, (res, its, meth) = n16.solve(rates, precision=0, tol=1e-12)
    assert res.max() <= 1e-12 and (meth == 0).all()
    states = np.flatnonzero(x[row])
    assert len(states) == 2048
    # the relative residual of a component's vector bounds its error by the conditioning that
    # the anchor leaves; 1e-10 in L1 is what the batch tests allow at this tolerance
    want = dense(flip_masks(n16.net), 16, rates[row], states)
    assert np.abs(x[row, states] - want).sum() <= 1e-10
    # the other sets' vectors do not depend on it (the same kernel solves both batches)
    others = np.delete(np.arange(B), row)
    if B > 1:
        few = rates.copy()
        few[row] = few[others[0]]
        y, _ = n16.solve(few, precision=0, tol=1e-12)
        np.testing.assert_array_equal(x[others], y[others])
    for opts in ({"graph": 1}, {"graph": 1}, {"precision": 1}):
        y, (res, _, _) = n16.solve(rates, **{"precision": 0, "tol": 1e-12, **opts})
        assert res.max() <= 1e-12
        np.testing.assert_array_equal(x, y)  # vectors are FP64 in both precisions


def test_no_allocation_and_many(ctx, n16):
    rates = batch(8820, 250, 16)[15:18]
    x, _ = n16.solve(rates, precision=0, tol=1e-12)
    y, (res, _, _) = n16.solve(rates, "solve_noalloc", precision=0, tol=1e-12)
    assert res.max() <= 1e-12
    np.testing.assert_array_equal(x, y)
    out = DeviceArray(ctx, x.shape, np.float64)
    dr = DeviceArray.from_host(ctx, rates)
    for graph in (0, 1, 1):
        solve_plan.solve_many(ctx, [n16.p], [3], [dr.ptr], [out.ptr], precision=0, tol=1e-12, graph=graph)
        np.testing.assert_array_equal(out.download(), x)


def test_class_api_and_full_export(ctx, n16):
    rates = batch(8820, 250, 16)[16]
    s = solver(ctx, n16.t, n16.g, rates, n16.x0)  # to the default 1e-13
    s.solve()
    states = np.flatnonzero(s.final_state)
    want = dense(flip_masks(n16.net), 16, rates, states)
    assert np.abs(s.final_state[states] - want).sum() <= 1e-10
    term = s.solution_term
    np.testing.assert_allclose(term.data[np.argsort(term.indices)], s.final_state[states], rtol=1e-9, atol=1e-16)


@pytest.mark.parametrize("seed", [1842, 2368])
def test_device_wide(ctx, seed):
    """524,288 unknowns; one of the 16 sets misses 1e-12 with its first anchor (by 20 to 30 times)."""
    k = Kept(ctx, synth.generate(20, 0, 7, 5)[0])
    rates = batch(seed, 16, 20)
    x, (res, its, meth) = k.solve(rates, precision=1, tol=1e-12)
    assert res.max() <= 1e-12 and (meth == 0).all()
    mask = flip_masks(k.net)
    for b in range(16):
        # a residual of 1e-12 beside the anchor's 1, which is half of the largest entry at least;
        # the anchor's own row holds what the 524,287 others leave
        y = generator_times(mask, 20, rates[b], x[b])
        assert np.abs(y).max() <= 2 * 724 * 1e-12 * x[b].max()
    # a set's vector does not depend on the others'
    for b in (0, 7, 15):
        y, _ = k.solve(np.repeat(rates[[b]], 16, axis=0), precision=1, tol=1e-12)
        np.testing.assert_array_equal(y[b], x[b])
