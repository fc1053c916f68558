"""The surrogate by rows (widths up to 256, 4 hidden layers, 2048 outputs) against the
layer-by-layer kernels: workgroups of 4 and of 16 rows, the last one partial, and of 32-row tiles, widths that are no
multiple of a tile, both padded hidden widths, few and many output tiles per wave, more
than 256 rows or outputs in a sum."""
import numpy as np
import pytest

from paraexastolog_amd.surrogate import DeviceArray, Surrogate

pytestmark = pytest.mark.gpu

# inputs, hidden, hidden layers, outputs, rows
SHAPES = [(1, 1, 1, 2, 1), (13, 37, 2, 33, 15), (32, 128, 1, 512, 16), (33, 129, 3, 513, 17), (40, 256, 3, 2047, 31),
          (256, 255, 4, 777, 289), (27, 256, 2, 2048, 600), (20, 100, 2, 70, 1030), (32, 256, 3, 1500, 1025)]


def case(n_in, hidden, layers, n_out, rows):
    dims = [n_in] + [hidden] * layers + [n_out]
    rng = np.random.default_rng(n_in + rows)
    p = np.concatenate([a for i, o in zip(dims[:-1], dims[1:])
                        for a in (rng.normal(0, np.sqrt(2.0 / i), i * o), rng.normal(0, 0.1, o))]).astype(np.float32)
    x = rng.uniform(np.log(0.1), np.log(10), (rows, n_in)).astype(np.float32)
    t = rng.dirichlet(np.ones(n_out) * 0.3, rows).astype(np.float32)
    return dims, p, x, t


def widened(dims, p):
    """The same function with 264 hidden units, which runs layer by layer: the added
    units have zero weights and biases.  Also the places of the parameters in it."""
    big = [dims[0]] + [264] * (len(dims) - 2) + [dims[-1]]
    q, at, off, boff = [], [], 0, 0
    for a, b, c, d in zip(dims[:-1], dims[1:], big[:-1], big[1:]):
        w = np.zeros((c, d), np.float32)
        w[:a, :b] = p[off:off + a * b].reshape(a, b)
        q += [w.ravel(), np.pad(p[off + a * b:off + a * b + b], (0, d - b))]
        at += [(boff + np.arange(a)[:, None] * d + np.arange(b)).ravel(), boff + c * d + np.arange(b)]
        off, boff = off + a * b + b, boff + c * d + d
    return np.concatenate(q), np.concatenate(at)


@pytest.mark.parametrize("shape", SHAPES)
def test_forward_and_gradients(ctx, shape):
    dims, p, x, t = case(*shape)
    s = Surrogate(ctx, dims[0], dims[-1], hidden=dims[1], hidden_layers=len(dims) - 2, seed=5)
    s.set_params(p)
    pw, at = widened(dims, p)
    r = Surrogate(ctx, dims[0], dims[-1], hidden=264, hidden_layers=len(dims) - 2, seed=5)
    r.set_params(pw)
    got, ref = s.forward(x), r.forward(x)
    # the logits are the same sums; of the softmax's up to 2048 terms in another order,
    # each addition may round by 2^-24
    np.testing.assert_allclose(got, ref, rtol=2048 * 2.0 ** -24, atol=1e-12)
    warm = DeviceArray(ctx, got.shape, np.float64)
    dx = DeviceArray.from_host(ctx, x)
    s.predict_warm_device(len(x), dx.ptr, warm.ptr)
    np.testing.assert_array_equal(warm.download(), got.astype(np.float64))
    g, loss = s.gradients(x, t)
    g2, loss2 = s.gradients(x, t)
    assert np.array_equal(g, g2) and loss == loss2
    rg, rloss = r.gradients(x, t)
    assert abs(loss - rloss) < 1e-4 * max(1.0, abs(rloss))
    off = 0
    for a, b in zip(dims[:-1], dims[1:]):
        for size in (a * b, b):
            gg, rr = g[off:off + size], rg[at[off:off + size]]
            # what the gradients are held to against the FP64 reference
            assert np.abs(gg - rr).max() <= 2e-2 * np.abs(rr).max() + 1e-12, off
            off += size


@pytest.mark.parametrize("shape", SHAPES[1:])
def test_step_and_operand_copies(ctx, shape):
    # a step is Adam on the gradients; what the step leaves for the next products is
    # what setting the same parameters anew makes of them
    dims, p, x, t = case(*shape)
    mk = lambda: Surrogate(ctx, dims[0], dims[-1], hidden=dims[1], hidden_layers=len(dims) - 2, seed=5)
    s, u = mk(), mk()
    s.set_params(p)
    dx, dt = DeviceArray.from_host(ctx, x), DeviceArray.from_host(ctx, t)
    g, _ = s.gradients(x, t)
    s.train_step_device(len(x), dx.ptr, dt.ptr, 1e-3)
    q = s.params()
    g = g.astype(np.float64)
    # first step: the moments over their corrections are the gradient and its square
    want = p - 1e-3 * g / (np.abs(g) + 1e-8)
    # 1e-3 times the rounding of some ten FP32 operations, and the masters' own rounding
    np.testing.assert_allclose(q, want, rtol=1.2e-7, atol=1e-3 * 4e-6)
    u.set_params(q)
    np.testing.assert_array_equal(s.forward(x), u.forward(x))
    np.testing.assert_array_equal(s.gradients(x, t)[0], u.gradients(x, t)[0])
