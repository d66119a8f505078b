"""The two kernels of a training step at the edges of their tiles: 32 rows per
workgroup, 16 rows per fragment and 256 rows per stage of the weight
gradients (128 of the bias gradients)."""
import numpy as np
import pytest

from cubez_amd import World, scenes, surrogate
from tests.test_gpu_surrogate import NO, bf16, ref_forward

pytestmark = pytest.mark.gpu


def _model(seed=0):
    rng = np.random.default_rng(seed)
    w = World(scenes.batched(0, 2))
    p = np.concatenate([np.concatenate([rng.uniform(-1, 1, i * o) * np.sqrt(6.0 / i), rng.uniform(-0.1, 0.1, o)])
                        for i, o in surrogate.LAYERS]).astype(np.float32)
    norm = np.concatenate([rng.normal(0, 1, 40), rng.uniform(0.5, 2, 40), rng.normal(0, 1, NO),
                           rng.uniform(0.5, 2, NO)]).astype(np.float32)
    w.sur_set_norm(norm)
    w.sur_set_params(p)
    return w, p, norm, rng


def _grad(params, norm, X, Y):
    """FP64 backprop with the kernels' BF16 roundings of activations, weights
    and dL/dZ."""
    mo, so = norm[80:80 + NO].astype(np.float64), norm[80 + NO:].astype(np.float64)
    y, _, acts, zs = ref_forward(params, norm, X)
    e = y - (Y - mo) / so
    dz = bf16((2.0 * e / e.size).astype(np.float32)).astype(np.float64)
    out, layers = [], surrogate.unpack(params)
    for l in range(len(layers) - 1, -1, -1):
        out.append((dz.T @ acts[l], dz.sum(axis=0)))
        if l > 0:
            s = 1.0 / (1.0 + np.exp(-zs[l - 1]))
            dz = (dz @ bf16(layers[l][0]).astype(np.float64)) * s * (1.0 + zs[l - 1] * (1.0 - s))
            dz = bf16(dz.astype(np.float32)).astype(np.float64)
    return out[::-1], np.mean(e * e)


def test_gradient_at_the_edges_of_the_tiles():
    """Both sides round to BF16 at the same places, so they differ by FP32
    sums (some 1e-6) and by the few roundings those tip over: a share of
    1e-6 / 2^-8 of the values by 2^-8 each, 6e-5 of a norm per rounding and
    seven of them; a row or a column that is lost is 1e-2 and more at these
    batches."""
    w, params, norm, rng = _model()
    for rows in (1, 31, 32, 33, 64, 65, 127, 129, 255, 256, 257, 511, 513, 4096, 4097, 777):
        X = rng.normal(0, 1.0, (rows, 40)).astype(np.float32)
        Y = rng.normal(0, 1.0, (rows, NO)).astype(np.float32)
        g, loss = w.sur_grad(X, Y)
        want, lref = _grad(params, norm, X, Y)
        assert abs(loss - lref) < 1e-3 * lref, rows
        off = 0
        for l, (gw, gb) in enumerate(want):
            for part in (gw, gb):
                got = g[off:off + part.size].reshape(part.shape)
                off += part.size
                assert np.linalg.norm(got - part) < 2e-3 * np.linalg.norm(part), (rows, l, part.shape)
        assert off == g.size
    w.close()


@pytest.mark.parametrize("batch", [1, 33, 288])
def test_training_step_is_adam_on_the_sampled_rows(batch):
    """Each step against the gradient of the rows it samples and Adam in
    float32 (bias corrections from powf: 6e-5 of an update, updates at most
    about lr), and the packed weights against freshly uploaded ones."""
    w, params, norm, rng = _model(1)
    rows, lr, seed = 777, 1e-3, 5
    X = rng.normal(0, 1.0, (rows, 40)).astype(np.float32)
    Y = rng.normal(0, 1.0, (rows, NO)).astype(np.float32)
    w.sur_load_dataset(X, Y)
    f, m, v = np.float32, np.zeros_like(params), np.zeros_like(params)
    mask = (1 << 64) - 1
    for t in range(1, 4):
        idx = []
        for i in range(batch):
            z = ((seed + t) * 0xD1B54A32D192ED03 + (i + 1) * 0x9E3779B97F4A7C15) & mask
            z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & mask
            z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
            idx.append((z ^ (z >> 31)) % rows)
        p = w.sur_get_params()
        g, loss = w.sur_grad(X[idx], Y[idx])
        assert w.sur_train(1, batch, lr, seed + t)[0] == f(loss)
        m = f(0.9) * m + (f(1) - f(0.9)) * g
        v = f(0.999) * v + (f(1) - f(0.999)) * g * g
        c1, c2 = f(1) / (f(1) - f(0.9) ** f(t)), f(1) / (f(1) - f(0.999) ** f(t))
        want = p - f(lr) * (m * c1) / (np.sqrt(v * c2) + f(1e-8))
        got = w.sur_get_params()
        np.testing.assert_allclose(got, want, rtol=2.0**-23, atol=2e-4 * lr)
        with World(scenes.batched(0, 2)) as fresh:
            fresh.sur_set_norm(norm)
            fresh.sur_set_params(got)
            assert np.array_equal(fresh.sur_predict(X), w.sur_predict(X))
            gf, lf = fresh.sur_grad(X, Y)
        gw, lw = w.sur_grad(X, Y)
        assert lf == lw and np.array_equal(gf, gw)
    w.close()
