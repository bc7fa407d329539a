"""Training passes of the learned model where their tiling has its edges: fewer samples than a tile of 16,
tiles past a group of four chains, a chain's eight tiles at once exceeded (above 2^19 samples), and the rows a
training step draws by itself against the same rows given explicitly."""
import numpy as np
import pytest

import components_amd as ca
import oracle

pytestmark = pytest.mark.gpu

GROUPS = [(0, 384), (384, 448), (448, 4544), (4544, 4608), (4608, 4672), (4672, 4673)]
M64 = (1 << 64) - 1


def rows_of(rng, n):
    X = np.column_stack([rng.uniform(0, 8, n), rng.uniform(0, 8, n), rng.uniform(0, 10, n), rng.uniform(0, 14, n),
                         rng.uniform(0, 1, n), rng.integers(0, 4, n)]).astype(np.float32)
    return X, rng.uniform(0, 6, n).astype(np.float32)


def model():
    m = ca.Mlp(seed=7)
    w = m.get_weights()
    w[384:448] += 0.05  # keep first-layer units active
    m.set_weights(w)
    return m, w


def close(g, ref):
    for lo, hi in GROUPS:  # bf16 products summed in f32, as the oracle rounds them
        assert np.linalg.norm(g[lo:hi] - ref[lo:hi]) < 2e-3 * (np.linalg.norm(ref[lo:hi]) + 1e-12), (lo, hi)


@pytest.mark.parametrize("n", [1, 15, 17, 65, 511, 513, 4097])
def test_gradients_at_tile_edges(n):
    X, y = rows_of(np.random.default_rng(n), n)
    m, w = model()
    g, loss = m.gradients(X, y)
    m.close()
    ref, rloss = oracle.mlp_grad(w.astype(np.float64), X, y, bf16=True)
    assert loss == pytest.approx(rloss, rel=1e-4)
    close(g, ref)


@pytest.mark.parametrize("n", [(1 << 19) + 16, 700001])
def test_gradients_of_long_chains(n):
    """Repeated rows: the batch's gradient is the mean of its parts'."""
    base = 4097
    X, y = rows_of(np.random.default_rng(2), base)
    m, w = model()
    g, loss = m.gradients(np.resize(X, (n, 6)), np.resize(y, n))
    m.close()
    whole, part = divmod(n, base)
    ref, rloss = oracle.mlp_grad(w.astype(np.float64), X, y, bf16=True)
    ref, rloss = ref * (whole * base / n), rloss * (whole * base / n)
    if part:
        pg, pl = oracle.mlp_grad(w.astype(np.float64), X[:part], y[:part], bf16=True)
        ref, rloss = ref + pg * (part / n), rloss + pl * (part / n)
    assert loss == pytest.approx(rloss, rel=1e-4)
    close(g, ref)


def drawn(seed, step, batch, count):
    """Rows of one step: SplitMix64 of a counter, scaled to the dataset."""
    mix = oracle.splitmix64_mix
    base = mix((mix((seed & 0xFFFFFFFF) ^ (12 << 40)) + 12) & M64)
    return np.array([(mix((base + (step * batch + i + 1) * 0x9E3779B97F4A7C15) & M64) * count) >> 64
                     for i in range(batch)], np.int64)


@pytest.mark.parametrize("batch", [16, 100, 8192])
def test_step_draws_and_updates(batch):
    X, y = rows_of(np.random.default_rng(4), 30011)
    m, w = model()
    m.add_dataset(X, y)
    rows = drawn(5, 0, batch, len(y))
    g, loss = m.gradients(X[rows], y[rows])
    st = m.train(steps=1, batch=batch, lr=3e-3, seed=5)
    after = m.get_weights()
    assert st["first_loss"] == loss and st["last_loss"] == loss  # the same sums in the same order
    # Adam's first step: m / bc1 = g, v / bc2 = g^2
    g = g.astype(np.float64)
    step = 3e-3 * g / (np.abs(g) + 1e-8)
    moved = np.abs(g) > 1e-12
    assert np.allclose((w - after)[moved], step[moved], rtol=1e-3, atol=1e-6)
    assert np.array_equal(after[g == 0], w[g == 0])
    # and the bf16 copies are the new weights'
    s = m.forward(X[:100])
    m.close()
    ref = oracle.mlp_forward(after.astype(np.float64), X[:100], bf16=True)
    assert np.linalg.norm(s - ref) / np.linalg.norm(ref) < 1e-4
