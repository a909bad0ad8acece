"""The estimator's fused passes (networks of at most 128 inputs and hidden units) at the edges of their
tiles and widths, and the first widths past them (generic passes), against the float64 oracle.

Tolerances: FP32 sums of at most 129 products a layer, four or fewer layers deep, are within
129 * 2^-24 * layers < 4e-5 of their terms' magnitude; gradients sum as many rows again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [  # inputs, hidden units, hidden layers, rows: tile edges (32 rows, 16 inputs, 32 units), a
    # pass of more tiles than work-groups, one layer, the deepest that fits, and widths past the limit
    (32, 128, 3, 1), (32, 128, 3, 31), (32, 128, 3, 33), (32, 128, 3, 9001), (1, 1, 1, 5), (16, 32, 2, 32),
    (17, 33, 2, 70), (128, 128, 1, 64), (31, 100, 8, 100), (127, 65, 4, 129), (129, 64, 2, 50), (20, 129, 2, 50)]


@pytest.mark.parametrize("n_in,n_hidden,layers,n", SHAPES)
def test_passes_match_oracle(engine, n_in, n_hidden, layers, n):
    from oracle import mlp_ref

    m = engine.mlp(n_in=n_in, n_hidden=n_hidden, n_hidden_layers=layers, seed=3)
    try:
        dims = [n_in] + [n_hidden] * layers + [1]
        rng = np.random.default_rng(n_in * 1000 + n)
        p = m.parameters() + rng.uniform(-0.05, 0.05, m.n_params).astype(np.float32)  # biases too
        m.set_parameters(p)
        p = m.parameters()
        x = rng.uniform(0, 1, (n, n_in)).astype(np.float32)
        y = rng.uniform(0, 1, n).astype(np.float32)
        want, _ = mlp_ref.forward(p, dims, x)
        assert np.allclose(m.forward(x), want, rtol=1e-4, atol=1e-4 * max(np.abs(want).max(), 1e-3))
        loss, g = m.gradients(x, y)
        loss_ref, g_ref = mlp_ref.loss_and_grads(p, dims, x, y)
        assert abs(loss - loss_ref) <= 1e-4 * loss_ref
        assert np.allclose(g, g_ref, rtol=1e-3, atol=1e-4 * np.abs(g_ref).max())
        assert np.array_equal(m.parameters(), p)  # gradients change nothing
    finally:
        m.free()


@pytest.mark.parametrize("n_in,n_hidden,layers,n,batch", [(32, 128, 3, 700, 256), (17, 33, 2, 100, 100), (20, 129, 1, 64, 64)])
def test_updates_match_oracle(engine, n_in, n_hidden, layers, n, batch):
    """One epoch of Adam whose minibatches all hold the same row, so that their shuffling plays no
    part, against Adam in float64 on the oracle's gradients.  A weight may round to the neighbouring
    bfloat16 value: 2^-8 of it."""
    from oracle import mlp_ref

    m = engine.mlp(n_in=n_in, n_hidden=n_hidden, n_hidden_layers=layers, seed=9)
    try:
        dims = [n_in] + [n_hidden] * layers + [1]
        rng = np.random.default_rng(n)
        master = m.parameters().astype(np.float64)
        x = np.repeat(rng.uniform(0, 1, (1, n_in)).astype(np.float32), n, axis=0)
        y = np.full(n, 3.0, np.float32)
        m.set_parameters(master.astype(np.float32))
        loss = m.train(x, y, epochs=1, batch=batch, lr=1e-3, seed=1)
        m1, m2, total = np.zeros(m.n_params), np.zeros(m.n_params), 0.0
        for step, start in enumerate(range(0, n, batch), 1):
            k = min(batch, n - start)
            sq, g = mlp_ref.loss_and_grads(mlp_ref.bf16_round(master), dims, x[:k], y[:k])
            total += sq * k
            m1, m2 = 0.9 * m1 + 0.1 * g, 0.999 * m2 + 0.001 * g * g
            master -= 1e-3 * (m1 / (1 - 0.9 ** step)) / (np.sqrt(m2 / (1 - 0.999 ** step)) + 1e-8)
        want = mlp_ref.bf16_round(master)
        got = m.parameters()
        assert np.allclose(got, want, rtol=2.0 ** -7, atol=1e-5)
        assert np.mean(got != want) < 0.01
        assert abs(loss - total / n) <= 1e-4 * total / n
    finally:
        m.free()
