"""GPU parity of the surrogate network kernels (BF16 MFMA products, FP32
accumulation, Adam) against the CPU restatement oracle/mlp_ref.py, which
rounds to BF16 at the same points and sums in float64.

Tolerances: the GPU sums in float32 in another order, so a value rounded to
BF16 can land one BF16 step (2^-8 relative) away from the oracle's; that
moves outputs and gradients by about 1e-3 relative.  Forward: rel-L2 5e-3;
gradients: rel-L2 2e-2 per layer; Adam (pure FP32): 1e-6.
"""
import numpy as np
import pytest

import se2dr_fork_amd as S
from conftest import rel_l2
from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu

SMALL = [66, 128, 128, 192]
FULL = [66, 1024, 1024, 1024, 4096]  # the surrogate's network


def layer_slices(widths):
    off = 0
    for i, o in zip(widths[:-1], widths[1:]):
        yield slice(off, off + o * i), slice(off + o * i, off + o * i + o)
        off += o * i + o


def test_init_matches_oracle():
    m = S.Mlp(SMALL, batch=64, seed=11)
    np.testing.assert_array_equal(m.params(), M.init_params(SMALL, 11).astype(np.float32))
    m.close()


@pytest.mark.parametrize("widths,batch,rows", [(SMALL, 64, 100), (FULL, 256, 300)])
def test_forward_matches_oracle(widths, batch, rows):
    m = S.Mlp(widths, batch=batch, seed=5)
    rng = np.random.default_rng(1)
    x = rng.standard_normal((rows, widths[0])).astype(np.float32)
    y = m.forward(x)
    y0, _ = M.forward(m.params(), widths, x)
    assert rel_l2(y, y0) < 5e-3
    m.close()


@pytest.mark.parametrize("widths,batch", [(SMALL, 64), (FULL, 256)])
def test_gradient_matches_oracle(widths, batch):
    m = S.Mlp(widths, batch=batch, seed=9)
    rng = np.random.default_rng(2)
    x = rng.standard_normal((batch, widths[0])).astype(np.float32)
    t = rng.standard_normal((batch, widths[-1])).astype(np.float32)
    loss, g = m.gradient(x, t)
    loss0, g0 = M.loss_and_gradient(m.params(), widths, x, t)
    assert loss == pytest.approx(loss0, rel=1e-3)
    for sw, sb in layer_slices(widths):
        assert rel_l2(g[sw], g0[sw]) < 2e-2
        assert rel_l2(g[sb], g0[sb]) < 2e-2
    # BF16 storage changes the gradient only a little against exact FP64 arithmetic
    _, g64 = M.loss_and_gradient(m.params(), widths, x, t, bf=False)
    assert rel_l2(g, g64) < 5e-2
    m.close()


def test_adam_step_matches_oracle():
    m = S.Mlp(SMALL, batch=64, seed=3)
    p0 = m.params().astype(np.float64)
    rng = np.random.default_rng(4)
    g1, g2 = rng.standard_normal(m.nparams) * 1e-2, rng.standard_normal(m.nparams) * 1e-2
    m.adam_step(g1, 1e-3)
    m.adam_step(g2, 1e-3)
    p, mm, vv = M.adam_step(p0, 0 * p0, 0 * p0, g1.astype(np.float32).astype(np.float64), 1, 1e-3)
    p, mm, vv = M.adam_step(p, mm, vv, g2.astype(np.float32).astype(np.float64), 2, 1e-3)
    np.testing.assert_allclose(m.params(), p, rtol=1e-5, atol=1e-7)
    m.close()


def test_training_reduces_the_loss():
    rng = np.random.default_rng(5)
    x = rng.uniform(-1, 1, (512, 66)).astype(np.float32)
    A = rng.standard_normal((66, 192)) / 8
    t = np.sin(x @ A).astype(np.float32)
    m = S.Mlp(SMALL, batch=64, seed=1)
    m.set_data(x, t)
    losses = m.train(40, lr=1e-3, seed=2)
    assert np.all(np.isfinite(losses)) and losses[-1] < 0.2 * losses[0]
    # the trained network predicts the training rows better than their mean
    y = m.forward(x)
    assert rel_l2(y, t) < 0.5 * rel_l2(np.broadcast_to(t.mean(axis=0), t.shape), t)
    train_ms, fwd_ms = m.timing()
    assert train_ms > 0 and fwd_ms > 0
    m.close()


def test_mlp_argument_errors():
    with pytest.raises(S.Se2wError, match="multiple of 64"):
        S.Mlp([66, 100, 64], batch=64)
    with pytest.raises(S.Se2wError):
        S.Mlp([66, 64, 64], batch=48)
    m = S.Mlp(SMALL, batch=64)
    with pytest.raises(S.Se2wError, match="64 rows"):
        m.gradient(np.zeros((32, 66)), np.zeros((32, 192)))
    with pytest.raises(S.Se2wError, match="training data"):
        m.train(1)
    m.close()


@pytest.mark.parametrize("rows", [1, 16, 17, 32, 33, 64, 65, 129, 300])
def test_forward_rows_at_the_edges_of_tiles_and_chunks(rows):
    """Row counts on both sides of the row tiles (16, 32, 64), of a batch and
    of the downloaded chunks; a row's result does not depend on the others."""
    m = S.Mlp(SMALL, batch=128, seed=5)
    x = np.random.default_rng(3).standard_normal((rows, SMALL[0])).astype(np.float32)
    y = m.forward(x)
    y0, _ = M.forward(m.params(), SMALL, x)
    assert rel_l2(y, y0) < 5e-3
    np.testing.assert_array_equal(m.forward(x[-1:]), y[-1:])
    m.close()


@pytest.mark.parametrize("widths,batch", [([66, 64, 64], 64), (SMALL, 192), ([1, 320, 64, 128], 128)])
def test_a_training_step_is_its_gradient_and_one_adam_step(widths, batch):
    """One batch trained equals the stored gradient of the same (shuffled)
    rows followed by one Adam step, bit for bit: the grouped kernel forms and
    applies the gradients in the order in which the gradient entry stores
    them."""
    rng = np.random.default_rng(6)
    x = rng.standard_normal((batch, widths[0])).astype(np.float32)
    t = rng.standard_normal((batch, widths[-1])).astype(np.float32)
    s, mask, order = 7, (1 << 64) - 1, list(range(batch))
    for i in range(batch - 1, 0, -1):  # Fisher-Yates on a splitmix64 stream
        s = (s + 0x9E3779B97F4A7C15) & mask
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & mask
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & mask
        j = int(((z ^ (z >> 31)) >> 11) * (1.0 / 9007199254740992.0) * (i + 1))
        order[i], order[j] = order[j], order[i]
    a, b = S.Mlp(widths, batch=batch, seed=8), S.Mlp(widths, batch=batch, seed=8)
    a.set_data(x, t)
    loss = a.train(1, lr=1e-3, seed=7)[0]
    loss_b, g = b.gradient(x[order], t[order])
    b.adam_step(g, 1e-3)
    np.testing.assert_array_equal(a.params(), b.params())
    assert loss == pytest.approx(loss_b, rel=1e-6)
    a.close()
    b.close()


def test_padded_rows_in_several_blocks():
    """Weights and training rows whose padded copies pass through the host in
    more than one block of 2^20 values, the last one not full: parameters come
    back as they were set, and a trained batch sees its own rows."""
    widths = [70, 9280, 64]  # first layer: rows of 70 padded to 128, 8192 of 9280 in the first block
    m = S.Mlp(widths, batch=64, seed=3)
    p = np.random.default_rng(1).uniform(-0.1, 0.1, m.nparams).astype(np.float32)
    m.set_params(p)
    np.testing.assert_array_equal(m.params(), p)
    m.close()
    small, n = [70, 64, 64], 8192 + 192
    rng = np.random.default_rng(2)
    x, t = rng.standard_normal((n, 70)).astype(np.float32), rng.standard_normal((n, 64)).astype(np.float32)
    a = S.Mlp(small, batch=n, seed=4)  # one batch of all rows: a row out of place changes the gradient
    a.set_data(x, t)
    loss = a.train(1, lr=1e-3, seed=7)[0]
    y = S.Mlp(small, batch=n, seed=4).forward(x)
    assert loss == pytest.approx(float(np.mean((y.astype(np.float64) - t) ** 2)), rel=1e-5)
    a.close()


@pytest.mark.parametrize("win,rows", [(16384, [1, 15, 16, 17, 48, 63, 64, 65, 7 * 64 + 5]), (300000, [1, 2, 6, 70])])
def test_forward_inputs_in_several_pieces(win, rows):
    """Wide inputs, of which a batch passes through the pinned buffer in pieces
    (16 rows, 1 row), on both sides of pieces and batches and round the ring
    of five pieces: every row as in a call of its own."""
    m = S.Mlp([win, 64, 64], batch=64, seed=5)
    x = np.random.default_rng(3).standard_normal((max(rows), win)).astype(np.float32)
    one = np.concatenate([m.forward(r) for r in x])
    y0, _ = M.forward(m.params(), [win, 64, 64], x[:16])
    assert rel_l2(one[:16], y0) < 5e-3
    for n in rows:
        np.testing.assert_array_equal(m.forward(x[:n]), one[:n])
    m.close()


@pytest.mark.parametrize("rows", [1, 16, 17, 63, 64, 65, 127, 128, 129, 192, 6 * 128 + 5, 7 * 128 + 70, 13 * 128])
def test_forward_in_several_chunks_of_several_batches(rows):
    """Batches of 128 rows whose outputs come down in two chunks of 64, row
    counts on both sides of chunks and batches and several times round the
    four output and five input slots: the rows of calls of their own."""
    m = S.Mlp([66, 64, 4096], batch=128, seed=6)
    x = np.random.default_rng(4).standard_normal((rows, 66)).astype(np.float32)
    want = np.concatenate([m.forward(x[r:r + 48]) for r in range(0, rows, 48)])
    np.testing.assert_array_equal(m.forward(x), want)
    y0, _ = M.forward(m.params(), [66, 64, 4096], x[-48:])
    assert rel_l2(want[-len(x[-48:]):], y0) < 5e-3
    m.close()
