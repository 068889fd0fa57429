"""GPU tests of the sum over a training batch's blocks where losing a part of it
shows: one sample, in the first, last or any other row of the sum, has a target
so far off that its row is nearly all of the gradient; and the sum followed by
Adam from moments that are not zero, where the size of the gradient counts."""
import numpy as np
import pytest

from oracle import warm_mlp as M

pytestmark = pytest.mark.gpu

# (samples, the sample that dominates): 16 samples a row up to 1,024 rows,
# 128 rows a chunk of the sum; past 1,024 rows the groups wrap
CASES = [(1, 0), (17, 16), (2048, 2047), (2049, 2048), (2049, 0), (2049, 2032), (4096, 4095), (4097, 4096),
         (4097, 2048), (16384, 16383), (16385, 16384), (16385, 14336), (20001, 20000)]


def _samples(count, dominant):
    rng = np.random.default_rng(count + dominant)
    X = rng.uniform(-1, 1, size=(count, 8)).astype(np.float32)
    y = rng.uniform(-1, 1, size=count).astype(np.float32)
    y[dominant] = 1.0e4 * max(1.0, count / 1000.0)
    return X, y


@pytest.mark.parametrize("count,dominant", CASES)
def test_no_row_is_lost(pbf, count, dominant):
    """Against the numpy gradient: bf16 operands leave 1e-2 of its norm (the
    bound of the other gradient tests), a lost row nearly all of it."""
    X, y = _samples(count, dominant)
    m = pbf.WarmModel(count)
    m.init(3)
    p = m.params()
    m.add_samples(X, y)
    g, _ = m.gradient(0, count)
    ref, _ = M.gradient(p, X, y, rounding=True)
    rest = np.delete(np.arange(count), dominant)
    if count > 1:  # (the others' share, as a mean over `count`)
        others = M.gradient(p, X[rest], y[rest], rounding=True)[0] * (len(rest) / count)
        assert np.linalg.norm(others) <= 0.05 * np.linalg.norm(ref)
    assert np.linalg.norm(g - ref) <= 1e-2 * np.linalg.norm(ref)
    m.close()


@pytest.mark.parametrize("count,dominant", CASES)
def test_one_batch_epoch_from_moments(pbf, count, dominant):
    """train over one batch against gradient and adam_step from the same
    parameters and moments.  The first step's gradient is half of the second's,
    so the update is lr (0.045 + 0.1) g / 0.19 / sqrt(0.625 g^2), 0.965 lr where
    |g| is well above eps, and changes by less than lr times the relative change
    of g: 1e-3 lr for the rounding of the two sums' orders (1e-4 of a sum that
    one row dominates), and by 0.08 lr if g were twice as large."""
    X, y = _samples(count, dominant)
    m = pbf.WarmModel(count)
    m.init(3)
    p = m.params()
    m.add_samples(X, y)
    lr = 1e-3
    g0, _ = m.gradient(0, count)

    def start():
        m.set_params(p)
        m.adam_step(np.float32(0.5) * g0, 1e-12)  # moments, and (nearly) the same parameters

    start()
    q = m.params()
    g, loss = m.gradient(0, count)
    m.adam_step(g, lr)
    stepped = m.params()
    start()
    trained_loss = m.train(1, count, lr, 9)
    trained = m.params()
    big = np.abs(g) > 1e-2 * np.abs(g).max()
    assert big.any()
    assert np.abs(stepped - q)[big].min() > 0.9 * lr
    assert np.abs(trained - stepped)[big].max() <= 1e-3 * lr + 2 * np.spacing(np.abs(p).max())
    assert abs(trained_loss - loss) <= 1e-5 * abs(loss)
    m.close()
