"""Training steps on small batches (their own kernels) against the large-batch
kernels, which the FP64 oracle pins: the same gradients from a batch and from
that batch repeated until it takes the large path, and weights, their BF16
copies and the transposed copies consistent after Adam steps."""
import numpy as np
import pytest

from qiron import surrogate as S

pytestmark = pytest.mark.gpu


def blocks(net, H):
    sizes = [net.k_in * H, H, H * H, H, H * H, H, H, 1]
    o = np.cumsum([0] + sizes)
    return [slice(o[k], o[k + 1]) for k in range(8)]


# (inputs, width, rows, repeats): 16-row and ragged-to-32 batches, one chunk of
# 256 rows and several, K below one slice and up to 16 slices. The mean over a
# power-of-two number of repeats scales every term exactly, so both sides
# differ by the order of FP32 sums and, where such a difference crosses a
# rounding boundary, a BF16 ulp (2^-8) of a few activations per thousand:
# within 1e-3 of a block's norm.
@pytest.mark.parametrize("n_in,H,rows,reps", [(5, 64, 16, 1024), (5, 64, 272, 64), (203, 256, 400, 32), (33, 512, 1040, 8),
                                              (1000, 128, 48, 512), (17, 64, 8208, 2)])
def test_small_batch_gradients_match_large_batch(ctx, n_in, H, rows, reps):
    net = S.MLP(n_in, H, seed=11)
    rng = np.random.default_rng(rows)
    x = rng.uniform(-1, 1, size=(rows, n_in)).astype(np.float32)
    t = rng.normal(size=rows).astype(np.float32)
    ls, gs = net.gradients(x, t)
    ll, gl = net.gradients(np.tile(x, (reps, 1)), np.tile(t, reps))
    assert abs(ls - ll) <= 1e-4 * ll
    for k, b in enumerate(blocks(net, H)):
        a, r = gs[b].astype(np.float64), gl[b].astype(np.float64)
        assert np.linalg.norm(a - r) <= 1e-3 * np.linalg.norm(r), k


@pytest.mark.parametrize("n_in,H,batch", [(5, 64, 16), (203, 256, 272), (40, 512, 1024)])
def test_small_batch_epoch_is_adam_on_the_gradients(ctx, n_in, H, batch):
    net = S.MLP(n_in, H, seed=12)
    rng = np.random.default_rng(batch)
    x = rng.uniform(-1, 1, size=(batch, n_in)).astype(np.float32)
    t = rng.normal(size=batch).astype(np.float32)
    p0 = net.params().astype(np.float64)
    loss, g = net.gradients(x, t)
    net.set_data(x, t)
    lr = 1e-3
    assert abs(net.train_epoch(batch, lr, 1) - loss) <= 1e-5 * loss
    # a first Adam step is -lr g / (|g| + 1e-8); where |g| is above 1e-3 of the
    # largest, the order of the sums (rows shuffled) cannot move it by 1e-2, and
    # the FP32 update rounds to half an ulp of the parameter
    g = g.astype(np.float64)
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    d = net.params().astype(np.float64) - p0
    ref = -lr * g / (np.abs(g) + 1e-8)
    assert np.all(np.abs(d - ref)[big] <= 1e-2 * lr + 2.0 ** -24 * np.abs(p0[big]))
    # after more steps, a network given these parameters has the same copies
    for s in range(3):
        net.train_epoch(batch, lr, 2 + s)
    other = S.MLP(n_in, H, seed=13)
    other.set_params(net.params())
    la, ga = net.gradients(x, t)
    lb, gb = other.gradients(x, t)
    assert la == lb and np.array_equal(ga, gb)
    assert np.array_equal(net.predict(x), other.predict(x))
