"""The fused training step (hidden width 256) against the layer-by-layer oracle
network, over the shapes its tiles and launches depend on: layer counts from
the smallest to the largest it takes, one member and several, minibatches of
one 64-row block up to more than its 256-row loads, and a width it does not
take (64: the layer-by-layer kernels)."""
import numpy as np
import pytest

from geliosphere_amd.surrogate import N_IN as NI
from oracle import surrogate_ref as R

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30))


@pytest.mark.parametrize("layers,members,rows,hidden", [(1, 1, 1, 256), (1, 3, 64, 256), (2, 2, 65, 256), (4, 4, 256, 256),
                                                        (4, 4, 320, 256), (7, 5, 577, 256), (8, 1, 130, 256), (2, 2, 100, 64)])
def test_gradients_over_shapes(layers, members, rows, hidden):
    from geliosphere_amd.surrogate import Surrogate
    rng = np.random.default_rng(layers * 1000 + rows)
    s = Surrogate(0, seed=5, n_hidden_layers=layers, n_members=members, hidden=hidden, batch=64)
    x = rng.normal(0, 1, (rows, NI)).astype(np.float32)
    y = rng.normal(-1, 0.5, (rows, 30)).astype(np.float32)
    w = rng.uniform(0.1, 2, (rows, 30)).astype(np.float32)
    s.set_normalization(np.zeros(NI), np.ones(NI), np.full(NI, -10.0), np.full(NI, 10.0))
    g, loss = s.gradients(x, y, w)
    pm, lay = s.layout()
    P = s.get_params().astype(np.float64)
    xp = R.pad_inputs(x.astype(np.float64), np.zeros(NI), np.ones(NI))
    yp, wp = np.zeros((rows, R.PAD)), np.zeros((rows, R.PAD))
    yp[:, :30], wp[:, :30] = y, w
    for m in range(members):
        l_ref, g_ref = R.loss_and_grads(R.unpack(P[m * pm:(m + 1) * pm], lay), xp, yp, wp, emulate_bf16=True)
        assert abs(loss[m] - l_ref) <= 2e-3 * abs(l_ref)
        # every layer by itself: bf16 rounding of activations and gradients, 2^-9
        # relative per layer passed
        for (wo, bo, n_out, n_in), (gw, gb) in zip(lay, g_ref):
            gm = g[m * pm:(m + 1) * pm].astype(np.float64)
            assert rel_l2(gm[wo:wo + n_out * n_in], np.asarray(gw).ravel()) < 1e-2
            assert rel_l2(gm[bo:bo + n_out], np.asarray(gb).ravel()) < 1e-2


@pytest.mark.parametrize("batch,layers", [(64, 1), (320, 4), (512, 7)])
def test_one_training_step_is_adam_on_the_gradients(batch, layers):
    """One minibatch holding every row (in some order): the updated parameters
    are Adam's first step on the gradients of all rows."""
    from geliosphere_amd.surrogate import Surrogate
    rng = np.random.default_rng(batch)
    lr, wd = 1e-3, 1e-2
    s = Surrogate(0, seed=6, n_hidden_layers=layers, n_members=2, batch=batch, lr=lr, weight_decay=wd)
    x = rng.normal(0, 1, (batch, NI)).astype(np.float32)
    y = rng.normal(-1, 0.5, (batch, 30)).astype(np.float32)
    w = rng.uniform(0.1, 2, (batch, 30)).astype(np.float32)
    s.set_normalization(np.zeros(NI), np.ones(NI), np.full(NI, -10.0), np.full(NI, 10.0))
    p0 = s.get_params().astype(np.float64)
    g = s.gradients(x, y, w)[0].astype(np.float64)
    s.train(x, y, w, 1)
    # the first step: m / c1 = g, sqrt(v / c2) = |g|
    want = p0 - lr * (g / (np.abs(g) + 1e-8) + wd * p0)
    got = s.get_params().astype(np.float64)
    # the rows are summed in another order: gradients near zero may turn round
    firm = np.abs(g) > 1e-4 * np.abs(g).max()
    assert firm.mean() > 0.5
    assert np.max(np.abs(got - want)[firm]) < 1e-3 * lr + 1e-6
    assert np.max(np.abs(got - want)) <= 2.01 * lr
    # the next prediction uses the updated weights
    t = Surrogate(0, seed=9, n_hidden_layers=layers, n_members=2, batch=batch)
    t.set_params(s.get_params())
    t.set_normalization(*s.get_normalization())
    assert np.array_equal(s.predict(x)[0], t.predict(x)[0])
