"""The padding columns of W1 and W3 take no part in the network, whatever finite
values a caller set them to: predictions, losses, gradients and the prediction
after an optimiser step are the same bit for bit (up to 8,192 slots, whose partial
gradients are one chunk).  A padding weight that is no number makes the prediction
none, as zero times it does."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc
from oracle import surrogate_ref as sr

pytestmark = pytest.mark.gpu


def solver():
    t = sc.preset_tunables(0)
    p = sa.scene_lattice(60, 50, 0.4, 0.05, seed=9, x0=0.25, y0=0.25)
    rng = np.random.default_rng(9)
    p["v_x"] = rng.uniform(-2, 2, len(p)).astype(np.float32)
    p["v_y"] = rng.uniform(-2, 2, len(p)).astype(np.float32)
    s = sa.Solver(t, sa.make_box(30, 24), len(p))
    s.upload(p)
    s.phase("hash")
    return s


def answers(s, p, target):
    m = sa.Surrogate(seed=1)
    m.params = p
    m.zero_grads()
    pred = m.predict(s)
    loss = m.backward(s, target)
    grads = m.grads()
    m.adam(1e-2)
    return pred, np.float32(loss), grads, m.predict(s)


@pytest.mark.parametrize("columns", [slice(6, 8), slice(8, 14), slice(6, 16)])
def test_padding_columns_have_no_effect(columns):
    s = solver()
    rng = np.random.default_rng(4)
    p = sr.random_params(31).astype(np.float32)
    target = rng.normal(0, 0.1, (s.n, 2)).astype(np.float32)
    want = answers(s, p, target)
    q = p.copy()
    w1 = q[sr.oW1:sr.oW2].reshape(sr.H, sr.KE)
    w1[:, columns] = rng.uniform(-3, 3, w1[:, columns].shape)
    q[sr.oW3:sr.oW4].reshape(sr.H, sr.KN)[:, 69:] = rng.uniform(-3, 3, (sr.H, sr.KN - 69))
    for what, a, b in zip(("prediction", "loss", "gradients", "next prediction"),
                          answers(s, q, target), want):
        same = a.tobytes() == b.tobytes()
        assert same, what
    m = sa.Surrogate(seed=1)
    w1[17, 11] = np.nan
    m.params = q
    assert np.isnan(m.predict(s)).all()
    s.close()
