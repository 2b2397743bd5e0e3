"""The network's kernels at the edges of their tiles: groups of 16 particles
that are not full, scenes that end inside a workgroup's four groups or one
particle into the next slot range, edge lists of no edge, of a part of a
16-edge tile and of more than the LDS edge buffer holds.  Tolerances are those
of the full-size comparison with the FP64 oracle (BF16 weights and
activations), stated there."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc
from oracle import surrogate_ref as sr
from tests.test_gpu_surrogate import device_weights, oracle_batch

pytestmark = pytest.mark.gpu


def batch(counts, spacing):
    t = sc.preset_tunables(0)
    scenes = []
    for k, n in enumerate(counts):
        nx = max(1, int(np.ceil(np.sqrt(n))))
        p = sa.scene_lattice(nx, -(-n // nx), spacing, 0.1 * spacing, seed=3 + k, x0=0.25,
                             y0=0.25)[:n].copy()
        rng = np.random.default_rng(k)
        p["v_x"] = rng.uniform(-1, 1, n).astype(np.float32)
        p["v_y"] = rng.uniform(-1, 1, n).astype(np.float32)
        scenes.append(p)
    s = sa.Solver.batch([(t, sa.make_box(20, 16), len(p)) for p in scenes])
    s.upload_batch(np.concatenate(scenes), counts)
    s.phase("hash")
    return s, np.concatenate(scenes), [(t, 0.0, 1.0, 0)] * len(counts)


@pytest.mark.parametrize("counts,spacing", [
    ([1], 0.5), ([15, 2], 0.5), ([16, 17, 1], 0.5), ([63, 65], 0.4), ([255, 257], 0.5),
    ([300], 3.0),    # nobody within h
    ([700], 0.12),   # 200 neighbours: many flushes of the edge buffer a group
])
def test_partial_groups(counts, spacing):
    s, state, meta = batch(counts, spacing)
    m = sa.Surrogate(seed=1)
    p = sr.random_params(31).astype(np.float32)
    m.params = p
    pd = device_weights(p)
    want, _, _ = oracle_batch(pd, state, counts, meta, 0)
    err = np.abs(m.predict(s).astype(np.float64) - want) / sr.DS
    scale = np.abs(want).max() / sr.DS
    assert err.max() <= 0.02 * (1 + scale), (err.max(), scale)
    rng = np.random.default_rng(7)
    target = (want + rng.normal(0, 0.02, want.shape)).astype(np.float32)
    _, g_ref, loss_ref = oracle_batch(pd, state, counts, meta, 0, target)
    m.zero_grads()
    loss = m.backward(s, target)
    g = m.grads().astype(np.float64)
    assert abs(loss - loss_ref) <= 0.05 * loss_ref, (loss, loss_ref)
    for name, a, b in (("W1", sr.oW1, sr.oW2), ("W2", sr.oW2, sr.ob2), ("b2", sr.ob2, sr.oW3),
                       ("W3", sr.oW3, sr.oW4), ("W4", sr.oW4, sr.ob4), ("b4", sr.ob4, sr.NPARAMS)):
        norm = np.linalg.norm(g_ref[a:b])
        if norm == 0:
            assert not g[a:b].any(), name
        else:
            rel = np.linalg.norm(g[a:b] - g_ref[a:b]) / norm
            assert rel <= 0.05, (name, rel)
    s.close()
