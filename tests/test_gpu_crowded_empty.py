"""Middle contexts with an empty scene: its tile holds no particle and has no
plan, whatever an earlier upload's sort left in its place.  The scene's padding
must be counted all the same, or the cell starts of the scenes after it shift,
and where it is the first scene its tile steps the sloshing clock.  Scenes whose
bottom tiles are crowded are stepped, one of them is uploaded again as empty,
and the size rule's results must equal one lane's bit for bit."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu


def crowded_at_the_bottom(seed):
    """4,900 particles of up to 200 candidates each (20 tiles a scene, fewer than
    the list holds) below 36,000 of 25."""
    low = sa.scene_lattice(70, 70, 0.2, 0.01, seed=seed)
    high = sa.scene_lattice(200, 180, 0.6, 0.01, seed=seed + 1, y0=16.0)
    p = np.concatenate([low, high])
    p["id"] = np.arange(len(p))
    return p


@pytest.mark.parametrize("cap", [0, 30])
@pytest.mark.parametrize("empty", [0, 1, 3])
def test_scene_uploaded_again_as_empty(empty, cap):
    tun, _, _ = sc.dam_break(1, 1)
    box = sa.make_box(140, 130)
    parts = [crowded_at_the_bottom(2 * k) for k in range(4)]
    left = [p[:0] if k == empty else p for k, p in enumerate(parts)]
    got = []
    for lanes in (0, 1):
        s = sa.Solver.batch([(tun, box, len(p)) for p in parts])
        s.set_gather_lanes(lanes)
        s.set_bucket_cap(cap)
        for k in range(4):
            s.set_scene_forcing(k, 2.0 + k, 0.5)
        out = []
        for scenes in (parts, left, parts):
            s.upload_batch(np.concatenate(scenes), [len(p) for p in scenes])
            for steps, graph in ((2, False), (3, True), (8, True)):
                s.step(steps, graph=graph)
                out.append(s.download().tobytes())
            out.append(s.counters())
        s.close()
        got.append(out)
    assert got[0] == got[1]
