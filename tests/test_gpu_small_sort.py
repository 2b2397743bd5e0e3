"""The small contexts' one-launch sort: the same states, cells and counters, bit
for bit, as with one lane per particle, whose sort scans, scatters and
reorders.  Grids end just below, at and just above each of its sizes of counts
(2,048 to 32,768, above which the other sort runs); cells hold more members than
their lists' rows; a batch ends in an empty scene."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu


def state(s, parts, counts=None):
    """A run that changes between the sorts' callers, and what it leaves."""
    out = []
    if counts is None:
        s.upload(parts)
    else:
        s.upload_batch(parts, counts)
    s.step(3)
    s.snapshot_save()
    s.step(20)
    out.append(s.download())
    for name in ("viscosity", "gravity", "predict", "hash_density", "relax", "update_velocities"):
        s.phase(name)
    s.step(2)
    out.append(s.download())
    s.snapshot_restore(np.ones(s.nscenes, np.int32))
    s.phase("viscosity")
    s.step(9, graph=False)
    out += [s.download(), s.read_sorted("id"), s.read_sorted("key")]
    return [a.tobytes() for a in out] + [a.tobytes() for a in s.cells()[:2]] + [s.counters()]


def both(make, parts, counts=None):
    got = []
    for lanes in (0, 1):
        s = make()
        s.set_gather_lanes(lanes)
        got.append(state(s, parts, counts))
        s.close()
    assert got[0] == got[1]


# columns x rows + padding cell + the end: the counts
@pytest.mark.parametrize("cols,rows", [(1, 1), (2045, 1), (2046, 1), (2047, 1), (62, 66), (63, 65),
                                       (89, 92), (91, 90), (8191, 2), (127, 129), (169, 193),
                                       (182, 180), (258, 127), (173, 190)])
def test_grid_sizes(cols, rows):
    tun, _, _ = sc.dam_break(1, 1)
    h = tun.smoothing_radius
    box = sa.make_box((cols - 0.5) * h, (rows - 0.5) * h)
    rng = np.random.default_rng(cols)
    parts = sa.scene_lattice(37, 31, 0.4 * h, 0.01, seed=cols)
    parts["x"] = np.minimum(parts["x"], box.max_x)
    parts["y"] = np.minimum(parts["y"], box.max_y * rng.uniform(0.9, 1.0, len(parts)))
    both(lambda: sa.Solver(tun, box, len(parts)), parts)


@pytest.mark.parametrize("n", [127, 128, 129, 700])
def test_cells_past_their_lists(n):
    """n members in each of three neighbouring cells and one far from them."""
    tun, box, _ = sc.dam_break(1, 1, (40, 30))
    h = tun.smoothing_radius
    rng = np.random.default_rng(n)
    parts = np.zeros(4 * n, sa.PARTICLE)
    cell = rng.permutation(np.repeat([7, 8, 9, 25], n))
    parts["x"] = (cell + rng.uniform(0.05, 0.95, 4 * n)) * h
    parts["y"] = (3 + rng.uniform(0.05, 0.95, 4 * n)) * h
    parts["id"] = np.arange(4 * n)
    both(lambda: sa.Solver(tun, box, len(parts)), parts)


def test_batch_with_an_empty_scene():
    scenes = [sc.dam_break(nx, 20, (30 + nx, 25), seed=nx) for nx in (1, 13, 40)]
    scenes.append((scenes[0][0], scenes[0][1], scenes[0][2][:0]))
    parts = np.concatenate([p for _, _, p in scenes])
    both(lambda: sa.Solver.batch([(t, b, max(1, len(p))) for t, b, p in scenes]), parts,
         [len(p) for _, _, p in scenes])
