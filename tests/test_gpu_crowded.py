"""Middle contexts: four lanes per particle walk the crowded tiles that the
planner lists.  The rule's choice must leave what one lane per particle leaves,
bit for bit: at both ends of the sizes that list, where no tile, some tiles or
more tiles than the list holds are crowded, with the cap, between the callers
that make plans, and in a batch."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu


def state(s):
    out = []
    s.step(3)
    s.snapshot_save()
    out.append(s.download())
    s.step(40)
    out.append(s.download())
    s.phase("hash_density")
    s.phase("relax")
    s.step(2)
    out.append(s.download())
    s.snapshot_restore(np.ones(s.nscenes, np.int32))
    s.phase("viscosity")
    s.step(5, graph=False)
    out.append(s.download())
    return [a.tobytes() for a in out] + [s.counters()]


def both(make, cap):
    got = []
    for lanes in (0, 1):
        s = make()
        s.set_gather_lanes(lanes)
        s.set_bucket_cap(cap)
        got.append(state(s))
        s.close()
    assert got[0] == got[1]


@pytest.mark.parametrize("cap", [0, 30])
@pytest.mark.parametrize("n,spacing", [(131073, 0.5), (200000, 0.5), (262144, 0.5), (262145, 0.5),
                                       (140000, 0.2), (262144, 0.25), (150001, 0.9)])
def test_rule_matches_one_lane(n, spacing, cap):
    def make():
        nx = int(np.sqrt(n)) + 1
        tun, _, _ = sc.dam_break(1, 1)
        box = sa.make_box(nx * spacing * 2.3, nx * spacing * 1.6)
        parts = sa.scene_lattice(nx, -(-n // nx), spacing, 0.01, seed=n)[:n].copy()
        s = sa.Solver(tun, box, n)
        s.upload(parts)
        return s
    both(make, cap)


def test_batch_with_crowded_and_sparse_scenes():
    tun, _, _ = sc.dam_break(1, 1)
    scenes = [(sa.make_box(70, 60), sa.scene_lattice(200, 150, 0.2, 0.01, seed=1)),
              (sa.make_box(260, 200), sa.scene_lattice(300, 301, 0.6, 0.01, seed=2)),
              (sa.make_box(60, 50), sa.scene_lattice(77, 130, 0.3, 0.01, seed=3))]

    def make():
        s = sa.Solver.batch([(tun, b, len(p) + 300) for b, p in scenes])
        s.upload_batch(np.concatenate([p for _, p in scenes]), [len(p) for _, p in scenes])
        return s
    both(make, 0)
