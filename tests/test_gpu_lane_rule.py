"""Both sides of each line of the size rule for lanes per particle (sixteen up
to half a 256-slot tile per CU, four up to two, else one): the rule's choice
must give one lane's results bit for bit, viscosity, cap and all, in the first
steps and in a compressed state with cells cut by the cap."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cap", [0, 30])
@pytest.mark.parametrize("n", [1, 17, 32768, 32769, 131072, 131073])
def test_rule_matches_one_lane(n, cap):
    nx = max(1, int(np.sqrt(n)))
    tun, box, parts = sc.dam_break(nx, -(-n // nx), (nx * 1.2 + 3, nx * 0.8 + 3), seed=n)
    parts = parts[:n].copy()
    got = []
    for lanes in (0, 1):
        s = sa.Solver(tun, box, n)
        s.set_gather_lanes(lanes)
        s.set_bucket_cap(cap)
        s.upload(parts)
        s.step(3)
        early = s.download()
        s.step(90)
        got.append((early.tobytes(), s.download().tobytes(), s.counters()))
        s.close()
    assert got[0] == got[1]
