"""The pair terms at the edges of their common form (sph_uncommon_pair).

A wave evaluates its pairs by cheap expressions valid for distances between
1e-6 and a little below h, and again by the whole ones when any lane holds a
pair outside that: coincident and nearly coincident particles (the 1e-6 nudge,
roots of tiny squares), pairs at the very edge of h, an impulse that is no
number.  Two particles at each such distance, among others at ordinary ones,
must follow the oracle's gather form bit for bit, with one and with four lanes
per particle.
"""
import numpy as np
import pytest

import sph_amd as sa
from oracle import pyoracle as po
from tests.common import assert_bitexact, dam_break_tunables

pytestmark = pytest.mark.gpu


def separations(h):
    f = np.float32
    h = f(h)
    edge = [f(h * (1 - 2.0 ** -k)) for k in (18, 19, 20, 21, 22)]
    return ([f(0), f(1e-30), f(2.0 ** -48), f(2.0 ** -49), f(9e-7), f(1e-6), f(1.1e-6), f(1.4e-6),
             f(0.5) * h, np.nextafter(h, f(0)), h, np.nextafter(h, f(9))] + edge)


@pytest.mark.parametrize("lanes", [1, 4])
@pytest.mark.parametrize("h", [1.0, 1.3])
def test_pairs_at_the_edges(h, lanes):
    for sep in separations(h):
        box = po.make_box(12 * h, 9 * h)
        t = dam_break_tunables(smoothing_radius=h, sigma=0.3, beta=0.2)
        p = np.zeros(70, po.P32)
        # the pair in the corner (where tiny distances are floats), then
        # ordinary company
        p["x"][1] = sep
        rng = np.random.default_rng(5)
        p["x"][2:] = rng.uniform(0.4 * h, 8 * h, 68).astype(np.float32)
        p["y"][2:] = rng.uniform(0.0, 4 * h, 68).astype(np.float32)
        p["v_x"] = rng.uniform(-1, 1, 70).astype(np.float32)
        p["v_x"][:2] = 0.0
        p["x_prev"], p["y_prev"], p["id"] = p["x"], p["y"], np.arange(70)
        s = sa.Solver(sa.Tunables.from_buffer_copy(bytes(t)), sa.AABB.from_buffer_copy(bytes(box)),
                      len(p))
        s.set_gather_lanes(lanes)
        s.upload(p)
        g = po.GatherSim(box, t, len(p))
        g.set_state(p)
        for step in (1, 2, 3):
            s.step(1)
            g.step(1)
            assert_bitexact(s.download(), g.get_state(), what=f"h {h}, sep {sep}, step {step}")
        s.close()


@pytest.mark.parametrize("lanes", [1, 4])
def test_impulse_that_is_no_number(lanes):
    """An impulse of inf * 0 passes the clamp as NaN, and a pair that moves
    apart adds nothing even then."""
    box = po.make_box(12, 9)
    t = dam_break_tunables(sigma=float(np.finfo(np.float32).max), beta=0.2)
    rng = np.random.default_rng(6)
    p = np.zeros(64, po.P32)
    p["x"] = rng.uniform(0.5, 6, 64).astype(np.float32)
    p["y"] = rng.uniform(0.5, 4, 64).astype(np.float32)
    p["v_x"] = rng.uniform(-5, 5, 64).astype(np.float32)
    p["x_prev"], p["y_prev"], p["id"] = p["x"], p["y"], np.arange(64)
    s = sa.Solver(sa.Tunables.from_buffer_copy(bytes(t)), sa.AABB.from_buffer_copy(bytes(box)), 64)
    s.set_gather_lanes(lanes)
    s.upload(p)
    g = po.GatherSim(box, t, 64)
    g.set_state(p)
    s.step(2)
    g.step(2)
    got, want = s.download(), g.get_state()
    for f in ("x", "y", "v_x", "v_y"):
        assert np.array_equal(np.isnan(got[f]), np.isnan(want[f])), f
        ok = ~np.isnan(want[f])
        assert np.array_equal(got[f][ok], want[f][ok]), f
