"""One network on contexts of different sizes.  Shadow judging's density buffers
must grow with the context: the larger context's states, flags and shadow
statistics after a smaller one's macro-steps must equal those after a larger
one's.  A prediction is not applied to a context larger than it covers."""
import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu


def batch(nx, ny, seed):
    t = sc.preset_tunables(0)
    parts = [sa.scene_lattice(nx, ny, 0.5, 0.01, seed=seed + k) for k in range(4)]
    s = sa.Solver.batch([(t, sa.make_box(nx * 1.1 + 4, ny * 1.0 + 4), len(p)) for p in parts])
    s.upload_batch(np.concatenate(parts), [len(p) for p in parts])
    s.step(5)
    return s


def macro_steps(first, steps):
    m = sa.Surrogate(seed=4)
    m.set_shadow(2)
    small = batch(*first, seed=50)
    for _ in range(4):
        m.macro_step(small, 0.05)
    assert m.shadow_stats()["shadowed"] > 0
    m.set_shadow(2)  # the statistics begin anew
    large = batch(90, 80, seed=60)
    flags = [m.macro_step(large, 0.05).tolist() for _ in range(steps)]
    st = m.shadow_stats()
    assert st["shadowed"] > 0
    out = large.download().tobytes(), flags, st
    small.close()
    large.close()
    return out


def test_network_goes_on_to_a_larger_context():
    a, b = macro_steps((12, 10), 6), macro_steps((90, 80), 6)
    assert a[1] == b[1] and a[2] == b[2]
    same = a[0] == b[0]
    assert same


def test_prediction_of_a_smaller_context_is_refused():
    m = sa.Surrogate(seed=4)
    small, large = batch(12, 10, seed=1), batch(90, 80, seed=2)
    m.predict(small)
    before = large.download()
    with pytest.raises(sa.SphError, match="smaller context"):
        m.apply(large)
    same = large.download().tobytes() == before.tobytes()
    assert same
    m.apply(small)  # the prediction is still there
    m.predict(large)
    m.apply(large)
    small.close()
    large.close()
