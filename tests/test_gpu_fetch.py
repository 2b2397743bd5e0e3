"""Large results reach the caller's memory in pieces through pinned memory; they
must hold what the plain copies of the sorted fields hold.  Sizes just below and
at the least size of that path, at one, two and three halves of the pinned
memory and a little more, and with remainders of 4, 8 and 12 bytes; several
threads at once, each with its own context."""
import threading

import numpy as np
import pytest

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu

AOS = np.dtype(sa.PARTICLE).itemsize
MB = 1 << 20


def solver(n):
    nx = int(np.ceil(np.sqrt(n)))
    tun, box, parts = sc.dam_break(nx, -(-n // nx), (nx * 0.6 + 3, nx * 0.6 + 3), seed=n)
    parts = parts[:n].copy()
    s = sa.Solver(tun, box, n)
    s.upload(parts)
    s.step(2)
    return s


def check(s, rounds=2):
    n = s.n
    for _ in range(rounds):
        ids = s.read_sorted("id")
        x, y = s.read_sorted("x"), s.read_sorted("y")
        vx = s.read_sorted("v_x")
        xy, p = s.download_positions(), s.download()
        assert np.array_equal(xy[ids, 0], x) and np.array_equal(xy[ids, 1], y)
        assert np.array_equal(p["x"][ids], x) and np.array_equal(p["y"][ids], y)
        assert np.array_equal(p["v_x"][ids], vx)
        assert np.array_equal(p["id"], np.arange(n))
        s.step(1)
        q = s.pack_coords()
        assert q.shape == (n, 2) and np.array_equal(q, s.pack_coords())


@pytest.mark.parametrize("n", [MB // AOS, MB // AOS + 1, 2 * MB // AOS + 1, 4 * MB // AOS + 2,
                               6 * MB // AOS + 3, MB // 8 - 1, MB // 8, MB // 4, MB // 4 + 1,
                               MB // 2, MB // 2 + 1, 3 * MB // 4 + 5])
def test_sizes(n):
    s = solver(n)
    check(s)
    s.close()


def test_threads_with_their_own_contexts():
    solvers = [solver(150000 + 1001 * k) for k in range(4)]
    failed = []

    def run(s):
        try:
            check(s, rounds=4)
        except BaseException as e:  # noqa: BLE001
            failed.append(e)
    threads = [threading.Thread(target=run, args=(s,)) for s in solvers]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in solvers:
        s.close()
    assert not failed, failed
