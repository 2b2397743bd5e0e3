"""Calls that find no device memory: they say so, and the context goes on as it
was.  sph_set_gather_lanes keeps the shape that the context had; a snapshot that
found no memory may be saved later.  The allocations fail in a process of their
own, whose library finds a hipMalloc that can be told to."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

HIPMALLOC = r"""
#include <stddef.h>
static int (*real)(void **, size_t);
static int left = -1; /* calls until one fails; below 0: none does */
void set_real(void *f) { real = (int (*)(void **, size_t))f; }
void fail_after(int calls) { left = calls; }
int armed(void) { return left >= 0; }
int hipMalloc(void **p, size_t bytes)
{
    if (left >= 0 && left-- == 0)
        return 2; /* hipErrorOutOfMemory */
    return real(p, bytes);
}
"""

HOOK = r"""
import ctypes, sys
mem = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
hip = ctypes.CDLL("/opt/rocm/lib/libamdhip64.so")
mem.set_real(ctypes.cast(hip.hipMalloc, ctypes.c_void_p))
import sph_amd as sa
from sph_amd import scenes as sc
import numpy as np

def refused(call, calls):
    mem.fail_after(calls)
    try:
        call()
        raise SystemExit("no error")
    except sa.SphError as e:
        assert "hipMalloc" in str(e), e
    assert not mem.armed()
"""

LANES = HOOK + r"""
nx, ny, before, wanted, calls = map(int, sys.argv[2:])
tun, box, parts = sc.dam_break(nx, ny, seed=3)
got = []
for fails in (False, True):
    s = sa.Solver(tun, box, len(parts))
    s.set_gather_lanes(before)
    s.upload(parts)
    s.step(20)
    if fails:
        refused(lambda: s.set_gather_lanes(wanted), calls)
    s.step(3, graph=False)
    s.step(20)
    s.phase("hash_density")
    got.append([s.download().tobytes(), s.counters()])
    if fails:
        s.set_gather_lanes(wanted)
    s.step(20)
    got[-1].append(s.download().tobytes())
    s.close()
assert got[0] == got[1]
print("as before")
"""

SNAPSHOT = HOOK + r"""
for calls in range(9):
    tun, box, parts = sc.dam_break(70, 61, seed=calls)
    s = sa.Solver(tun, box, len(parts))
    s.upload(parts)
    s.step(7)
    refused(s.snapshot_save, calls)
    s.snapshot_save()
    want = s.download().tobytes()
    s.step(5)
    assert s.download().tobytes() != want
    s.snapshot_restore(np.ones(1, np.int32))
    assert s.download().tobytes() == want
    s.close()
print("as before")
"""


@pytest.fixture(scope="module")
def library(tmp_path_factory):
    d = tmp_path_factory.mktemp("hipmalloc")
    (d / "m.c").write_text(HIPMALLOC)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(d / "m.so"), str(d / "m.c")], check=True)
    return str(d / "m.so")


def run(library, code, *args):
    cmd = [sys.executable, "-c", code, library, *map(str, args)]
    r = subprocess.run(cmd, cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "as before" in r.stdout, r.stdout + r.stderr


@pytest.mark.parametrize("nx,ny,before,wanted,calls", [
    (64, 64, 1, 4, 0),    # the four-lane gathers' plans
    (64, 64, 0, 4, 0),    # ... after sixteen lanes
    (400, 400, 1, 0, 0),  # a middle context's plans,
    (400, 400, 1, 0, 1),  # its list's length
    (400, 400, 1, 0, 2),  # and its list
])
def test_lanes_keep_their_shape(library, nx, ny, before, wanted, calls):
    run(library, LANES, nx, ny, before, wanted, calls)


def test_snapshot_is_saved_later(library):
    run(library, SNAPSHOT)
