"""Where results may be fetched to: pageable memory, pinned memory (whole and
from the middle of an allocation) and device memory hold the same bytes, below
and above the size from which the pinned ring takes pageable ones."""
import numpy as np
import pytest
import torch

import sph_amd as sa
from sph_amd import scenes as sc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(64, 64), (400, 401), (701, 700)])
def test_pageable_pinned_and_device_memory(nx, ny):
    tun, box, parts = sc.dam_break(nx, ny, seed=nx)
    n = len(parts)
    s = sa.Solver(tun, box, n)
    s.upload(parts)
    s.step(3)
    m = sa.Surrogate(seed=2)
    L = sa.lib()
    calls = [("sph_download", 13 * n, lambda p: L.sph_download(s._h, p)),
             ("sph_download_positions", 2 * n, lambda p: L.sph_download_positions(s._h, p)),
             ("sph_pack_coords_i16", n, lambda p: L.sph_pack_coords_i16(s._h, p)),
             ("sph_surrogate_predict", 2 * n, lambda p: L.sph_surrogate_predict(m._h, s._h, p))]
    for name, words, call in calls:
        want = np.zeros(words, np.int32)
        assert call(want.ctypes.data) == 0
        pinned = torch.zeros(words + 12, dtype=torch.int32, pin_memory=True)
        device = torch.zeros(words, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        print(name, n, flush=True)
        for t, at in ((pinned, 0), (pinned, 4), (device, 0)):
            assert call(t.data_ptr() + 4 * at) == 0
            got = t.cpu().numpy()[at:at + words]
            same = got.tobytes() == want.tobytes()
            assert same, (name, t.device, at)
    s.close()
