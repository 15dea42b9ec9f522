"""The chained scan's words are zero again for the next launch: many launches
in a row, over grids of different numbers of workgroups, most of whose columns
have nothing to copy, so that a workgroup's last act is publishing its sum."""

import numpy as np
import pytest
import torch

from voroffset_amd import _native

pytestmark = pytest.mark.gpu


def test_launches_in_a_row():
    ctx = _native.Context(0)
    vols = []
    for nx, ny, seed in ((600, 400, 1), (37, 29, 2), (1300, 700, 3), (512, 3, 4)):
        rng = np.random.default_rng(seed)
        off = np.zeros(nx * ny + 1, np.int64)
        off[1:] = np.cumsum(np.where(rng.random(nx * ny) < 0.001, 2, 0))
        z = np.tile([10.0, 20.0], off[-1] // 2 or 1)
        d = torch.from_numpy(off).cuda(), torch.from_numpy(z).float().cuda()
        vols.append((nx, ny, off, d))
    torch.cuda.synchronize()
    try:
        for k in range(150):
            nx, ny, off, (d_off, d_z) = vols[k % 4 if k % 3 else 2]
            out, count, _ = ctx.morph_device("dilation", "fp32", 0.0, nx, ny, d_off.data_ptr(), d_z.data_ptr(), 0.0, 100.0)
            assert count == off[-1], (k, nx, ny)
            got = _native.to_host(out.offsets, np.int64, nx * ny + 1)
            assert np.array_equal(got, off), (k, nx, ny)
    finally:
        ctx.close()
