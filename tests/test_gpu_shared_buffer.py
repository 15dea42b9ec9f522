"""Resident volumes whose offsets do not begin at 0: one volume of many that
share an endpoint buffer.  Results begin at 0, and what a call reserves goes by
the volume's own endpoints, wherever they lie."""

import numpy as np
import pytest
import torch

from voroffset_amd import _native, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [0, 1 << 20, 10 ** 11])
@pytest.mark.parametrize("form", ["one pass", "two sweeps"])
@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("op,r", [("dilation", 1.5), ("dilation", 7.0), ("erosion", 2.0), ("closing", 3.0), ("opening", 2.0)])
def test_offsets_begin_anywhere(monkeypatch, first, form, prec, op, r):
    if form == "two sweeps":
        monkeypatch.setenv("VO_PASS1", "zsweep")
    ctx = _native.Context(0)
    monkeypatch.undo()
    vol = synth.poisson_columns(53, 38, lam=5, zmax=300, seed=8, z_margin=12)
    t, dt = (torch.float32, np.float32) if prec == "fp32" else (torch.float64, np.float64)
    z = torch.from_numpy(vol.z).to(t).cuda()
    off, moved = torch.from_numpy(vol.off).cuda(), torch.from_numpy(vol.off + first).cuda()
    torch.cuda.synchronize()

    def result(o, base):
        v, n, _ = ctx.morph_device(op, prec, r, vol.nx, vol.ny, o.data_ptr(), base, *vol.z_range())
        return _native.to_host(v.offsets, np.int64, v.nx * v.ny + 1), _native.to_host(v.z, dt, n)

    try:
        want = result(off, z.data_ptr())
        free = torch.cuda.mem_get_info()[0]
        got = result(moved, z.data_ptr() - first * z.element_size())  # (the buffer it shares begins that far before)
        assert got[0][0] == 0 and np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])
        assert free - torch.cuda.mem_get_info()[0] < 64 << 20
    finally:
        ctx.close()
