"""The no-alloc entry point over the forms of the one-pass dilation: grids on
both sides of the 512 tiles up to which four wavefronts share one, sparse and
dense columns, lists past the room the scratch leaves them.  The results are
those of the allocating entry point, bit for bit, and a volume is refused only
where the two sweeps refuse it."""

import numpy as np
import pytest
import torch

from voroffset_amd import _native, synth

pytestmark = pytest.mark.gpu


def contexts():
    one = _native.Context(0)
    with pytest.MonkeyPatch.context() as m:
        m.setenv("VO_PASS1", "zsweep")
        two = _native.Context(0)
    return one, two


@pytest.mark.parametrize("prec,side", [("fp32", 100), ("fp32", 183), ("fp32", 200), ("fp64", 64), ("fp64", 130)])
@pytest.mark.parametrize("lam", [0.5, 3.0, 12.0])
@pytest.mark.parametrize("op,r", [("dilation", 1.0), ("dilation", 4.0), ("dilation", 6.5), ("dilation", 20.0),
                                  ("closing", 3.0)])
def test_same_as_allocating(prec, side, lam, op, r):
    vol = synth.poisson_columns(side, side - 3, lam=lam, zmax=700, mean_len=30.0, seed=side, z_margin=int(r) + 3)
    t = torch.float32 if prec == "fp32" else torch.float64
    off, z = torch.from_numpy(vol.off).cuda(), torch.from_numpy(vol.z).to(t).cuda()
    torch.cuda.synchronize()
    args = (op, prec, r, vol.nx, vol.ny, off.data_ptr(), z.data_ptr(), *vol.z_range())
    one, two = contexts()
    try:
        out, count, _ = one.morph_device(*args)
        want_off = _native.to_host(out.offsets, np.int64, out.nx * out.ny + 1)
        want = _native.to_host(out.z, np.float32 if prec == "fp32" else np.float64, count)

        def no_alloc(c):
            o_off = torch.zeros(vol.nx * vol.ny + 1, dtype=torch.int64, device="cuda")
            o_z = torch.zeros(count + 1, dtype=t, device="cuda")
            torch.cuda.synchronize()
            try:
                got, _ = c.morph_device_noalloc(*args, o_off.data_ptr(), o_z.data_ptr(), count + 1)
            except _native.VoError as e:
                assert e.code == _native.ERR_CAPACITY, str(e)
                return False
            assert got == count
            assert np.array_equal(o_off.cpu().numpy(), want_off)
            assert np.array_equal(o_z[:count].cpu().numpy(), want)
            return True

        # (what the two sweeps take in the scratch, the one-pass form takes)
        assert no_alloc(one) or not no_alloc(two)
    finally:
        one.close()
        two.close()
