"""Calls that fail, and the ones after them.  The input check of a resident
volume goes along with its one-pass dilation, whose kernels have to stay
within their memory on any endpoints its offsets index; and a call that fails
leaves nothing behind that a later one takes for its own."""

import numpy as np
import pytest
import torch

import oracle
from voroffset_amd import _native, synth

from .helpers import compare_csr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = _native.Context(0)
    yield c
    c.close()


def resident(off, z, prec):
    t = torch.float32 if prec == "fp32" else torch.float64
    d = torch.from_numpy(np.asarray(off, np.int64)).cuda(), torch.from_numpy(np.asarray(z)).to(t).cuda()
    torch.cuda.synchronize()
    return d


def no_alloc(ctx, op, prec, r, nx, ny, off, z, zlo, zhi, guard=4096):
    """The no-alloc call; returns offsets and endpoints, and looks at the words past
    the output buffers."""
    cap = 32 * nx * ny
    o_off = torch.full((nx * ny + 1 + guard,), -7, dtype=torch.int64, device="cuda")
    o_z = torch.full((cap + guard,), -7.0, dtype=z.dtype, device="cuda")
    torch.cuda.synchronize()
    try:
        count, _ = ctx.morph_device_noalloc(op, prec, r, nx, ny, off.data_ptr(), z.data_ptr(), zlo, zhi, o_off.data_ptr(),
                                            o_z.data_ptr(), cap)
    finally:
        torch.cuda.synchronize()
        assert bool((o_off[nx * ny + 1:] == -7).all()) and bool((o_z[cap:] == -7.0).all())
    return o_off[:nx * ny + 1].cpu().numpy(), o_z[:count].cpu().numpy()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("r", [2.5, 6.5, 12.0])
@pytest.mark.parametrize("entry", ["resident", "no_alloc"])
def test_unsorted_columns(ctx, prec, r, entry):
    """Many segments with their ends exchanged and in no order: 64 x 64
    columns, four wavefronts a tile, lists of 12 in the no-alloc scratch."""
    nx = ny = 64
    rng = np.random.default_rng(int(10 * r))
    k = 14
    off = np.arange(nx * ny + 1, dtype=np.int64) * 2 * k
    z = np.round(rng.uniform(0.0, 4000.0, 2 * k * nx * ny))
    d_off, d_z = resident(off, z, prec)
    with pytest.raises(_native.VoError) as e:
        if entry == "resident":
            ctx.morph_device("dilation", prec, r, nx, ny, d_off.data_ptr(), d_z.data_ptr(), 0.0, 4000.0)
        else:
            no_alloc(ctx, "dilation", prec, r, nx, ny, d_off, d_z, 0.0, 4000.0)
    assert e.value.code == _native.ERR_ARGUMENT, str(e.value)
    # the context, and the scratch, still work
    vol = synth.poisson_columns(24, 20, lam=4, zmax=400, seed=3, z_margin=20)
    d_off, d_z = resident(vol.off, vol.z, prec)
    got = no_alloc(ctx, "dilation", prec, r, vol.nx, vol.ny, d_off, d_z, *vol.z_range())
    seen = vol.like(vol.off, d_z.cpu().numpy().astype(np.float64))
    bad, err = compare_csr(got[0], got[1].astype(np.float64), *oracle.morph(seen, "dilation", r))
    assert len(bad) == 0 and err <= (1e-9 if prec == "fp64" else 1e-4)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("r", [6.5, 12.0, 40.0])
@pytest.mark.parametrize("side", [24, 200])
def test_non_finite_endpoints(ctx, prec, value, r, side):
    """Endpoints that are not numbers, among them first and last ones: waiting
    segments without an order of their own."""
    rng = np.random.default_rng(side)
    k = 5
    off = np.arange(side * side + 1, dtype=np.int64) * 2 * k
    z = np.sort(np.round(rng.uniform(0.0, 900.0, (side * side, 2 * k)), 2), axis=1).ravel()
    z[rng.integers(0, z.size, z.size // 7)] = value
    d_off, d_z = resident(off, z, prec)
    with pytest.raises(_native.VoError) as e:
        ctx.morph_device("dilation", prec, r, side, side, d_off.data_ptr(), d_z.data_ptr(), 0.0, 900.0)
    assert e.value.code == _native.ERR_ARGUMENT, str(e.value)


@pytest.mark.parametrize("form", ["one pass", "two sweeps"])
def test_growth_table_after_a_failure(monkeypatch, form):
    """A call fails (injected) where its larger radius has the context give
    the growth table's memory back for more; the earlier radius follows."""
    monkeypatch.setenv("VO_INJECT_HIP_ERROR", "hipFree")
    if form == "two sweeps":
        monkeypatch.setenv("VO_PASS1", "zsweep")
    c = _native.Context(0)
    monkeypatch.undo()
    nx, ny = 3, 2  # (few enough endpoints that no other buffer grows)
    off, z = [0, 2, 2, 2, 2, 2, 2], np.array([10.0, 20.0])
    d_off, d_z = resident(off, z, "fp64")

    def dilated(r):
        out, count, _ = c.morph_device("dilation", "fp64", r, nx, ny, d_off.data_ptr(), d_z.data_ptr(), 0.0, 100.0)
        return _native.to_host(out.z, np.float64, count).reshape(-1, 2)

    try:
        want = [[10.0 - h, 20.0 + h] for y in range(ny) for x in range(nx) for h in [np.sqrt(4.5 * 4.5 - x * x - y * y)]]
        assert np.array_equal(dilated(4.5), want)
        for _ in range(3):
            with pytest.raises(_native.VoError) as e:
                dilated(30.5)
            assert e.value.code == _native.ERR_DEVICE and "injected" in str(e.value)
            assert np.array_equal(dilated(4.5), want)
    finally:
        c.close()
