"""The one-pass form of a dilation (the default up to R = 255) against the two
sweeps (VO_PASS1=zsweep), bit for bit, and against the oracle: tiles of 8 x 8
columns cut by the grid, radii at the edges of its variants, lists past their
LDS entries and past their first room, columns of more segments than its
summaries count, empty and touching columns."""

import os

import numpy as np
import pytest
import torch

import oracle
from voroffset_amd import _native, synth
from voroffset_amd.volume import CompressedVolume

from .helpers import compare_csr

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def contexts():
    one = _native.Context(0)
    old = os.environ.get("VO_PASS1")
    os.environ["VO_PASS1"] = "zsweep"
    try:
        two = _native.Context(0)
    finally:
        if old is None:
            del os.environ["VO_PASS1"]
        else:
            os.environ["VO_PASS1"] = old
    yield one, two
    one.close()
    two.close()


def both(contexts, vol, op, prec, r):
    zlo, zhi = vol.z_range()
    res = [c.morph_host(op, prec, r, vol.nx, vol.ny, vol.off, vol.z, zlo, zhi)[:2] for c in contexts]
    assert np.array_equal(res[0][0], res[1][0])
    assert np.array_equal(res[0][1], res[1][1])
    return res[0]


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("nx,ny", [(1, 1), (7, 9), (8, 8), (65, 3), (3, 70), (129, 41)])
@pytest.mark.parametrize("r", [0.0, 0.9, 3.0, 5.0, 7.9, 8.0, 12.3, 31.5, 32.0, 64.0])
def test_grids_and_radii(contexts, prec, nx, ny, r):
    vol = synth.poisson_columns(nx, ny, lam=4, zmax=500, seed=nx + 7 * ny, z_margin=int(r) + 3)
    off, z = both(contexts, vol, "dilation", prec, r)
    if prec == "fp64" and nx * ny <= 300:
        bad, err = compare_csr(off, z, *oracle.morph(vol, "dilation", r))
        assert len(bad) == 0 and err <= 1e-9


@pytest.mark.parametrize("op", ["erosion", "closing", "opening"])
@pytest.mark.parametrize("r", [2.5, 9.0])
def test_solids(contexts, op, r):
    vol = synth.ball_union(9, 60, seed=int(r), rmin=5.0, rmax=14.0, pad=14)
    for prec in ("fp32", "fp64"):
        both(contexts, vol, op, prec, r)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("r", [2.0, 5.5, 20.0, 40.0])
def test_one_wavefront_per_tile(contexts, prec, r):
    """More tiles than share wavefronts (512): one wavefront each."""
    vol = synth.poisson_columns(233, 150, lam=5, zmax=600, seed=int(r), z_margin=int(r) + 3)
    both(contexts, vol, "dilation", prec, r)


@pytest.mark.parametrize("r", [100.0, 255.0])
def test_large_radii(contexts, r):
    vol = synth.poisson_columns(300, 20, lam=1.0, mean_len=15.0, zmax=3000, seed=11)
    both(contexts, vol, "dilation", "fp32", r)


def column_volume(nx, ny, columns, zext):
    cols = [columns.get(i, []) for i in range(nx * ny)]
    return CompressedVolume.from_columns(nx, ny, cols, origin=(0.0, 0.0, 0.0), extent=(float(nx), float(ny), zext))


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("n", [3, 4, 8, 9, 24, 25, 200, 600])
def test_many_intervals(contexts, prec, n):
    """Columns keeping n separate intervals: within the LDS entries, past
    them, past the first room (the tile is done again with more), and past what the
    form takes (the sweeps do the volume)."""
    vol = column_volume(20, 11, {25: [float(4 * k + j) for k in range(n) for j in (0, 1)],
                                 97: [4.0 * k + 0.5 + j for k in range(n) for j in (0, 0.25)]}, 4.0 * n)
    for r in (0.5, 1.2):
        off, z = both(contexts, vol, "dilation", prec, r)
        assert np.diff(off).max() == 2 * n
    both(contexts, vol, "dilation", prec, 9.0)


def test_column_of_many_segments(contexts):
    """More segments in a column than its summary word counts: 70,000 thin
    ones that the dilation fuses."""
    n = 70000
    z = np.arange(2 * n, dtype=np.float64) * 0.5
    vol = column_volume(9, 3, {4: z.tolist(), 13: [100.0, 40000.0]}, n + 10.0)
    zlo, zhi = vol.z_range()
    off, got, _ = contexts[0].morph_host("dilation", "fp64", 2.5, vol.nx, vol.ny, vol.off, vol.z, zlo, zhi)
    for c, (dx, dy) in {4: (0, 0), 3: (1, 0), 6: (2, 0), 22: (0, 2)}.items():
        h = np.sqrt(6.25 - dx * dx - dy * dy)
        assert got[off[c]:off[c + 1]].tolist() == [0.0 - h, z[-1] + h]


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_points_and_touching_segments(contexts, prec):
    rng = np.random.default_rng(5)
    cols = {}
    for c in range(23 * 17):
        v = np.sort(rng.integers(0, 120, 2 * int(rng.integers(0, 6)))) / 4.0
        cols[c] = v.tolist()
    vol = column_volume(23, 17, cols, 40.0)
    for r in (1.0, 2.5, 5.0, 13.0):
        both(contexts, vol, "dilation", prec, r)


def on_device(ctx, vol, op, prec, r):
    """The call on a volume whose size only the device knows."""
    t = torch.float32 if prec == "fp32" else torch.float64
    off, z = torch.from_numpy(vol.off).cuda(), torch.from_numpy(vol.z).to(t).cuda()
    if z.numel() == 0:
        z = torch.zeros(1, dtype=t, device="cuda")
    torch.cuda.synchronize()
    out, count, _ = ctx.morph_device(op, prec, r, vol.nx, vol.ny, off.data_ptr(), z.data_ptr(), *vol.z_range())
    got_off = torch.zeros(out.nx * out.ny + 1, dtype=torch.int64, device="cuda")
    got = torch.zeros(max(count, 1), dtype=t, device="cuda")
    copies = [(got_off.data_ptr(), out.offsets, got_off.numel() * 8)]
    if count:
        copies.append((got.data_ptr(), out.z, count * got.element_size()))
    torch.cuda.synchronize()
    ctx.copy_device(copies)
    return got_off.cpu().numpy(), got[:count].cpu().numpy()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("lam", [1.0, 4.0])
@pytest.mark.parametrize("op,r", [("dilation", 2.5), ("dilation", 9.9), ("dilation", 15.5), ("dilation", 16.0),
                                  ("closing", 2.5), ("closing", 10.0), ("erosion", 3.5), ("opening", 3.0)])
def test_shared_tiles_of_sparse_volumes(contexts, prec, lam, op, r):
    """More than 512 tiles, few and many segments a column: known to the host
    (from host memory) or only to the device, and in a complement."""
    vol = synth.poisson_columns(233, 150, lam=lam, mean_len=60.0, zmax=600, seed=int(10 * r), z_margin=int(r) + 3)
    both(contexts, vol, op, prec, r)
    one, two = [on_device(c, vol, op, prec, r) for c in contexts]
    assert np.array_equal(one[0], two[0]) and np.array_equal(one[1], two[1])


@pytest.mark.parametrize("nx,ny", [(1, 511), (512, 1), (19, 27), (512, 256), (131073, 1), (683, 769)])
@pytest.mark.parametrize("op", ["dilation", "erosion"])
def test_offsets_of_one_launch(contexts, nx, ny, op):
    """Grids at the edges of a workgroup's columns (512 or 2048) and of the
    rule between the two; small and large results in turn, so that the output
    is once too small for the launch; empty columns and an empty result."""
    for lam in (0.0, 3.0, 0.2, 6.0):
        vol = synth.poisson_columns(nx, ny, lam=lam, zmax=200, mean_len=30.0, seed=3, z_margin=8)
        one, two = [on_device(c, vol, op, "fp32", 1.5) for c in contexts]
        assert np.array_equal(one[0], two[0]) and np.array_equal(one[1], two[1])
