"""Batches whose lists outgrow their room: the volumes are redone alone, the
next batch reserves more, and the estimate that admits jobs knows it; a single
volume redone with more room, or given up, leaves batches as they are.  And
batches of few tiles, which two wavefronts share, and of many, one each."""

import numpy as np
import pytest
import torch

from voroffset_amd import _native, serve, synth
from voroffset_amd.volume import CompressedVolume

pytestmark = pytest.mark.gpu


def layers(nx, ny, n, pitch=16.0):
    """n separate segments in every column."""
    z = (np.arange(n)[:, None] * pitch + np.array([0.0, 4.0])).ravel()
    off = np.arange(nx * ny + 1, dtype=np.int64) * 2 * n
    return CompressedVolume(nx, ny, off, np.tile(z, nx * ny), origin=(0.0, 0.0, -20.0),
                            extent=(float(nx), float(ny), n * pitch + 40.0), spacing=1.0, padding=0)


class Batch:
    def __init__(self, items, prec):
        self.prec, self.keep, self.jobs = prec, [], []
        for op, vol, r in items:
            t = torch.float32 if prec == "fp32" else torch.float64
            d = torch.from_numpy(vol.off).cuda(), torch.from_numpy(vol.z).to(t).cuda()
            self.keep.append(d)
            self.jobs.append((op, r, vol.nx, vol.ny, d[0].data_ptr(), d[1].data_ptr(), *vol.z_range()))
        torch.cuda.synchronize()

    def run(self, ctx):
        dt = np.float32 if self.prec == "fp32" else np.float64
        outs, _ = ctx.morph_batch_device(self.prec, self.jobs)
        return [(_native.to_host(v.offsets, np.int64, v.nx * v.ny + 1), _native.to_host(v.z, dt, c)) for v, c in outs]

    def alone(self, ctx):
        dt = np.float32 if self.prec == "fp32" else np.float64
        res = []
        for op, r, nx, ny, off, z, zlo, zhi in self.jobs:
            v, c, _ = ctx.morph_device(op, self.prec, r, nx, ny, off, z, zlo, zhi)
            res.append((_native.to_host(v.offsets, np.int64, nx * ny + 1), _native.to_host(v.z, dt, c)))
        return res


def equal(a, b):
    return all(np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1]) for x, y in zip(a, b))


def test_room_after_an_overflow():
    prec, side = "fp32", 200
    items = [("closing", layers(side, side, 30), 3.0) for _ in range(6)]
    batch = Batch(items, prec)
    other = _native.Context(0)
    free0 = torch.cuda.mem_get_info()[0]
    ctx = _native.Context(0)
    try:
        assert ctx.list_capacity() == 24
        want = batch.alone(other)
        assert equal(batch.run(ctx), want) and ctx.last_batch_alone() == len(items)
        assert ctx.list_capacity() == 48
        free0 -= free_of(other)
        assert equal(batch.run(ctx), want) and ctx.last_batch_alone() == 0
        used = free0 - torch.cuda.mem_get_info()[0]
        need = sum(serve.footprint_bytes(side * side, vol.z.size, op, 4, ocap=ctx.list_capacity()) for op, vol, _ in items)
        assert used <= need + (16 << 20), (used, need)
        assert equal(batch.run(ctx), want) and equal(batch.run(ctx), want)  # captured, replayed
    finally:
        ctx.close()
        other.close()


def free_of(ctx):
    """Device memory `ctx` holds."""
    before = torch.cuda.mem_get_info()[0]
    ctx.close()
    return torch.cuda.mem_get_info()[0] - before


def test_single_volumes_leave_batches_alone():
    ctx = _native.Context(0)
    try:
        for n in (30, 200, 700):  # redone with more room, and given up
            vol = layers(9, 9, n)
            zlo, zhi = vol.z_range()
            off, _, _ = ctx.morph_host("dilation", "fp64", 3.0, 9, 9, vol.off, vol.z, zlo, zhi)
            assert np.diff(off).max() == 2 * n
        assert ctx.list_capacity() == 24
    finally:
        ctx.close()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("volumes,side", [(3, 40), (6, 128), (7, 128), (4, 300)])
def test_shared_tiles(prec, volumes, side):
    """A launch of up to 1280 (FP64 1024) tiles has two wavefronts a tile."""
    ctx = _native.Context(0)
    try:
        for radii in ((2.0, 3.5), (4.0, 9.0), (10.0, 24.0)):
            items = [(synth.OPS[k % 4], synth.poisson_columns(side, side - k, lam=2.0 + k, zmax=400, seed=k, z_margin=30),
                      radii[0] + (radii[1] - radii[0]) * k / volumes) for k in range(volumes)]
            batch = Batch(items, prec)
            assert equal(batch.run(ctx), batch.alone(ctx))
    finally:
        ctx.close()
