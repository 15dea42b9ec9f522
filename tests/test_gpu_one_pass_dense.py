"""The one-pass form on the volumes that the rule gives to the two sweeps:
asked for by name (VO_PASS1=direct) it gives what they give
(VO_PASS1=zsweep), bit for bit.  Small radii, dense columns, tiny and thin
grids, every number of wavefronts a tile, lists past their room."""

import numpy as np
import pytest

from voroffset_amd import _native
from voroffset_amd.volume import CompressedVolume

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def contexts():
    made = []
    for form in ("direct", "zsweep"):
        with pytest.MonkeyPatch.context() as m:
            m.setenv("VO_PASS1", form)
            made.append(_native.Context(0))
    yield made
    for c in made:
        c.close()


def volume(nx, ny, segments, seed, zext=500.0):
    rng = np.random.default_rng(seed)
    k = rng.poisson(segments, nx * ny)
    off = np.zeros(nx * ny + 1, np.int64)
    np.cumsum(2 * k, out=off[1:])
    col = np.repeat(np.arange(nx * ny), 2 * k)
    z = rng.integers(0, int(8 * zext), col.size)
    return CompressedVolume(nx, ny, off, z[np.lexsort((z, col))] / 8.0, origin=(0.0, 0.0, -10.0),
                            extent=(float(nx), float(ny), zext + 20.0), spacing=1.0, padding=0)


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
@pytest.mark.parametrize("nx,ny,segments",
                         [(nx, ny, k) for nx, ny in ((8, 8), (7, 13), (33, 41), (400, 1), (1, 400), (700, 2), (190, 180),
                                                     (270, 250))
                          for k in (3, 9, 25, 60) if nx * ny * k <= 700_000])
@pytest.mark.parametrize("r", [0.0, 0.9, 1.0, 1.9, 2.0, 2.9, 4.0, 5.5])
def test_as_the_sweeps(contexts, prec, nx, ny, segments, r):
    vol = volume(nx, ny, segments, segments)
    args = ("dilation", prec, r, nx, ny, vol.off, vol.z, *vol.z_range())
    a, b = [c.morph_host(*args)[:2] for c in contexts]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])


@pytest.mark.parametrize("op", ["erosion", "closing", "opening"])
@pytest.mark.parametrize("segments", [4, 20])
@pytest.mark.parametrize("r", [1.0, 2.0, 3.3])
def test_operations(contexts, op, segments, r):
    vol = volume(60, 45, segments, 7)
    args = (op, "fp32", r, 60, 45, vol.off, vol.z, *vol.z_range())
    a, b = [c.morph_host(*args)[:2] for c in contexts]
    assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
