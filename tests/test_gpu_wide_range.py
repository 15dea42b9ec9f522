"""FP64 endpoints that no float holds.  The one-pass dilation keeps covers as
floats rounded to the safe side: past the largest float, and below the
smallest, they still claim no more than the lists hold.  Results equal those
of the two sweeps, which look at doubles only, and the oracle's."""

import numpy as np
import pytest

import oracle
from voroffset_amd import _native
from voroffset_amd.volume import CompressedVolume

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def contexts():
    one = _native.Context(0)
    with pytest.MonkeyPatch.context() as m:
        m.setenv("VO_PASS1", "zsweep")
        two = _native.Context(0)
    yield one, two
    one.close()
    two.close()


@pytest.mark.parametrize("scale", [1e-46, 1e-41, 1.0, 1e35, 2e37, 1e38, 1e39, 1e200])
@pytest.mark.parametrize("nx,ny", [(5, 3), (13, 11), (40, 24), (233, 150)])
@pytest.mark.parametrize("r", [0.0, 5.0, 13.0])
def test_covers_at_any_scale(contexts, scale, nx, ny, r):
    rng = np.random.default_rng(nx + int(r))
    cols = []
    for c in range(nx * ny):
        # around zero, and growing away from the first columns, so that later ones stick out
        v = np.sort(rng.uniform(-5.0, 5.0, 2 * int(rng.integers(0, 4)))) * (1.0 + c / (nx * ny))
        cols.append((v * scale).tolist())
    vol = CompressedVolume.from_columns(nx, ny, cols, origin=(0.0, 0.0, -20.0 * scale),
                                        extent=(float(nx), float(ny), 40.0 * scale))
    got = [c.morph_host("dilation", "fp64", r, nx, ny, vol.off, vol.z, *vol.z_range())[:2] for c in contexts]
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    if nx * ny < 1000 and scale >= 1.0:  # (the oracle joins what is nearer than 1e-10, as the reference does)
        off, z = oracle.morph(vol, "dilation", r)
        assert np.array_equal(got[0][0], off)
        assert np.allclose(got[0][1], z, rtol=1e-12, atol=1e-9)
