"""vo_last_stats: output endpoints, and the tiles whose lists outgrew their
room and were computed again."""

import numpy as np
import pytest

from voroffset_amd import _native
from voroffset_amd.volume import CompressedVolume

pytestmark = pytest.mark.gpu


def test_tiles_computed_again():
    ctx = _native.Context(0)
    try:
        def dilate(n):
            """One column of n separate segments in the second of three tiles."""
            cols = [[] for _ in range(24 * 8)]
            cols[24 * 3 + 11] = [float(4 * k + j) for k in range(n) for j in (0, 1)]
            vol = CompressedVolume.from_columns(24, 8, cols, origin=(0.0, 0.0, 0.0), extent=(24.0, 8.0, 4.0 * n))
            off, _, _ = ctx.morph_host("dilation", "fp64", 0.5, 24, 8, vol.off, vol.z, *vol.z_range())
            assert ctx.last_stats()[0] == off[-1] == 2 * n
            return ctx.last_stats()[1]

        assert dilate(24) == 0
        assert dilate(40) == 1      # 24, then 48
        assert dilate(40) == 0      # the room is kept
        assert dilate(90) == 1      # 48, then 96
        assert dilate(300) == 3     # 48, 96 and 192, then 384
    finally:
        ctx.close()
