"""The rasterizer's tiles against the oracle, bit for bit: triangle counts at the edges
of a wavefront's piece (21) and a workgroup's step (84), columns at and past
the hits kept between its phases (8), dexels without a triangle, grids cut by
the tiles, and grids past the tiles whose hits are kept."""

import numpy as np
import pytest

import oracle
from voroffset_amd import _native

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = _native.Context(0)
    yield c
    c.close()


def layers(n, seed, side=9.0):
    """n triangles over each other, in no order of height."""
    rng = np.random.default_rng(seed)
    V, F = [], []
    for i, z in enumerate(rng.permutation(n)):
        V += [(-side, -side, z), (3 * side, -side + 0.1, z + 0.25), (-side + 0.2, 3 * side, z + 0.5)]
        F.append((3 * i, 3 * i + 1, 3 * i + 2))
    return np.array(V, float).reshape(-1, 3), np.array(F, np.int32).reshape(-1, 3)


def check(ctx, V, F, nx, ny, ox, oy, s):
    want, got = oracle.rasterize(V, F, nx, ny, ox, oy, s), ctx.rasterize(V, F, nx, ny, ox, oy, s)
    assert np.array_equal(want[0], got[0]) and np.array_equal(want[1], got[1])
    return np.diff(got[0])


@pytest.mark.parametrize("n", [1, 7, 8, 9, 20, 21, 22, 83, 84, 85, 169])
def test_counts(ctx, n):
    V, F = layers(n, n)
    cols = check(ctx, V, F, 13, 19, -2.0, -3.0, 1.0)
    assert cols.max() == n


@pytest.mark.parametrize("n", [6, 40])
def test_scattered(ctx, n):
    """Small triangles everywhere: tiles of few and many, kept and swept again."""
    rng = np.random.default_rng(n)
    k = 60 * n
    centre = rng.uniform(0, 50, (k, 1, 3)) * [1, 0.6, 1]
    V = (centre + rng.uniform(-4, 4, (k, 3, 3))).reshape(-1, 3)
    F = np.arange(3 * k, dtype=np.int32).reshape(-1, 3)
    for nx, ny, s in ((50, 30, 1.0), (8, 8, 4.0), (1, 70, 0.5), (101, 61, 0.5)):
        check(ctx, V, F, nx, ny, 0.0, 0.0, s)


def test_more_tiles_than_keep_hits(ctx):
    V, F = layers(10, 3)
    check(ctx, V, F, 2056, 2048, -500.0, -500.0, 1.0)
    check(ctx, V, F, 2048, 2048, -500.0, -500.0, 1.0)
