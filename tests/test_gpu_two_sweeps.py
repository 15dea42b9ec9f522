"""The two sweeps asked for by name (VO_PASS1=zsweep): radii from 256 up, dense
columns at small radii and lists past the one-pass form's room take them by
themselves.  Their axis, their lists past their room, their tuning table and
their batched program, against the oracle and the default context."""

import numpy as np
import pytest

import oracle
from voroffset_amd import _native, synth
from voroffset_amd.volume import CompressedVolume

from .helpers import compare_csr, quantize_fp32

pytestmark = pytest.mark.gpu


@pytest.fixture
def sweeps(monkeypatch):
    """Contexts of the two sweeps, with more of the environment if given."""
    made = []

    def make(**env):
        with monkeypatch.context() as m:
            for k, v in dict(env, VO_PASS1="zsweep").items():
                m.setenv(k, v)
            made.append(_native.Context(0))
        return made[-1]

    yield make
    for c in made:
        c.close()


def check(got, ref, prec):
    bad, err = compare_csr(got[0], got[1], *ref)
    assert len(bad) == 0 and err <= (1e-9 if prec == "fp64" else 1e-4), (bad[:5], err)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("op", ["dilation", "erosion", "closing", "opening"])
def test_axis(sweeps, prec, op):
    vol = synth.poisson_columns(70, 45, lam=5, zmax=400, seed=17, z_margin=20)
    vol = vol if prec == "fp64" else quantize_fp32(vol)
    args = (op, prec, 6.5, vol.nx, vol.ny, vol.off, vol.z, *vol.z_range())
    x, y = [sweeps(VO_AXIS=a).morph_host(*args)[:2] for a in ("x", "y")]
    assert np.array_equal(x[0], y[0]) and np.array_equal(x[1], y[1])
    one = _native.Context(0)
    try:
        default = one.morph_host(*args)[:2]
    finally:
        one.close()
    assert np.array_equal(x[0], default[0]) and np.array_equal(x[1], default[1])


@pytest.mark.parametrize("r", [0.4, 0.9, 2.0])
def test_overfull_tiles(sweeps, r):
    cols = [[] for _ in range(70 * 3)]
    cols[5 + 70] = [float(k) for k in range(0, 160, 2)]  # 40 separate segments
    cols[66 + 140] = [float(k) for k in range(0, 90, 3)]
    vol = CompressedVolume.from_columns(70, 3, cols, origin=(0.0, 0.0, 0.0), extent=(70.0, 3.0, 200.0))
    got = sweeps().morph_host("dilation", "fp64", r, 70, 3, vol.off, vol.z, *vol.z_range())[:2]
    check(got, oracle.morph(vol, "dilation", r), "fp64")


def test_tuned_shapes_give_the_same(sweeps):
    vol = synth.poisson_columns(96, 80, lam=6, zmax=512, seed=21)
    ctx = sweeps()
    d_off, d_z = _native.DeviceArray(vol.off), _native.DeviceArray(vol.z)
    try:
        def result(r):
            v, n, _ = ctx.morph_device("dilation", "fp64", r, vol.nx, vol.ny, d_off.address, d_z.address, *vol.z_range())
            return _native.to_host(v.offsets, np.int64, vol.ncols + 1), _native.to_host(v.z, np.float64, n)

        radii = (3.0, 12.0, 20.0)
        before = [result(r) for r in radii]
        ctx.autotune("fp64", vol.nx, vol.ny, d_off.address, d_z.address, [3.0, 12.0, 20.0], reps=1)
        for a, b in zip(before, [result(r) for r in radii]):
            assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1])
    finally:
        d_off.free()
        d_z.free()


@pytest.mark.parametrize("prec", ["fp32", "fp64"])
def test_batched_program(sweeps, prec):
    """Every radius class (one, two and four coverage words) and operation, on
    three calls in a row (eager, captured, replayed)."""
    dt = np.float32 if prec == "fp32" else np.float64
    rng = np.random.default_rng(4)
    keep, jobs = [], []
    for k in range(12):
        r = float([rng.uniform(1.5, 31), rng.uniform(32, 63), rng.uniform(64, 127)][k % 3])
        vol = synth.poisson_columns(int(rng.integers(20, 90)), int(rng.integers(20, 90)), lam=float(rng.uniform(2, 6)),
                                    zmax=400, seed=70 + k, z_margin=int(r) + 4)
        d_off, d_z = _native.DeviceArray(vol.off), _native.DeviceArray(vol.z.astype(dt))
        keep += [d_off, d_z]
        jobs.append((synth.OPS[k % 4], r, vol.nx, vol.ny, d_off.address, d_z.address, *vol.z_range()))
    one = _native.Context(0)

    def results(ctx):
        outs, _ = ctx.morph_batch_device(prec, jobs)
        return [(_native.to_host(v.offsets, np.int64, v.nx * v.ny + 1), _native.to_host(v.z, dt, c)) for v, c in outs]

    try:
        want = results(one)
        ctx = sweeps()
        for call in range(3):
            got = results(ctx)
            assert ctx.last_batch_alone() == 0
            for k, (a, b) in enumerate(zip(want, got)):
                assert np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]), (call, k, jobs[k][:2])
    finally:
        for d in keep:
            d.free()
        one.close()
