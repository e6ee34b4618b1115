"""TV steps of thin volumes: no interior along an axis (no gradient anywhere), fewer rows
than a workgroup walks, and the rows at which the plan for large volumes takes over."""
import numpy as np
import pytest

import hip_log
import mexct
import oracle as O

SHAPES = [(1, 40, 60), (2, 41, 33), (40, 1, 60), (70, 2, 35), (64, 30, 1), (64, 30, 2), (100, 3, 40),
          (3, 3, 100), (1000, 11, 930), (1000, 12, 850)]


def test_large_volumes_of_few_rows():
    # 17 workgroups along x, one along y, and slices of 12 a workgroup from 12 rows on
    got = hip_log.record([dict(op="tv", N=[1000, ny, nz], steps=2) for ny, nz in ((12, 850), (11, 930))])
    grid = [next(k[1][0] for k in c["kernels"] if k[0].startswith("tv_step_kernel")) for c in got]
    assert grid[0] == 17 * 71 + 1 and grid[1] < 17 * 78


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_thin(gpu, shape):
    r = np.random.Generator(np.random.PCG64(sum(shape)))
    x = np.asfortranarray(r.uniform(0.01, 0.03, shape).astype(np.float32))
    ref = x
    for _ in range(2):
        g = O.tv_gradient(ref)
        with np.errstate(all="ignore"):  # a norm of 0 gives NaN, as the reference's does
            a = np.float32(-0.01) / np.float32(np.sqrt(np.sum(g.astype(np.float64) ** 2)))
            ref = (a * g + ref).astype(np.float32)
    got = mexct.CUDAmex_TVmin_3D(x, 0.01, steps=2)
    assert np.array_equal(got, ref, equal_nan=True)
    assert np.isnan(got).all() == (min(shape) < 3)


@pytest.mark.gpu
def test_thin_osc_tv(gpu):
    # the reconstruction's TV steps of a volume of two columns: NaN, which it zeroes
    r = np.random.Generator(np.random.PCG64(2))
    W, H, n = 2, 9, 6
    pre = np.asfortranarray(r.uniform(0.9e4, 1.1e4, (W, H, n)).astype(np.float32))
    post = np.asfortranarray((pre * r.uniform(0.5, 0.9, pre.shape)).astype(np.float32))
    ang = (np.arange(n) * 1.0).astype(np.float32)
    for geom in ("par3d", "cone3d"):
        got = mexct.OSC_TV_recon(pre, post, ang, {"type": geom, "SAD": 100.0}, 3, 0.1, 2, 1, 1.0,
                                 tv_steps=3, picks=np.ones(3, np.int32))
        assert np.array_equal(got, np.zeros((W, W, H), np.float32)), geom
