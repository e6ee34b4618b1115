"""Cone f32 backprojections, bit for bit against the oracle at odd sizes and around the
sources and heights where the LDS kernel gives way to the general one: 64x64, 57x97,
129x150, 90x192, 17x40 and 256x50 take the LDS kernel, with 16 slices per wave, the
others (and the angle that is not finite) the general one.  Every variant of the LDS
kernel is in test_cone_variants.py."""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu

# slices: around 64 and 128, 16 per wave; columns: odd, partial tiles; views: around
# the four of a group; sources: far and near; tall detectors, whose edge rows are read
CASES = [(64, 64, 9, 1000.0), (57, 97, 6, 300.0), (33, 129, 5, 44.0), (33, 130, 4, 30.0),
         (129, 150, 3, 400.0), (200, 70, 4, 600.0), (200, 61, 3, 250.0), (24, 600, 7, 60.0),
         (90, 192, 1, 150.0), (48, 65, 13, 52.0), (17, 40, 8, 200.0), (256, 50, 2, 900.0)]


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("W,H,n,sad", CASES)
def test_cone_bp_equals_oracle(gpu, W, H, n, sad, bad):
    print(f"cone bp W={W} H={H} n={n} sad={sad} bad={bad}", flush=True)
    r = np.random.Generator(np.random.PCG64(W + H))
    P = np.asfortranarray(r.uniform(-1, 1, (W, H, n)).astype(np.float32))
    ang = (np.arange(n) * (2 * np.pi / n) + 0.03).astype(np.float32)
    if bad:
        for v in (np.nan, np.inf, -np.inf):
            P[r.integers(0, W), r.integers(0, H), r.integers(0, n)] = v
        P[0, 0, 0], P[-1, -1, -1] = np.inf, np.nan
    got = mexct.CUDAmex_BP(P, sad, ang, 2)
    assert np.array_equal(got, O.bp(P, sad, ang, 2), equal_nan=True)


def test_cone_bp_angle_not_finite(gpu):
    W, H, n = 40, 70, 6
    P = np.asfortranarray(np.ones((W, H, n), np.float32))
    ang = (np.arange(n) * 1.0).astype(np.float32)
    ang[4] = np.nan
    got = mexct.CUDAmex_BP(P, 300.0, ang, 2)
    assert np.array_equal(np.isnan(got), np.isnan(O.bp(P, 300.0, ang, 2)))
