"""The row filter on the matrix cores: widths around its tiles of 16 outputs, 4
inputs and 64 outputs per wave group, the widest and the first past it (direct
kernel), row counts around the 16 and 32 of a workgroup, and non-finite rows."""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu

CASES = [(2, 3, 3), (15, 16, 2), (16, 5, 3), (17, 17, 2), (63, 4, 4), (64, 3, 11), (65, 2, 8), (129, 3, 5),
         (191, 4, 4), (257, 3, 3), (301, 5, 7), (385, 2, 3), (449, 3, 2), (512, 2, 2), (513, 3, 2),
         (700, 2, 3), (768, 2, 2), (769, 2, 2), (20, 64, 300), (70, 57, 299)]


@pytest.mark.parametrize("W,H,n", CASES)
def test_filter_widths(gpu, W, H, n):
    print(f"filter W={W} H={H} n={n}", flush=True)
    r = np.random.Generator(np.random.PCG64(W * n))
    sino = np.asfortranarray(r.uniform(size=(W, H, n)).astype(np.float32))
    ang = (np.arange(n) * (np.pi / n)).astype(np.float32)
    got = mexct.preFilterSinogram(sino, {"type": "cone3d", "SAD": 4.0 * W}, ang, "hamming", 1.0)
    ref = O.prefilter(sino, "cone3d", 4.0 * W, ang, "hamming", 1.0)
    # one rounding of an FP64 sum to float, then two float operations: 2^-22 of
    # a value; the sums' own differences are of the order of 1e-13
    assert np.abs(got - ref).max() <= 1e-6 * np.abs(ref).max()


def test_filter_keeps_bad_rows_apart(gpu):
    W, H, n = 100, 21, 2
    r = np.random.Generator(np.random.PCG64(3))
    sino = np.asfortranarray(r.uniform(size=(W, H, n)).astype(np.float32))
    ang = np.array([0.0, 0.5], np.float32)
    good = mexct.preFilterSinogram(sino, {"type": "par3d"}, ang, "ramp", 1.0)
    sino[3, 4, 0], sino[99, 20, 1], sino[0, 0, 1] = np.nan, np.inf, -np.inf
    got = mexct.preFilterSinogram(sino, {"type": "par3d"}, ang, "ramp", 1.0)
    for v, k in ((4, 0), (20, 1), (0, 1)):
        assert not np.isfinite(got[:, v, k]).any()
        got[:, v, k] = good[:, v, k]
    assert np.array_equal(got, good)
