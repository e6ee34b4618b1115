"""The range of voxel values in which the TV step takes its fast square root and
division: the oracle's bits at both ends, on both sides of each, and where values
of both ends meet in one stencil."""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu


def _step(x, c):
    """One step from the oracle's float gradient, with a norm summed in FP64."""
    g = O.tv_gradient(x)
    with np.errstate(all="ignore"):
        a = np.float32(-c) / np.float32(np.sqrt(np.sum(g.astype(np.float64) ** 2)))
        return (a * g + x).astype(np.float32)


def test_quotient_below_the_normal_range(gpu):
    # neighbours 9 2^-94 apart beside one of 3 2^56: a quotient of 1.5 of the least
    # subnormal, half way between two floats
    x = np.full((6, 6, 6), np.float32(2.0 ** -76), np.float32)
    x[3, 2, 2] = np.float32(2.0 ** -76 + 9 * 2.0 ** -94)
    x[3, 1, 2] = np.float32(3 * 2.0 ** 56)
    x = np.asfortranarray(x)
    got = mexct.CUDAmex_TVmin_3D(x, 2.0 ** 100, steps=1)
    assert np.array_equal(got, _step(x, 2.0 ** 100))


@pytest.mark.parametrize("lo,hi", [(-76, -75), (-78, -74), (20, 22), (21, 24), (-76, 22), (-80, 26),
                                   (-100, -99), (57, 59), (-40, 0)])
def test_values_at_the_ends(gpu, lo, hi):
    # magnitudes of 2^lo .. 2^hi, either sign, zeros and flat parts among them, in
    # blocks of a few voxels, so that whole waves and parts of them are in range
    r = np.random.Generator(np.random.PCG64(hi - lo + 200))
    shape = (70, 24, 13)
    v = np.ldexp(r.uniform(1, 2, shape), r.integers(lo, hi, shape)) * r.choice([-1, 0, 1, 1], shape)
    v[:20, :7, :6] = np.ldexp(1.0, lo)
    v[30:50, 9:, 3:] += np.ldexp(1.0, hi - 1)
    x = np.asfortranarray(v.astype(np.float32))
    c = float(np.ldexp(1.0, hi))
    got = mexct.CUDAmex_TVmin_3D(x, c, steps=1)
    assert np.array_equal(got, _step(x, c))
