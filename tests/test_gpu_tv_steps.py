"""The TV step kernel at the edges of its tiles: lanes (30 or 62 outputs of 32
or 64), rows per lane, slices per workgroup, volumes without an interior, and
values for which its fast square root and division step aside.  The 20-step
result is compared bit for bit with the same steps' gradients formed by the
oracle and the update taken in float, up to the norm's last bit.
"""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu


def _steps(x, c, n):
    """n steps with the oracle's float gradient and a norm summed in FP64."""
    for _ in range(n):
        g = O.tv_gradient(x)
        with np.errstate(all="ignore"):
            a = np.float32(-c) / np.float32(np.sqrt(np.sum(g.astype(np.float64) ** 2)))
            x = (a * g + x).astype(np.float32)
    return x


SHAPES = [(1, 1, 1), (3, 3, 3), (30, 5, 4), (31, 9, 5), (62, 17, 3), (63, 64, 6), (95, 33, 13),
          (2, 40, 9), (40, 2, 9), (129, 70, 34), (250, 210, 200)]


@pytest.mark.parametrize("shape", SHAPES)
def test_tv_steps_equal_oracle_gradient(gpu, shape):
    r = np.random.Generator(np.random.PCG64(sum(shape)))
    x = np.asfortranarray((0.02 + 0.002 * r.standard_normal(shape)).astype(np.float32))
    x[: shape[0] // 3] = 0.02  # a flat part: zero gradients and zero square roots
    n = 2 if x.size > 1e6 else 5
    got = mexct.CUDAmex_TVmin_3D(x, 0.01, steps=n)
    ref = _steps(x, 0.01, n)
    # the step is a = c / |g| with |g| rounded once from an FP64 sum: the same
    # float unless two summation orders straddle a rounding boundary
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("value", [np.nan, np.inf, 3e30, 1e-30, 1e-42])
def test_tv_steps_extreme_values(gpu, value):
    r = np.random.Generator(np.random.PCG64(4))
    x = np.asfortranarray(r.uniform(size=(37, 20, 11)).astype(np.float32))
    if np.isfinite(value) and value < 1:
        x = np.asfortranarray((x * value).astype(np.float32))  # every difference tiny
    else:
        x[20, 9, 5] = value
    got = mexct.CUDAmex_TVmin_3D(x, 0.01, steps=1)
    assert np.array_equal(got, _steps(x, 0.01, 1), equal_nan=True)
