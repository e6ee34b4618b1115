"""Cone projections from copies whose z rows are lengthened (tight rows within 64
bytes of a multiple of 4096), against the oracle, at the heights where that
begins and ends."""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H", [499, 500, 508, 516, 517, 1012])
def test_long_rows_equal_oracle(gpu, H):
    W, n = 24, 2
    print(f"fp rows H={H}", flush=True)
    r = np.random.Generator(np.random.PCG64(H))
    V = np.asfortranarray(r.uniform(0, 1, (W, W, H)).astype(np.float32))
    ang = np.array([0.3, 2.2], np.float32)
    assert np.array_equal(mexct.CUDAmex_FP(V, 300.0, ang, n, 2), O.fp(V, 300.0, ang, n, 2))


@pytest.mark.parametrize("H", [500, 512, 517])
@pytest.mark.parametrize("st,name", [(mexct.F16, "f16"), (mexct.BF16, "bf16")])
def test_long_rows_two_byte(gpu, st, name, H):
    W, n = 24, 2
    print(f"fp rows {name} H={H}", flush=True)
    r = np.random.Generator(np.random.PCG64(H))
    V = np.asfortranarray(r.uniform(0, 1, (W, W, H)).astype(np.float32))
    ang = np.array([0.3, 2.2], np.float32)
    ref = O.fp(V, 300.0, ang, n, 2)
    got = mexct.CUDAmex_FP(V, 300.0, ang, n, 2, storage=st)
    # a sample of values below 1, 0.5 on average, is off by at most nine f16
    # roundings of 2^-12 (four differences, the packed lerps), or one bf16 one of
    # 2^-9: below 2^-7 of the largest sum
    assert np.abs(got - ref).max() <= 2.0 ** -7 * np.abs(ref).max()
