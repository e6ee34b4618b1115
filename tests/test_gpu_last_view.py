"""Backprojections that end at each view of a group of eight (by detector columns) and of
four (from LDS): the kernels stop staging there.  The sum over n views is, bit for bit,
that of the oracle."""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu


# par and fan: 32, 64 and 128 slices a workgroup (two stages of four views); cone
@pytest.mark.parametrize("geom,W,H", [(0, 40, 30), (1, 33, 61), (1, 120, 260), (0, 256, 256), (2, 64, 64),
                                      (2, 130, 130)])
def test_last_view(gpu, geom, W, H):
    r = np.random.Generator(np.random.PCG64(W + geom))
    P = r.uniform(-1, 1, (W, H, 18)).astype(np.float32)
    ang = (np.arange(18) * 0.35 + 0.1).astype(np.float32)
    cx, cy = r.integers(0, W, (2, 300))
    for n in list(range(1, 10)) + [11, 12, 15, 16, 17, 18]:
        print(f"bp geom={geom} W={W} H={H} n={n}", flush=True)
        p = np.asfortranarray(P[:, :, :n])
        got = mexct.CUDAmex_BP(p, 500.0, ang[:n], geom)
        assert np.array_equal(got[cx, cy], O.bp_cols(p, 500.0, ang[:n], geom, cx, cy)), n
