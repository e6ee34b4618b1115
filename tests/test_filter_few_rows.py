"""The row filter of few rows: its outputs are shared out over the CUs, with the bits
that the same rows have in a large sinogram, where a workgroup takes whole rows."""
import numpy as np
import pytest

import hip_log


@pytest.mark.parametrize("W,rows,least", [(768, 100, 84), (700, 360, 253), (513, 2, 9), (640, 2900, 364),
                                          (512, 4096, 256)])
def test_workgroups(W, rows, least):
    # up to 12 shares of 64 outputs for each 16 rows, until every CU has one
    (c,) = hip_log.record([dict(op="filter", W=W, H=1, n=rows, geom=0)])
    grids = [k[1] for k in c["kernels"] if k[0].startswith("prefilter_mfma")]
    assert len(grids) == 1 and grids[0][0] * grids[0][1] >= least


@pytest.mark.gpu
@pytest.mark.parametrize("W", [30, 64, 65, 130, 300, 449, 513, 640, 700, 768])
def test_same_bits_as_in_a_large_sinogram(gpu, W):
    import torch

    from mexct import device

    n = 5000
    ang = (np.arange(n) / 64.0).astype(np.float32)  # equal angle steps
    x = torch.from_numpy(np.random.Generator(np.random.PCG64(W)).uniform(-1, 1, (n, 1, W))
                         .astype(np.float32)).cuda()
    ctx = device.Context(0)
    want, got = (torch.full((n, 1, W), np.nan, device="cuda") for _ in range(2))
    ctx.prefilter(x, 0, 1000.0, ang, 3, 1.0, want)
    for rows in (2, 16, 17, 100, 383, 1000, 2047, 4080, 4081, 4097):
        print(f"filter W={W} rows={rows}", flush=True)
        got.fill_(np.nan)
        ctx.prefilter(x[:rows].contiguous(), 0, 1000.0, ang[:rows], 3, 1.0, got[:rows])
        assert torch.equal(got[:rows], want[:rows]), rows
        assert bool(torch.isnan(got[rows:]).all())
    ctx.close()
