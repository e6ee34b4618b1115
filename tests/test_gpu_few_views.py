"""Backprojections of one to five views by the general kernel, whose block order
changes with their number: every voxel is written, with the bits of a scan of many
views whose other views are zero, and the oracle's in f32."""
import numpy as np
import pytest

import mexct
import oracle as O
from mexct import device

pytestmark = pytest.mark.gpu


# near sources (general kernel in every storage) and the cone's far ones in 2 bytes
@pytest.mark.parametrize("geom,sad,st", [(2, 33.0, mexct.F32), (1, 33.0, mexct.F32), (2, 33.0, mexct.F16),
                                         (2, 500.0, mexct.F16), (2, 500.0, mexct.BF16)])
def test_few_views(gpu, geom, sad, st):
    import torch
    ctx = device.Context(0)
    for W, H in ((61, 70), (64, 33), (9, 3)):
        many = 12
        ang = (np.arange(many) * 0.37 + 0.1).astype(np.float32)
        P = np.random.Generator(np.random.PCG64(W)).uniform(-1, 1, (many, H, W)).astype(np.float32)
        P[0, 0, 0] = 1.0  # the f16 scale of every prefix
        for n in range(1, 6):
            print(f"bp geom={geom} sad={sad} storage={st} W={W} H={H} n={n}", flush=True)
            got, want = (torch.full((H, W, W), np.inf, device="cuda") for _ in range(2))
            p = torch.from_numpy(P).cuda()
            ctx.bp(p[:n].contiguous(), sad, ang[:n], geom, got, storage=st)
            p[n:] = 0.0
            ctx.bp(p, sad, ang, geom, want, storage=st)
            assert torch.equal(got, want), n
            if st == mexct.F32:
                ref = O.bp(np.asfortranarray(P[:n].transpose(2, 1, 0)), sad, ang[:n], geom)
                assert np.array_equal(got.cpu().numpy(), ref.transpose(2, 1, 0))
    ctx.close()
