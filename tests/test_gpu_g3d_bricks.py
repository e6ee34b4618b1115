"""The general-3D backprojector's bricks: every brick of the block order is
summed, for counts around its groups of 4 x 4 and for one layer up to several,
with enough rays to fill and drain both kinds of work queue."""
import numpy as np
import pytest

import mexct
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,W,H,n", [(5, 3, 9, 7, 3), (16, 12, 17, 16, 6), (17, 25, 33, 31, 8),
                                       (64, 13, 40, 24, 10), (66, 37, 41, 33, 9), (82, 49, 50, 20, 4)])
def test_every_brick(gpu, M, N, W, H, n):
    print(f"g3d bricks M={M} N={N} W={W} H={H} n={n}", flush=True)
    r = np.random.Generator(np.random.PCG64(M * N))
    # a source at 2 M opposite a flat detector whose rays cover the volume and
    # its surroundings; some rays along an axis exactly, some short of the volume
    pts = np.zeros((W, H, 6), np.float32)
    u = (np.arange(W) - (W - 1) / 2) * (2.6 * M / W)
    v = (np.arange(H) - (H - 1) / 2) * (2.6 * N / H)
    pts[:, :, 0] = -2.0 * M
    pts[:, :, 3] = 2.0 * M
    pts[:, :, 4] = u[:, None] + r.uniform(-0.3, 0.3, (W, H))
    pts[:, :, 5] = v[None, :] + r.uniform(-0.3, 0.3, (W, H))
    pts[: W // 4, 0, 1] = pts[: W // 4, 0, 4]
    pts[: W // 4, 0, 2] = pts[: W // 4, 0, 5] = 0.25 * N
    pts[0, 1, 3] = -1.5 * M
    pts = np.asfortranarray(pts)
    ang = (np.arange(n) * (2 * np.pi / n) + 0.1).astype(np.float32)
    ang[0] = 0.0
    P = np.asfortranarray(r.uniform(0, 1, (W, H, n)).astype(np.float32))
    ref = O.g3d_bp(P, ang, pts, M, N)
    got = mexct.CUDAmex_general3D_BP(P, ang, pts, M, N, mode=1)
    # exact integer sums of corners rounded at 2^-27 of the largest, once to float
    scale = np.abs(ref).max()
    assert scale > 0
    assert np.abs(got - ref).max() <= 1e-5 * scale
    assert np.linalg.norm(got.astype(np.float64) - ref) <= 1e-6 * np.linalg.norm(ref.astype(np.float64))
