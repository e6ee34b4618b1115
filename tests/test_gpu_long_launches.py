"""Calls whose launches hold 2^32 threads or more, which a grid dimension cannot:
each is split, and every ray, voxel and row is there."""
import numpy as np
import pytest

import mexct
import oracle as O
from mexct import device

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx(gpu):
    import torch
    c = device.Context(0)
    yield c
    c.close()
    torch.cuda.empty_cache()


def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


@pytest.mark.parametrize("geom,sad", [(0, 1000.0), (1, 60000.0)])
def test_column_backprojection(ctx, geom, sad):
    # 3000 x 3000 tiles of 512 threads
    import torch
    W, n = 24000, 2
    P = _rng(1).uniform(-1, 1, (W, 1, n)).astype(np.float32)
    ang = np.array([0.4, 2.1], np.float32)
    out = torch.full((1, W, W), np.inf, device="cuda")
    ctx.bp(torch.from_numpy(np.ascontiguousarray(P.transpose(2, 1, 0))).cuda(), sad, ang, geom, out)
    assert not bool(torch.isinf(out).any())
    cx, cy = _rng(2).integers(0, W, (2, 4000))
    cy[:2000] = _rng(3).integers(W // 2, 7 * W // 8, 2000)  # the last tiles within the circle
    got = out.cpu().numpy()[0, cy, cx]
    assert np.array_equal(got, O.bp_cols(np.asfortranarray(P), sad, ang, geom, cx, cy)[:, 0])


# cone: one ray per thread; parallel: four
@pytest.mark.parametrize("geom,n", [(2, (1 << 20) + 3), (0, (1 << 22) + 3)])
def test_projection_of_many_views(ctx, geom, n):
    import torch
    W, sad = 64, 300.0
    vol = _rng(4).uniform(-1, 1, (W, W, W)).astype(np.float32)
    ang = (np.arange(n, dtype=np.float64) * 1e-4).astype(np.float32)
    out = torch.full((n, W, W), np.inf, device="cuda")
    ctx.fp(torch.from_numpy(vol).cuda(), sad, ang, n, geom, out)
    views = np.unique(np.concatenate([[0, n // 2 - 1, n // 2, n // 2 + 1, n - 3, n - 2, n - 1],
                                      _rng(5).integers(0, n, 9)]))
    assert not any(bool(torch.isinf(c).any()) for c in out.split(1 << 18))
    want = O.fp(np.asfortranarray(vol.transpose(2, 1, 0)), sad, ang[views], len(views), geom)
    got = out[torch.from_numpy(views).cuda()].cpu().numpy()
    assert np.array_equal(got, want.transpose(2, 1, 0))


def test_x_fastest_projection_of_many_views(ctx):
    import torch
    W, H, n, sad = 4, 1 << 20, 258, 300.0
    vol = np.ones((H, W, W), np.float32)
    ang = (np.arange(n) * 0.01).astype(np.float32)
    out = torch.full((n, H, W), np.inf, device="cuda")
    ctx.fp(torch.from_numpy(vol).cuda(), sad, ang, n, 0, out)
    assert not bool(torch.isinf(out).any())
    rows = out[:, :32].cpu().numpy()  # the reference's grid computes 32 ceil(W / 32) rows
    assert bool((out[:, 32:] == 0).all())
    for v in (0, 255, 256, 257):
        want = O.fp(np.ones((W, W, 64), np.float32, order="F"), sad, ang[v:v + 1], 1, 0)
        assert np.array_equal(rows[v], want[:, :32, 0].T)  # a parallel ray sees its own slice only


def test_general_3d_atomic_backprojection_of_many_views(ctx):
    # rays that end short of the volume, but for the last view's, an eighth of a
    # turn on, which reach its corner
    import torch
    W, H, n, M, N = 4, 1, (1 << 24) + 2, 24, 20  # 256 threads a view
    pts = np.zeros((6, H, W), np.float32)
    pts[0], pts[3] = 100.0, 13.0
    pts[1] = pts[4] = np.linspace(-2, 2, W, dtype=np.float32)
    pts[2] = pts[5] = np.array([-7.2, -1.0, 0.3, 8.0], np.float32)
    ang = np.zeros(n, np.float32)
    ang[-1] = np.float32(np.pi / 4)
    p = torch.from_numpy(pts).cuda()
    sino = torch.ones((n, H, W), device="cuda")
    got, want = (torch.full((N, M, M), -7.0, device="cuda") for _ in range(2))
    ctx.g3d_bp(sino, ang, p, M, N, got, mode=2)
    ctx.g3d_bp(sino[-1:], ang[-1:], p, M, N, want, mode=2)
    assert bool((want != 0).any())
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)  # sums in any order


def test_row_filter_of_many_rows(ctx):
    # every row the same, so is its filtered one
    import torch
    W, H, n = 2, 1 << 20, 520
    sino = torch.empty((n, H, W), device="cuda")
    sino[..., 0], sino[..., 1] = 0.75, -0.25
    ang = (np.arange(n) / 64.0).astype(np.float32)
    out = torch.full((n, H, W), np.inf, device="cuda")
    ctx.prefilter(sino, 0, 1000.0, ang, 3, 1.0, out)
    few = torch.empty((2, 1, W), device="cuda")
    ctx.prefilter(sino[:2, :1].contiguous(), 0, 1000.0, ang[:2], 3, 1.0, few)
    assert bool((out == few[0, 0]).all())


def test_tv_steps(ctx):
    # constant but for spots in the first and the last slices: the gradient and its
    # norm are those of the spots' surroundings
    import torch
    nx, ny, nz, m = 3, 49216, 65535, 12
    r = _rng(6)
    small = np.full((2 * m, 2 * m, nx), 0.5, np.float32)
    small[2:5, 2:6, 1] += r.uniform(0, 0.1, (3, 4)).astype(np.float32)
    small[-5:-2, -6:-2, 1] += r.uniform(0, 0.1, (3, 4)).astype(np.float32)
    x = torch.full((nz, ny, nx), 0.5, device="cuda")
    x[:m, :m] = torch.from_numpy(small[:m, :m].copy()).cuda()
    x[-m:, -m:] = torch.from_numpy(small[-m:, -m:].copy()).cuda()
    ctx.tvmin(x, 0.01, steps=1)
    v = np.asfortranarray(small.transpose(2, 1, 0))
    g = O.tv_gradient(v)
    a = np.float32(-0.01) / np.float32(np.sqrt(np.sum(g.astype(np.float64) ** 2)))
    want = (a * g + v).astype(np.float32).transpose(2, 1, 0)
    assert np.array_equal(x[:m, :m].cpu().numpy(), want[:m, :m])
    assert np.array_equal(x[-m:, -m:].cpu().numpy(), want[-m:, -m:])
    assert float(x[m:-m].min()) == 0.5 == float(x[m:-m].max())
