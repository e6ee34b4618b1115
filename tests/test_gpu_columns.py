"""Parallel and fan projections by detector columns: the kernels that march
(project) or gather (backproject) several rows of a column at once, at the
edges of their row groups, lanes and tiles.

A parallel or fan sample has row weight exactly 0, so the column kernels
read one row where the general ones read two: they must give the general
kernels' bits, NaN included where a voxel or pixel of the second row is not
finite.
"""
import numpy as np
import pytest

import mexct
from mexct import device

pytestmark = pytest.mark.gpu

STORAGES = [mexct.F32, mexct.F16, mexct.BF16]


def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _spoil(a, seed):
    """A few values that are not finite, the corners' among them."""
    r = _rng(seed)
    for v in (np.nan, np.inf, -np.inf):
        a[tuple(r.integers(0, s) for s in a.shape)] = v
    a[0, 0, 0] = np.inf
    a[-1, -1, -1] = np.nan
    return a


# rows: one, a lane's 4 and its neighbours, past the 32 ceil(W/32) rows that
# the projector computes, several row groups; columns: around a block's; the
# last five are past the 1024 waves from which a lane takes four rows
FP_SIZES = [(2, 1, 3), (5, 3, 9), (16, 4, 8), (33, 5, 17), (31, 70, 5), (64, 129, 4), (100, 66, 11),
            (40, 3, 1200), (33, 1, 4100), (64, 129, 24), (130, 37, 40), (161, 130, 20)]


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("W,H,n", FP_SIZES)
def test_column_fp_equals_ray_fp(gpu, monkeypatch, W, H, n, bad):
    import torch
    ctx = device.Context(0)
    ang = (np.arange(n) * (2 * np.pi / n) + 0.03).astype(np.float32)
    v = _rng(W + H).uniform(-1, 1, (2, H, W, W)).astype(np.float32)
    if bad:
        v[0] = _spoil(v[0], W)
    vols = torch.from_numpy(v).cuda()
    for geom, sad in ((0, 300.0), (1, 1.5 * W), (1, 900.0)):
        for st in STORAGES:
            print(f"fp geom={geom} sad={sad} storage={st} W={W} H={H} n={n} bad={bad}", flush=True)
            got = torch.full((2, n, H, W), -7.0, device="cuda")
            ref = torch.full((2, n, H, W), -9.0, device="cuda")
            ctx.fp_batch(vols, sad, ang, n, geom, got, storage=st)
            monkeypatch.setenv("MEXCT_FP_LAYOUT", "wide64")  # the ray-per-lane kernel
            ctx.fp_batch(vols, sad, ang, n, geom, ref, storage=st)
            monkeypatch.delenv("MEXCT_FP_LAYOUT")
            g, r = got.cpu().numpy(), ref.cpu().numpy()
            assert np.array_equal(g, r, equal_nan=True), (geom, sad, st)
            assert np.isnan(r[0]).any() == bad and not np.isnan(r[1]).any()
    ctx.close()


@pytest.mark.parametrize("geom", [0, 1])
@pytest.mark.parametrize("st", STORAGES)
def test_column_osc_projection_equals_ray_projection(gpu, monkeypatch, geom, st):
    import torch
    ctx = device.Context(0)
    for W, H, n, subsets in ((34, 37, 11, 3), (9, 70, 5, 2)):
        print(f"osc geom={geom} storage={st} W={W} H={H} n={n}", flush=True)
        r = _rng(W)
        ang = (np.arange(n) * (2 * np.pi / n)).astype(np.float32)
        mu = r.uniform(0.001, 0.02, (H, W, W)).astype(np.float32)
        pre = r.uniform(0.5e5, 1e5, (n, H, W)).astype(np.float32)
        post = (pre * r.uniform(0.2, 0.9, pre.shape)).astype(np.float32)
        outs = []
        for force in (False, True):
            t = [torch.from_numpy(a).cuda() for a in (mu, pre, post)]
            if force:
                monkeypatch.setenv("MEXCT_FP_LAYOUT", "wide64")
            ctx.osc_iter(*t, subsets, np.arange(subsets), ang, 500.0, geom, storage=st)
            if force:
                monkeypatch.delenv("MEXCT_FP_LAYOUT")
            outs.append([a.cpu().numpy() for a in t])
        for a, b in zip(*outs):
            assert np.array_equal(a, b, equal_nan=True)
    ctx.close()


@pytest.mark.parametrize("st", [mexct.F16, mexct.BF16])
def test_column_fp_compensated_sums_equal_ray_fp(gpu, monkeypatch, st):
    # every ray longer than long_ray: both kernels sum sample pairs with compensation
    import ctypes as C

    import torch
    from mexct import _lib as L
    W, H, n = 50, 21, 6
    ang = (np.arange(n) * 0.7 + 0.1).astype(np.float32)
    vol = torch.from_numpy(_rng(3).uniform(0, 1, (H, W, W)).astype(np.float32)).cuda()
    ctx = device.Context(0)
    out = []
    for force in (False, True):
        o = torch.zeros((n, H, W), device="cuda")
        if force:
            monkeypatch.setenv("MEXCT_FP_LAYOUT", "wide64")
        torch.cuda.synchronize()
        L.check(L.lib().mexct_fp_dev(ctx._h, C.c_void_p(vol.data_ptr()), L.F32, W, H, 400.0,
                                     ang.ctypes.data_as(C.c_void_p), n, 0,
                                     C.c_void_p(o.data_ptr()), L.opts(st, long_ray=1)))
        ctx.sync()
        if force:
            monkeypatch.delenv("MEXCT_FP_LAYOUT")
        out.append(o.cpu().numpy())
    ctx.close()
    assert np.array_equal(out[0], out[1])
