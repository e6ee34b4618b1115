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


# slices: one, a lane's 4 (8) and its neighbours, up to several workgroups' 32 (64);
# columns: odd, around tiles of 8, the smallest circle; views: around a stage's.  All
# take the fewest slices per workgroup (test_column_variants.py has the others)
BP_SIZES = [(1, 5, 2), (3, 2, 3), (4, 1, 1), (9, 3, 5), (16, 16, 4), (33, 17, 7), (40, 65, 3), (23, 130, 9),
            (200, 131, 6), (370, 3, 2)]


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("W,H,n", BP_SIZES)
def test_column_bp_equals_oracle(gpu, W, H, n, bad):
    import torch

    import oracle as O
    ctx = device.Context(0)
    ang = (np.arange(n) * (2 * np.pi / n) + 0.03).astype(np.float32)
    p = _rng(W + H).uniform(-1, 1, (n, H, W)).astype(np.float32)
    if bad:
        p = _spoil(p, W)
    sino = torch.from_numpy(p).cuda()
    r = W // 2
    # the fan sources: one whose tiles reach many detector columns, a usual
    # one, and one within 20% of the circle (the general kernel)
    for geom, sad in ((0, 300.0), (1, 1.9 * r + 1), (1, 900.0), (1, 1.15 * r + 0.1)):
        want = np.ascontiguousarray(O.bp(np.asfortranarray(p.transpose(2, 1, 0)), sad, ang,
                                         geom).transpose(2, 1, 0))
        nan = np.isnan(want)
        for st in STORAGES:
            print(f"bp geom={geom} sad={sad} storage={st} W={W} H={H} n={n} bad={bad}", flush=True)
            got = torch.full((H, W, W), -7.0, device="cuda")
            ctx.bp(sino, sad, ang, geom, got, storage=st)
            g = got.cpu().numpy()
            if st == mexct.F32:
                assert np.array_equal(g, want, equal_nan=True), (geom, sad)
                continue
            assert np.array_equal(np.isnan(g), nan), (geom, sad, st)
            # a value's error: its storage rounding (2^-11, 2^-8 of max|P| = 1)
            # and, f16, two packed roundings of the column lerp, times the
            # distance weight, per view
            u = 1.0 if geom == 0 else sad / (sad - r)
            tol = n * u * u * (4 * 2.0 ** -11 if st == mexct.F16 else 1.1 * 2.0 ** -8)
            assert np.abs(g - want)[~nan].max(initial=0.0) <= tol, (geom, sad, st)
    ctx.close()


def test_column_bp_batch_equals_single(gpu):
    import torch
    ctx = device.Context(0)
    G, W, H, n = 3, 57, 21, 10
    ang = (np.arange(n) * 0.4).astype(np.float32)
    sinos = torch.from_numpy(_rng(5).uniform(-1, 1, (G, n, H, W)).astype(np.float32)).cuda()
    for geom in (0, 1):
        for st in STORAGES:
            a = torch.full((G, H, W, W), -7.0, device="cuda")
            ctx.bp_batch(sinos, 400.0, ang, geom, a, storage=st)
            for i in range(G):
                b = torch.full((H, W, W), -9.0, device="cuda")
                ctx.bp(sinos[i], 400.0, ang, geom, b, storage=st)
                assert torch.equal(a[i], b)
    ctx.close()
