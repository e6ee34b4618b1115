"""The variants of the parallel and fan kernels that work by detector columns: slices per
workgroup and window columns of the backprojector in each storage, rows per lane of
the OSC projections.  On the CPU, from the launches that the host code makes, each
case takes the variant that it stands for; on the GPU its result is compared with
the oracle (the general kernel for OSC)."""
import numpy as np
import pytest

import hip_log

F32, F16, BF16 = 0, 1, 2
NAME = {F32: "float", F16: "half", BF16: "mexct::bf16_t"}
# geometry, storage, slices, window columns -> W, H, SAD, batch; 9 views (a group of eight
# and one) each
CASES = [
    ((0, F32, 32, 16), (25, 32, 300.0, 2)), ((0, F32, 64, 16), (106, 107, 300.0, 1)),
    ((0, F32, 128, 16), (106, 194, 300.0, 1)),
    ((0, F16, 64, 16), (39, 36, 300.0, 1)), ((0, F16, 128, 16), (194, 68, 300.0, 1)),
    ((0, F16, 256, 16), (164, 193, 300.0, 1)),
    ((0, BF16, 64, 16), (26, 43, 300.0, 1)), ((0, BF16, 128, 16), (168, 78, 300.0, 1)),
    ((0, BF16, 256, 16), (157, 196, 300.0, 1)),
    ((1, F32, 32, 16), (46, 52, 230.0, 1)), ((1, F32, 32, 20), (30, 101, 57.4, 2)),
    ((1, F32, 32, 32), (27, 121, 25.8, 1)), ((1, F32, 64, 16), (31, 257, 155.0, 6)),
    ((1, F32, 64, 20), (70, 278, 127.1, 1)), ((1, F32, 64, 32), (62, 202, 74.0, 2)),
    ((1, F32, 128, 16), (106, 219, 530.0, 1)), ((1, F32, 128, 20), (170, 107, 292.5, 1)),
    ((1, F32, 128, 32), (115, 97, 114.9, 2)),
    ((1, F16, 64, 16), (20, 76, 100.0, 1)), ((1, F16, 64, 20), (56, 178, 108.8, 1)),
    ((1, F16, 64, 32), (23, 208, 25.1, 1)), ((1, F16, 128, 16), (183, 71, 915.0, 1)),
    ((1, F16, 128, 20), (126, 90, 183.7, 2)), ((1, F16, 128, 32), (117, 214, 159.5, 1)),
    ((1, F16, 256, 16), (177, 236, 885.0, 1)), ((1, F16, 256, 20), (168, 194, 261.5, 2)),
    ((1, F16, 256, 32), (278, 234, 288.9, 1)),
    ((1, BF16, 64, 16), (25, 47, 125.0, 1)), ((1, BF16, 64, 20), (37, 193, 66.5, 1)),
    ((1, BF16, 64, 32), (34, 38, 47.0, 1)), ((1, BF16, 128, 16), (114, 220, 570.0, 1)),
    ((1, BF16, 128, 20), (178, 67, 334.6, 1)), ((1, BF16, 128, 32), (233, 76, 324.0, 1)),
    ((1, BF16, 256, 16), (109, 217, 545.0, 6)), ((1, BF16, 256, 20), (207, 205, 305.0, 1)),
    ((1, BF16, 256, 32), (166, 227, 199.3, 1))]
VIEWS = 9
# storage, rows per lane -> W, H, views, subsets
OSC = [((F32, 1), (40, 40, 20, 4)), ((F32, 4), (128, 128, 40, 2)), ((F32, 4), (101, 130, 61, 3)),
       ((F16, 4), (130, 128, 34, 1)), ((BF16, 4), (128, 130, 70, 2)), ((F16, 1), (128, 128, 31, 1))]


def _id(c):
    return "-".join(str(v) for v in c[0]) + f"-{c[1][0]}x{c[1][1]}"


def test_cases_take_their_variants():
    got = hip_log.record([dict(op="bp", geom=g, st=st, W=W, H=H, n=VIEWS, sad=sad, items=G, ctx=i)
                          for i, ((g, st, _, _), (W, H, sad, G)) in enumerate(CASES)])
    for ((g, st, zb, cw), shape), c in zip(CASES, got):
        assert hip_log.names(c, "bpc_kernel", "bp_kernel") == [f"bpc_kernel<{g}, {NAME[st]}, {zb}, {cw}>"], shape
    assert len({c[0] for c in CASES}) == 3 * 3 * 4  # all there are
    got = hip_log.record([dict(op="osc", geom=g, st=st, W=W, H=H, n=n, subsets=k, ctx=3 * i + g)
                          for i, ((st, _), (W, H, n, k)) in enumerate(OSC) for g in (0, 1)])
    for i, ((st, z), _) in enumerate(OSC):
        for g in (0, 1):
            assert hip_log.names(got[2 * i + g], "fpc_kernel", "fpz_kernel") == [f"fpc_kernel<{g}, {NAME[st]}, 1, {z}>"]


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_bp_equals_oracle(gpu, case, bad):
    import torch

    import oracle as O
    from mexct import device

    (geom, st, _, _), (W, H, sad, G) = case
    n = VIEWS
    r = np.random.Generator(np.random.PCG64(W + H))
    P = r.uniform(-1, 1, (G, n, H, W)).astype(np.float32)
    if bad:
        for v in (np.nan, np.inf, -np.inf):
            P[r.integers(0, G), r.integers(0, n), r.integers(0, H), r.integers(0, W)] = v
        P[0, 0, 0, 0], P[-1, -1, -1, -1] = np.inf, np.nan
    ang = (np.arange(n) * (2 * np.pi / n) + 0.03).astype(np.float32)
    out = torch.full((G, H, W, W), 7.0, device="cuda")
    ctx = device.Context(0)
    ctx.bp_batch(torch.from_numpy(P).cuda(), sad, ang, geom, out, storage=st)
    ctx.close()
    got = out.cpu().numpy()
    y, x = np.ogrid[:W, :W]
    hw = W // 2 - 1
    assert (got[..., (x - hw) ** 2 + (y - hw) ** 2 >= hw * hw] == 0).all()
    cx, cy = (a.ravel() for a in np.meshgrid(np.arange(W), np.arange(W)))
    if W > 60:
        edge = np.flatnonzero(np.abs(np.hypot(cx - hw, cy - hw) - hw) < 1.0)
        pick = np.concatenate([r.choice(W * W, 1000, replace=False), r.choice(edge, 200)])
        cx, cy = cx[pick], cy[pick]
    # 2-byte storage: a value's rounding (2^-11, 2^-8 of max|P| = 1) and, f16, two packed
    # roundings of the column lerp, times the distance weight, per view
    u = 1.0 if geom == 0 else sad / (sad - W // 2)
    tol = n * u * u * (4 * 2.0 ** -11 if st == F16 else 1.1 * 2.0 ** -8)
    for g in range(G):
        want = O.bp_cols(np.asfortranarray(P[g].transpose(2, 1, 0)), sad, ang, geom, cx, cy)
        have = got[g][:, cy, cx].T
        if st == F32:
            assert np.array_equal(have, want, equal_nan=True), g
        else:
            nan = np.isnan(want)
            assert np.array_equal(np.isnan(have), nan)
            assert np.abs(have - want)[~nan].max() <= tol, g


@pytest.mark.gpu
@pytest.mark.parametrize("geom", [0, 1])
@pytest.mark.parametrize("case", OSC, ids=_id)
def test_osc_equals_ray_projection(gpu, monkeypatch, case, geom):
    import torch

    from mexct import device

    (st, _), (W, H, n, subsets) = case
    ctx = device.Context(0)
    r = np.random.Generator(np.random.PCG64(W))
    ang = (np.arange(n) * (2 * np.pi / n)).astype(np.float32)
    mu = r.uniform(0.001, 0.02, (H, W, W)).astype(np.float32)
    pre = r.uniform(0.5e5, 1e5, (n, H, W)).astype(np.float32)
    post = (pre * r.uniform(0.2, 0.9, pre.shape)).astype(np.float32)
    outs = []
    for force in (False, True):
        t = [torch.from_numpy(a).cuda() for a in (mu, pre, post)]
        if force:
            monkeypatch.setenv("MEXCT_FP_LAYOUT", "wide64")  # the ray-per-lane kernel
        ctx.osc_iter(*t, subsets, np.arange(subsets), ang, 500.0, geom, storage=st)
        if force:
            monkeypatch.delenv("MEXCT_FP_LAYOUT")
        outs.append([a.cpu().numpy() for a in t])
    ctx.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
