"""The variants of the cone f32 backprojection that gathers from LDS: slices per wave,
window columns and rows.  On the CPU, from the launches that the host code makes:
each case takes the variant that it stands for, and the copies stay within the
server's footprints.  On the GPU: each case bit for bit against the oracle."""
import numpy as np
import pytest

import hip_log

# (slices per wave, window columns, rows of LDS per column) -> W, H, views, SAD, batch:
# the smallest scans that take the variant and ones with partial tiles, a last workgroup
# of a few slices, views around a group of four
CASES = [((16, 16, 132), (20, 61, 9, 118.6, 1)), ((16, 16, 132), (65, 129, 4, 500.0, 1)),
         ((16, 20, 132), (20, 58, 5, 35.0, 1)), ((16, 20, 132), (75, 131, 7, 155.0, 1)),
         ((24, 16, 132), (81, 68, 5, 368.7, 4)), ((24, 16, 132), (256, 129, 3, 1000.0, 1)),
         ((24, 16, 196), (23, 329, 6, 63.8, 1)),
         ((24, 20, 132), (170, 66, 5, 401.0, 1)),
         ((24, 20, 196), (24, 207, 9, 50.8, 1)), ((24, 20, 196), (189, 167, 4, 360.0, 1)),
         ((32, 16, 196), (37, 381, 5, 195.7, 16)), ((32, 16, 196), (256, 250, 2, 1000.0, 1)),
         ((32, 20, 196), (110, 172, 6, 228.2, 4)), ((32, 20, 196), (256, 256, 3, 460.8, 1))]


def _id(c):
    (zr, cw, p), (W, H, n, sad, G) = c
    return f"{zr}-{cw}-{p}-{W}x{H}x{n}" + (f"-batch{G}" if G > 1 else "")


def test_cases_take_their_variants():
    got = hip_log.record([dict(op="bp", W=W, H=H, n=n, sad=sad, items=G, ctx=i)
                          for i, (_, (W, H, n, sad, G)) in enumerate(CASES)])
    for ((zr, cw, p), shape), c in zip(CASES, got):
        assert hip_log.names(c, "bpl_kernel", "bp_kernel") == [f"bpl_kernel<{zr}, {cw}, {p}, false>"], shape


@pytest.mark.gpu
@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("case", CASES, ids=_id)
def test_equals_oracle(gpu, case, bad):
    import torch

    import oracle as O
    from mexct import device

    _, (W, H, n, sad, G) = case
    r = np.random.Generator(np.random.PCG64(W + H))
    P = r.uniform(-1, 1, (G, n, H, W)).astype(np.float32)
    if bad:
        for v in (np.nan, np.inf, -np.inf):
            P[r.integers(0, G), r.integers(0, n), r.integers(0, H), r.integers(0, W)] = v
        P[0, 0, 0, 0], P[-1, -1, -1, -1] = np.inf, np.nan
    ang = (np.arange(n) * (2 * np.pi / n) + 0.03).astype(np.float32)
    out = torch.full((G, H, W, W), 7.0, device="cuda")
    ctx = device.Context(0)
    ctx.bp_batch(torch.from_numpy(P).cuda(), sad, ang, 2, out)
    ctx.close()
    # every column of a small volume; of a larger one 1000, and the circle's edge
    cx, cy = (a.ravel() for a in np.meshgrid(np.arange(W), np.arange(W)))
    hw = W // 2 - 1
    if W > 100:
        edge = np.flatnonzero(np.abs(np.hypot(cx - hw, cy - hw) - hw) < 1.0)
        pick = np.concatenate([r.choice(W * W, 1000, replace=False), r.choice(edge, 200)])
        cx, cy = cx[pick], cy[pick]
    got = out.cpu().numpy()
    y, x = np.ogrid[:W, :W]
    assert (got[..., (x - hw) ** 2 + (y - hw) ** 2 >= hw * hw] == 0).all()
    for g in range(G):
        want = O.bp_cols(np.asfortranarray(P[g].transpose(2, 1, 0)), sad, ang, 2, cx, cy)
        assert np.array_equal(got[g][:, cy, cx].T, want, equal_nan=True), g


@pytest.mark.gpu
@pytest.mark.parametrize("W,H", [(40, 64), (24, 207)])
def test_angle_not_finite(gpu, W, H):
    # both on the LDS kernel, as the next test asserts: the columns of that view have no
    # rows of their own, and every voxel of the circle is NaN
    import mexct
    import oracle as O

    n = 6
    P = np.asfortranarray(np.ones((W, H, n), np.float32))
    for v in (0, 3, 5):
        ang = np.arange(n, dtype=np.float32)
        ang[v] = np.nan
        got = mexct.CUDAmex_BP(P, 60.0, ang, 2)
        assert np.array_equal(got, O.bp(P, 60.0, ang, 2), equal_nan=True) and np.isnan(got).any()


def test_angle_not_finite_takes_the_lds_kernel():
    for c in hip_log.record([dict(op="bp", W=W, H=H, n=6, sad=60.0) for W, H in ((40, 64), (24, 207))]):
        assert [k[:10] for k in hip_log.names(c, "bpl_kernel", "bp_kernel")] == ["bpl_kernel"]


def test_a_batch_stays_within_its_items_footprints():
    # One scan takes the LDS kernel with 16 slices per wave.  A batch of them takes
    # more slices, or the general kernel, with a taller copy: at this many views by
    # more than the row starts that the footprint counts for each item.
    from mexct import serve

    for W, H, n, sad in ((130, 99, 60000, 1000.0), (100, 52, 60000, 800.0), (64, 50, 40, 500.0)):
        (got,) = hip_log.record([dict(op="bp", W=W, H=H, n=n, sad=sad, items=4)], memory=1 << 45)
        assert got["rc"] == 0
        staging = 4 * 4 * (W * H * n + W * W * H)
        assert got["held"] + staging <= 4 * serve.request_footprint(1, W, H, n, 2, sad), (W, H, n)
