"""The variants of the TV step: lanes and rows per lane, slices per workgroup, the sum of
many partials in a launch of its own, and the form without second volumes, whose bits
are the same.  On the CPU, from the launches that the host code makes, each case takes
the variant that it stands for.  On the GPU each step is compared with the oracle's
gradient of the step before."""
import numpy as np
import pytest

import hip_log

# lanes, rows per lane -> volumes, whose last workgroups along each axis are partial
CASES = [((32, 2), (31, 40, 23)), ((32, 2), (17, 72, 69)), ((32, 4), (104, 220, 27)),
         ((32, 4), (37, 155, 222)), ((32, 8), (171, 255, 155)), ((64, 2), (36, 19, 200)),
         ((64, 2), (127, 18, 80)), ((64, 4), (172, 164, 67)), ((64, 4), (281, 47, 150)),
         ((64, 8), (272, 214, 101)), ((64, 4), (384, 380, 371))]
STEPS = 3


def test_cases_take_their_variants():
    got = hip_log.record([dict(op="tv", N=list(N), steps=STEPS, ctx=i) for i, (_, N) in enumerate(CASES)])
    for ((lw, ry), N), c in zip(CASES, got):
        assert hip_log.names(c, "tv_step") == [f"tv_step_kernel<{lw}, {ry}, {f}>" for f in ("false", "true")], N
    # more than 4096 partials: summed by one workgroup between the steps, not by each
    scales = [sum(k[0] == "tv_scale_kernel" for k in c["kernels"]) for c in got]
    assert scales == [1] * (len(CASES) - 1) + [STEPS]


def _volume(shape):
    r = np.random.Generator(np.random.PCG64(sum(shape)))
    x = (0.02 + 0.002 * r.standard_normal(shape, dtype=np.float32)).astype(np.float32)
    x[: shape[0] // 3] = 0.02  # a flat part: zero gradients and zero square roots
    return np.asfortranarray(x)


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c[0] + c[1])))
def test_steps_equal_oracle_gradient(gpu, case):
    import mexct
    import oracle as O

    _, shape = case
    x = _volume(shape)
    for k in range(1, STEPS + 1):
        got = mexct.CUDAmex_TVmin_3D(_volume(shape), 0.01, steps=k)
        g = O.tv_gradient(x)
        a = np.float32(-0.01) / np.float32(np.sqrt(np.sum(g.astype(np.float64) ** 2)))
        # |g| is a float rounded from an FP64 sum: that of another order may be its neighbour
        near = (a, np.nextafter(a, np.float32(0)), np.nextafter(a, np.float32(-1e30)))
        assert any(np.array_equal(got, (b * g + x).astype(np.float32)) for b in near), k
        x = got


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(37, 40, 23), (250, 210, 200), (384, 380, 371)])
def test_without_second_volumes(gpu, shape):
    # captured on a context that has run single steps: an allocation would end the
    # capture, so the steps do without, and give the same bits
    import torch

    from mexct import device

    v = torch.from_numpy(_volume(shape).transpose(2, 1, 0).copy()).cuda()
    want = v.clone()
    ctx = device.Context(0)
    ctx.tvmin(want, 0.01, steps=5)
    ctx.close()
    s = torch.cuda.Stream()
    ctx = device.Context(0, stream=s, order_with_torch=False)
    x = v.clone()
    torch.cuda.synchronize()
    ctx.tvmin(x, 0.01, steps=1)
    torch.cuda.synchronize()
    held = ctx.workspace_bytes()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        ctx.tvmin(x, 0.01, steps=5)
    assert ctx.workspace_bytes() == held
    for _ in range(3):
        x.copy_(v)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(x, want)
    del graph
    x.copy_(v)
    torch.cuda.synchronize()
    ctx.tvmin(x, 0.01, steps=5)  # and with them, on the same context
    ctx.sync()
    assert ctx.workspace_bytes() > held and torch.equal(x, want)
    ctx.close()
