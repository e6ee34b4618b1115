"""The kernels that the cone f32 backprojection chooses from, on the CPU from the
launches and allocations that the host code makes."""
import hip_log


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
