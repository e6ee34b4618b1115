"""The bench states each operator's gather rate against the unit that its kernel gathers
through, seen from the kernels that the host code launches."""
import bench
import hip_log


def test_unit_of_each_kernel():
    # the bench's scan of cubes at SAD 1000; 2-byte storage through the vector caches
    sizes = (64, 72, 128, 200, 256, 384, 512)
    calls = [dict(op=op, W=s, H=s, n=512, sad=1000.0, st=st, ctx=i)
             for i, s in enumerate(sizes) for op in ("fp", "bp") for st in (0, 1)]
    for c, got in zip(calls, hip_log.record(calls, memory=1 << 44)):
        lds = bool(hip_log.names(got, "bpl_kernel"))
        f = bench.unit_frac(c["op"], c["st"], c["W"], bench.LDS_PEAK_GBS)
        if c["W"] > 68:
            assert f == ({"frac_of_lds_peak": 1.0} if lds else {"frac_of_vector_cache_peak": 2.0}), c
    assert "frac_of_lds_peak" in bench.unit_frac("bp", 0, 384, 1.0)
