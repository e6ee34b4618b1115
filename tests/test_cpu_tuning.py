"""A tuned choice serves the kernel that it was timed on and no other, seen from the
launches that the host code makes (the stand-in for the HIP runtime times every
candidate the same, so that tuning keeps the built-in choice)."""
import hip_log

CONE = {"op": "bp", "geom": 2, "W": 64, "H": 300, "n": 40}
FAN = {"op": "bp", "geom": 1, "W": 64, "H": 300, "n": 40}


def test_each_kernel_is_tuned_by_itself():
    # far sources take the LDS and the column kernel, near ones the general one, whose
    # z-range is 48 at 300 rows; the LDS kernel's row starts are 32 apart
    calls = [{"op": "autotune", "mode": 1}]
    for c in (CONE, FAN):
        calls += [dict(c, sad=400.0), dict(c, sad=36.0), dict(c, sad=400.0), dict(c, sad=36.0)]
    out = hip_log.record(calls)
    assert all(c["rc"] == 0 for c in out)
    for base, far, geom in ((1, "bpl_kernel", 2), (5, "bpc_kernel", 1)):
        def main(k):
            return [x[0] for x in out[base + k]["kernels"] if x[0].startswith(("bpl_k", "bpc_k", "bp_k"))]
        assert len(main(0)) > 3 and all(k.startswith(far) for k in main(0))
        assert len(main(1)) == 10  # 9 candidates and the call
        assert main(1)[-1].startswith(f"bp_kernel<{geom}, 48, float")
        assert len(main(2)) == 1 and main(2)[0] == main(0)[-1]
        assert main(3) == main(1)[-1:]


def test_tuned_config_finds_either():
    out = hip_log.record([{"op": "autotune", "mode": 1}, dict(CONE, sad=36.0), dict(CONE, op="tuned"),
                          dict(CONE, sad=400.0), dict(CONE, op="tuned"), dict(CONE, op="tuned", n=41)])
    assert [out[k]["cfg"][0] for k in (2, 4, 5)] == [1, 1, 0]
    assert out[2]["cfg"][2] == 48 and out[4]["cfg"][2] == 32
