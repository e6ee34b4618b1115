"""The TV step's second volumes are spare: a call that fits without them is never
refused for them, neither the TV call nor a later one of the context."""
import hip_log

GIB = 1 << 30
FUSED, PLAIN, UPDATE = "tv_step_kernel<64, 4, false>", "tv_step_kernel<64, 4, true>", "tv_axpy_kernel"
TV = {"op": "tv", "N": [512, 512, 512], "steps": 5}  # 0.5 GiB


def _count(call, name):
    return sum(k[0].startswith(name) for k in call["kernels"])


def test_a_later_call_gets_the_memory_back():
    fp = {"op": "fp", "W": 960, "H": 960, "n": 4}  # a 6.7 GiB copy
    tv, f, again = hip_log.record([TV, fp, dict(TV, N=[64, 64, 64])], memory=8 * GIB)
    assert tv["rc"] == 0 and _count(tv, FUSED) == 4 and tv["held"] > 3 * GIB // 2
    assert f["rc"] == 0 and f["error"] == ""
    assert f["held"] < 7.3 * GIB
    assert again["rc"] == 0


def test_a_call_without_room_for_them():
    (tv,) = hip_log.record([TV], memory=1.2 * GIB)
    assert tv["rc"] == 0 and tv["error"] == "" and tv["held"] < 0.6 * GIB
    assert (_count(tv, FUSED), _count(tv, PLAIN), _count(tv, UPDATE)) == (0, 5, 5)


def test_they_take_at_most_a_quarter_of_the_free_memory():
    for mem, fused in ((4.4 * GIB, 0), (4.8 * GIB, 4)):  # 0.5 GiB of which the gradient takes
        (tv,) = hip_log.record([TV], memory=mem)
        assert tv["rc"] == 0 and _count(tv, FUSED) == fused


def test_a_larger_volume_replaces_them():
    big = dict(TV, N=[512, 512, 1024])
    a, b, c = hip_log.record([TV, big, TV], memory=32 * GIB)
    assert [x["rc"] for x in (a, b, c)] == [0, 0, 0]
    assert _count(b, FUSED) == 4 and len(b["mallocs"]) >= 3 and not c["mallocs"]
    assert b["held"] == c["held"] < 3.1 * GIB
