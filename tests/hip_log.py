"""What calls of the C ABI do on the host, seen without a GPU: record() runs them in
a child process on a HIP runtime of bookkeeping alone (fake_hip.cpp) and returns,
call by call, the allocations and the kernels launched."""
import json
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
_lib = None

_CHILD = r"""
import ctypes as C, json, os, sys
import numpy as np
from mexct import _lib as L
l, p = L.lib(), C.c_void_p
log = open(os.environ["FAKE_HIP_LOG"], "a")
ctxs, res = {}, []
IN, IN2, OUT = p(1 << 40), p(1 << 41), p(1 << 42)

def ctx(k):
    if k not in ctxs:
        ctxs[k] = p()
        L.check(l.mexct_ctx_create(C.byref(ctxs[k]), 0, None))
    return ctxs[k]

for c in json.load(sys.stdin):
    log.write("call\n")
    log.flush()
    h, op = ctx(c.get("ctx", 0)), c["op"]
    n = c.get("n", 0)
    ang = (np.arange(max(n, 1)) * 0.01).astype(np.float32)
    a, sad, geom = ang.ctypes.data_as(p), c.get("sad", 1000.0), c.get("geom", 2)
    W, H, G = c.get("W"), c.get("H"), c.get("items", 1)
    o = L.opts(c.get("st", 0), c.get("steps", 0))
    if op == "autotune":
        rc = l.mexct_ctx_set_autotune(h, c["mode"])
    elif op == "fp":
        rc = l.mexct_fp_batch_dev(h, IN, 0, G, W, H, sad, a, n, geom, OUT, o)
    elif op == "bp":
        rc = l.mexct_bp_batch_dev(h, IN, 0, G, W, H, n, sad, a, geom, OUT, o)
    elif op == "filter":
        rc = l.mexct_prefilter_dev(h, IN, W, H, n, geom, sad, a, 3, 1.0, -1.0, OUT)
    elif op == "osc":
        k = c["subsets"]
        picks = np.arange(k, dtype=np.int32)
        rc = l.mexct_osc_iter_dev(h, OUT, W, H, IN, IN2, n, k, picks.ctypes.data_as(p), a, sad, geom, o)
    elif op == "tv":
        rc = l.mexct_tvmin_dev(h, OUT, *c["N"], 0.1, o)
    elif op == "tuned":
        cfg = (C.c_int32 * 4)()
        rc = l.mexct_tuned_config(1, geom, c.get("st", 0), W, H, n, cfg)
        res.append({"rc": rc, "cfg": list(cfg)})
        continue
    else:
        raise ValueError(op)
    res.append({"rc": rc, "error": l.mexct_last_error().decode(),
                "held": l.mexct_ctx_workspace_bytes(h)})
print(json.dumps(res))
"""


def _fake():
    global _lib
    if _lib is None:
        d = tempfile.mkdtemp(prefix="fake_hip_")
        _lib = os.path.join(d, "fake_hip.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-shared", os.path.join(HERE, "fake_hip.cpp"),
                        "-o", _lib, "-ldl"], check=True)
    return _lib


def record(calls, memory=None):
    """calls: dicts of op (fp, bp, filter, osc, tv, autotune, tuned) and its sizes;
    memory: bytes of device memory.  A dict a call: rc, error, held (workspace
    bytes after it), mallocs, kernels ((demangled name, grid, block, lds), ...)."""
    lib = _fake()
    fd, log = tempfile.mkstemp(dir=os.path.dirname(lib))
    os.close(fd)
    env = dict(os.environ, FAKE_HIP_LOG=log,
               LD_PRELOAD=(lib + " " + os.environ.get("LD_PRELOAD", "")).strip(),
               PYTHONPATH=os.path.join(os.path.dirname(HERE), "mex-cuda-ct_amd"))
    if memory is not None:
        env["FAKE_HIP_BYTES"] = str(int(memory))
    r = subprocess.run([sys.executable, "-c", _CHILD], input=json.dumps(calls), env=env, text=True,
                       capture_output=True)
    assert r.returncode == 0, r.stderr[-3000:]
    out = json.loads(r.stdout.splitlines()[-1])
    # (c++filt does not know _Float16's code, DF16_)
    names = subprocess.run(["c++filt"], input=open(log).read().replace("DF16_", "Dh"), text=True,
                           capture_output=True, check=True).stdout
    at = -1
    for c in out:
        c["mallocs"], c["kernels"] = [], []
    for line in names.splitlines():
        if line == "call":
            at += 1
        elif at >= 0 and line.startswith("malloc"):
            out[at]["mallocs"].append(int(line.split()[1]))
        elif at >= 0 and line.startswith("launch"):
            f = line[7:].rsplit(" ", 7)
            name = f[0].split("mexct::", 1)[-1].split("(")[0] if "mexct::" in f[0] else f[0]
            num = [int(v) for v in f[1:]]
            out[at]["kernels"].append((name, tuple(num[:3]), tuple(num[3:6]), num[6]))
    assert at == len(out) - 1
    return out


def names(call, *prefixes):
    """The kernels of a recorded call that begin with one of the prefixes, once each."""
    return sorted({k[0] for k in call["kernels"] if k[0].startswith(prefixes)})
