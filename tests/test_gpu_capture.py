"""Point calls that use temporary memory, on a stream under capture: the field
records its kernel that needs none, the reference network's calls are refused
(as the first call of a process and later), and the same calls work when the
capture has ended.  No graph is launched: one that held such an allocation,
replayed between eager calls, faulted the GPU.

Run as a program (with the call's name) it checks the process' first call.
"""
import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

if __name__ == "__main__":
    sys.path[:0] = [str(Path(__file__).resolve().parent), str(Path(__file__).resolve().parents[1])]

from helpers import L, ext, DeviceArray, byref, points, unit_dirs  # noqa: E402
from nerf_amd.device import Stream  # noqa: E402

pytestmark = pytest.mark.gpu

CALLS = ("ref_field", "ref_backward", "field")
THREAD_LOCAL = 1  # hipStreamCaptureModeThreadLocal


def _call(which, stream):
    """(the call on stream, its outputs, what it reads)"""
    n = 70001 if which == "field" else 5000  # field: enough points for its split route, which allocates
    p, d = DeviceArray.from_numpy(points(n, seed=1)), DeviceArray.from_numpy(unit_dirs(n, seed=2))
    if which == "field":
        model = ext.Model.create(ext.grid_desc(18, L.NERF_EXT_F16), seed=1, table_range=1.0)
        ms, out = model.struct(), DeviceArray((n, 4), np.float32)
        return lambda: L.call("nerf_ext_field_forward", byref(ms), p.ptr, d.ptr, n, out.ptr, stream.handle), [out], (model, p, d)
    m = ext.RefModel.create(ext.ref_mlp_init(0), ext.ref_mlp_init(1))
    if which == "ref_field":
        out = DeviceArray((n, 4), np.float32)
        return lambda: L.call("nerf_ext_ref_field_forward", m.density.ptr, m.color.ptr, p.ptr, d.ptr, n, out.ptr, None, stream.handle), [out], (m, p, d)
    draw = DeviceArray.from_numpy(np.random.default_rng(3).normal(0, 1e-2, (n, 4)).astype(np.float32))
    out = [DeviceArray((k,), np.float32) for k in (75776, 40960)]
    return lambda: L.call("nerf_ext_ref_backward", m.density.ptr, m.color.ptr, p.ptr, d.ptr, draw.ptr, n, 128.0, out[0].ptr, out[1].ptr, stream.handle), out, (m, p, d, draw)


def _check(which):
    hip = C.CDLL("libamdhip64.so")
    stream = Stream()
    call, outs, _keep = _call(which, stream)
    h, graph, nodes = C.c_void_p(stream.handle), C.c_void_p(), C.c_size_t(99)
    refused = ""
    assert hip.hipStreamBeginCapture(h, THREAD_LOCAL) == 0
    try:
        call()
    except L.NerfError as e:
        refused = str(e)
    assert hip.hipStreamEndCapture(h, C.byref(graph)) == 0 and graph.value
    assert hip.hipGraphGetNodes(graph, None, C.byref(nodes)) == 0 and hip.hipGraphDestroy(graph) == 0
    if which == "field":
        assert not refused and nodes.value == 1, (refused, nodes.value)
    else:
        assert "capturing" in refused and nodes.value == 0, (refused, nodes.value)
    call()
    stream.synchronize()
    assert all(np.any(o.numpy()) for o in outs)


@pytest.mark.parametrize("which", CALLS)
def test_later_call_under_capture(which):
    print(f"[case] {which} under capture, in this process", flush=True)
    _check(which)


@pytest.mark.parametrize("which", CALLS)
def test_first_call_of_a_process_under_capture(which):
    print(f"[case] {which} under capture, first call of a process", flush=True)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), which], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "checked" in r.stdout, r.stdout[-500:] + r.stderr[-1500:]


if __name__ == "__main__":
    _check(sys.argv[1])
    print("checked")
