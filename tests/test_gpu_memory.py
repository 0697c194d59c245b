"""What the library does when device memory is short: the optional memory goes
first and the calls give the same results.  Each case is a process of its own in
which a small library stands before hipMalloc, hipFree and
hipMallocFromPoolAsync and refuses what a limit does not allow.

Run as a program (with the case's name and the library's path) it is that process.
"""
import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

SHIM = r"""
#include <stddef.h>
#include <map>
#include <mutex>
typedef int (*Malloc)(void**, size_t);
typedef int (*Free)(void*);
typedef int (*FromPool)(void**, size_t, void*, void*);
static Malloc real_malloc; static Free real_free; static FromPool real_pool;
static std::mutex lock; static std::map<void*, size_t> sizes;
static long long live, limit = -1, last; static int fail_next, fail_pool, failed;
extern "C" {
void shim_real(void* m, void* f, void* p) { real_malloc = (Malloc)m; real_free = (Free)f; real_pool = (FromPool)p; }
void shim_limit(long long l) { limit = l; }
void shim_fail(int next, int pool) { fail_next = next; fail_pool = pool; failed = 0; }
long long shim_live() { return live; }
long long shim_last() { return last; }
int shim_failed() { return failed; }
int hipMalloc(void** p, size_t n) {
    std::lock_guard<std::mutex> g(lock);
    if (fail_next > 0 || (limit >= 0 && live + (long long)n > limit)) { if (fail_next > 0) --fail_next; ++failed; *p = 0; return 2; }
    int e = real_malloc(p, n);
    if (e == 0) { sizes[*p] = n; live += n; last = n; }
    return e;
}
int hipFree(void* p) {
    std::lock_guard<std::mutex> g(lock);
    auto it = sizes.find(p);
    if (it != sizes.end()) { live -= it->second; sizes.erase(it); }
    return real_free(p);
}
int hipMallocFromPoolAsync(void** p, size_t n, void* pool, void* stream) {
    if (fail_pool) { ++failed; *p = 0; return 2; }
    return real_pool(p, n, pool, stream);
}
}
"""

CASES = ("tables_last", "tables_given_up", "pool_given_back", "field_without_memory")


def _render_setup():
    from helpers import L, ext

    g = ext.scene_gaussians(32, seed=0)
    bits = ext.occupancy_from_scene(g, 128)
    model = ext.Model.create(ext.grid_desc(19, L.NERF_EXT_F16), seed=4, table_range=1.0)
    occ = ext.occupancy_struct(bits, 128)

    def render(r, views, _keep=bits):  # occ holds the bits' address only
        from helpers import synchronize

        cams = [ext.camera_orbit(0, i, 1.32, (0.5, 0.5, 0.5), 200, 160, 1111.0 * 200 / 800.0) for i in range(views)]
        rgba = r.render(model, occ, cams, 1024)[0]
        synchronize()
        return rgba.numpy().copy()

    return render


def _run(case, shim):
    from helpers import L, ext, DeviceArray, synchronize, byref, points, unit_dirs

    if case == "tables_last":
        # 2^25 possible samples: one chunk, cell tables.  In a byte less than the
        # render takes in all, and in what it takes without them, the tables stay
        # out, not a buffer it needs.
        render = _render_setup()
        before = shim.shim_live()
        r = ext.Renderer()
        want = render(r, 1)
        total, tables = shim.shim_live() - before, shim.shim_last()
        assert tables > 32 << 20 and shim.shim_failed() == 0
        del r
        for room in (total - 1, total - tables + (1 << 20)):
            shim.shim_limit(shim.shim_live() + room)
            shim.shim_fail(0, 0)
            r = ext.Renderer()
            assert np.array_equal(render(r, 1), want) and shim.shim_failed() > 0
            shim.shim_limit(-1)
            del r
    elif case == "tables_given_up":
        # A renderer that holds tables renders three views in the memory that
        # these take without any.
        render = _render_setup()
        before = shim.shim_live()
        r = ext.Renderer()
        want = render(r, 3)
        total, tables = shim.shim_live() - before, shim.shim_last()
        del r
        r = ext.Renderer()
        render(r, 1)
        shim.shim_limit(before + total - tables + (1 << 20))
        assert np.array_equal(render(r, 3), want) and shim.shim_failed() > 0
        shim.shim_limit(-1)
    elif case == "pool_given_back":
        n = 4096
        m = ext.RefModel.create(ext.ref_mlp_init(0), ext.ref_mlp_init(1))
        p, d, o = DeviceArray.from_numpy(points(n, seed=1)), DeviceArray.from_numpy(unit_dirs(n, seed=2)), DeviceArray((n, 4), np.float32)
        for _ in range(2):
            L.call("nerf_ext_ref_field_forward", m.density.ptr, m.color.ptr, p.ptr, d.ptr, n, o.ptr, None, None)
            synchronize()
            L.call("nerf_ext_release_scratch")
        out = C.c_void_p()
        shim.shim_fail(1, 0)  # an allocation that fails once is tried again
        L.call("nerf_ext_malloc", C.byref(out), 1 << 20)
        assert out.value and shim.shim_failed() == 1
        L.call("nerf_ext_free", out)
        shim.shim_fail(2, 0)
        with pytest.raises(L.NerfError):
            L.call("nerf_ext_malloc", C.byref(out), 1 << 20)
        shim.shim_fail(0, 1)
        with pytest.raises(L.NerfError):
            L.call("nerf_ext_ref_field_forward", m.density.ptr, m.color.ptr, p.ptr, d.ptr, n, o.ptr, None, None)
        shim.shim_fail(0, 0)
        L.call("nerf_ext_ref_field_forward", m.density.ptr, m.color.ptr, p.ptr, d.ptr, n, o.ptr, None, None)
        synchronize()
        assert np.any(o.numpy())
    else:
        n = 70001
        model = ext.Model.create(ext.grid_desc(18, L.NERF_EXT_F16), seed=1, table_range=1.0)
        ms = model.struct()
        p, d, o = DeviceArray.from_numpy(points(n, seed=1)), DeviceArray.from_numpy(unit_dirs(n, seed=2)), DeviceArray((n, 4), np.float32)
        got = []
        for fail in (0, 1):
            shim.shim_fail(0, fail)
            L.call("nerf_ext_field_forward", byref(ms), p.ptr, d.ptr, n, o.ptr, None)
            synchronize()
            assert (shim.shim_failed() > 0) == (fail > 0)
            got.append(o.numpy().view(np.uint32).copy())
        assert np.any(got[0]) and np.array_equal(got[0], got[1])


@pytest.fixture(scope="module")
def shim_path(tmp_path_factory):
    d = tmp_path_factory.mktemp("shim")
    (d / "shim.cpp").write_text(SHIM)
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", str(d / "shim.cpp"), "-o", str(d / "libshim.so")], check=True)
    return d / "libshim.so"


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES)
def test_short_memory(shim_path, case):
    print(f"[case] short memory: {case}", flush=True)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), case, str(shim_path)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "checked" in r.stdout, r.stdout[-500:] + r.stderr[-2500:]


if __name__ == "__main__":
    sys.path[:0] = [str(Path(__file__).resolve().parent), str(Path(__file__).resolve().parents[1])]
    shim = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)  # before libnerf.so: its calls bind to the shim
    shim.shim_live.restype = shim.shim_last.restype = C.c_longlong
    shim.shim_limit.argtypes = [C.c_longlong]
    hip = C.CDLL("libamdhip64.so")
    shim.shim_real(*(C.cast(getattr(hip, f), C.c_void_p) for f in ("hipMalloc", "hipFree", "hipMallocFromPoolAsync")))
    _run(sys.argv[1], shim)
    print("checked")
