"""Places of a persistent launch handed out to waves and lanes: no ray is left
out or taken twice, for counts below, at and beyond what the launch's waves
start with, and for the grid that the fixed scratch holds."""
import numpy as np
import pytest

from conftest import CORNELL, icosphere_scene
from test_gpu_trace import _assert_same_hits

pytestmark = pytest.mark.gpu

HIT = np.dtype([("t", "<f4"), ("prim", "<i4"), ("b1", "<f4"), ("b2", "<f4")])


@pytest.fixture(scope="module")
def rays(krr, oracle):
    s = krr.Scene(CORNELL)
    rng = np.random.default_rng(3)
    n = 600001
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = rng.random((n, 3), dtype=np.float32) * [0.8, 1.6, 0.8] + [-0.4, 0.2, -0.4]
    r[:, 3] = np.where(rng.random(n) < 0.3, 0.5, np.inf)
    r[:, 4:7] = rng.standard_normal((n, 3), dtype=np.float32)
    return s, r, oracle.trace_closest(s.desc, r), oracle.trace_any(s.desc, r)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 127, 128, 129, 4095, 4097, 131071, 131073, 262143, 262144, 262145, 524287, 524289, 600001])
def test_every_ray_is_traced_once(krr, gpu, rays, n):
    print(f"case: {n} rays", flush=True)
    s, r, closest, visible = rays
    accel = krr.Accel(s.desc)
    d = gpu.DeviceBuffer.from_numpy(r[:n])
    hits, vis = gpu.DeviceBuffer(16 * n), gpu.DeviceBuffer(4 * n)
    for k in range(2):  # a second pass finds the counter set anew
        for buf, size in ((hits, 16 * n), (vis, 4 * n)):
            buf.copy_from_numpy(np.full(size, 0xA5, np.uint8))
        accel.trace_closest(d.ptr, n, hits.ptr, 0)
        accel.trace_any(d.ptr, n, vis.ptr, 0)
        gpu.synchronize()
        _assert_same_hits(hits.to_numpy(HIT, (n,)), closest[:n])
        assert np.array_equal(vis.to_numpy(np.int32, (n,)), visible[:n])
    hits.copy_from_numpy(np.full(16 * n, 0xA5, np.uint8))
    accel.trace_closest_noalloc(d.ptr, n, hits.ptr, 0)
    gpu.synchronize()
    _assert_same_hits(hits.to_numpy(HIT, (n,)), closest[:n])
    accel.close()


@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (8, 8, 1), (9, 7, 1), (65, 33, 2), (500, 301, 1), (1031, 517, 1), (1031, 517, 2)])
@pytest.mark.parametrize("spheres", [0, 16, 160])
def test_every_pixel_is_rendered_once(krr, gpu, w, h, spp, spheres):
    """The megakernel pass hands out pixels as given shares (one sample, small
    trees) or from a counter; a launch held to few blocks makes many shares
    of each wave's.  The same film and rays, and no pixel left out."""
    print(f"case: {spheres} spheres {w}x{h} {spp} spp", flush=True)
    s = krr.Scene(icosphere_scene(count=spheres, level=2, res=(w, h)) if spheres else CORNELL)
    out = []
    for occupancy in (1.0, 0.05, 0.002):
        mk = krr.MegakernelPathTracer({"spp": spp, "max_depth": 5, "occupancy": occupancy})
        mk.set_scene(s.desc)
        mk.resize(w, h)
        film = gpu.DeviceBuffer.from_numpy(np.full((h, w, 4), np.nan, np.float32))
        for frame in (3, 4):
            mk.begin_frame(s.camera(0), frame)
            mk.render(film.ptr, 0)
        st = mk.stats()
        out.append((film.to_numpy(np.float32, (h, w, 4)), st["closest_rays"], st["shadow_rays"]))
        mk.close()
    assert np.isfinite(out[0][0]).all() and out[0][1] >= w * h * spp
    for o in out[1:]:
        assert np.array_equal(o[0], out[0][0]) and o[1:] == out[0][1:]


@pytest.mark.parametrize("n", [1000, 48601, 300000])
def test_both_traces_share_one_overflow_area(krr, gpu, n):
    """Closest hits and then as many shadow rays on a new accel allocate the
    stack's overflow area once: free device memory does not change between."""
    import ctypes as C
    print(f"case: {n} rays, one allocation", flush=True)
    s = krr.Scene(icosphere_scene(count=160, level=2, res=(32, 32)))
    rng = np.random.default_rng(n)
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3], r[:, 3], r[:, 4:7] = rng.random((n, 3)), np.inf, rng.standard_normal((n, 3))
    d, hits, vis = gpu.DeviceBuffer.from_numpy(r), gpu.DeviceBuffer(16 * n), gpu.DeviceBuffer(4 * n)

    def free():
        gpu.synchronize()
        f, t = C.c_size_t(), C.c_size_t()
        gpu.check(gpu.runtime().hipMemGetInfo(C.byref(f), C.byref(t)))
        return f.value

    seen = []
    for _ in range(3):
        accel = krr.Accel(s.desc, {"stack_lds_entries": 0})
        accel.trace_closest(d.ptr, n, hits.ptr, 0)
        a = free()
        accel.trace_any(d.ptr, n, vis.ptr, 0)
        seen.append((a, free()))
        accel.close()
    print(seen, flush=True)
    assert all(a == b for a, b in seen)
