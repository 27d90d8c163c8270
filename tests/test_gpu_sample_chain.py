"""A pixel's samples in one persistent launch.

With every depth in the persistent launch (wavefront_depths 0) a lane runs
all samples of the pixel it takes up, one after the other; with
wavefront_depths 1 each sample is a launch of its own.  Both keep the order
of the draws and of the radiance additions, so the films must be equal bit
for bit, for frames smaller and larger than the launch's lanes, with and
without ray refill, in media, and with the reference's running sum.
"""
import numpy as np
import pytest

from conftest import CORNELL, icosphere_scene
from test_gpu_render import gpu_render

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,spp,more", [
    (1, 1, 5, {}), (7, 3, 2, {}), (65, 1, 3, {"refill_lanes": 64}), (129, 67, 3, {"legacy_spp_accumulate": True}),
    (129, 67, 4, {"refill_lanes": 8, "trace_block_size": 64, "occupancy": 0.01}), (1033, 517, 2, {"refill_lanes": 16}), (1033, 517, 2, {})])
def test_chained_samples_equal_launches_per_sample(krr, gpu, w, h, spp, more):
    print(f"case: cornell {w}x{h} {spp} spp {more}", flush=True)
    s = krr.Scene(CORNELL)
    params = dict({"spp": spp, "max_depth": 6}, **more)
    a, sa = gpu_render(krr, gpu, s, w, h, params, frame_index=3, frames=2)
    b, sb = gpu_render(krr, gpu, s, w, h, dict(params, wavefront_depths=1), frame_index=3, frames=2)
    assert sa["closest_rays"] == sb["closest_rays"] and sa["shadow_rays"] == sb["shadow_rays"]
    assert np.array_equal(a, b)


def test_chained_samples_in_media(krr, gpu):
    print("case: icosphere field in a grid medium, 97x51, 3 spp", flush=True)
    s = krr.Scene(icosphere_scene(count=64, level=2, res=(97, 51), media=True, grid_res=48))
    params = {"spp": 3, "max_depth": 12, "rr_min_depth": 3}
    a, sa = gpu_render(krr, gpu, s, 97, 51, params)
    b, sb = gpu_render(krr, gpu, s, 97, 51, dict(params, wavefront_depths=1))
    assert sa["closest_rays"] == sb["closest_rays"] and sa["shadow_rays"] == sb["shadow_rays"]
    assert np.array_equal(a, b)


@pytest.mark.parametrize("w,h,spp,more", [(3, 1, 2, {}), (64, 64, 2, {}), (130, 127, 1, {"refill_lanes": 64}), (251, 190, 1, {"refill_lanes": 1}),
                                          (301, 203, 1, {"refill_lanes": 12, "trace_block_size": 256}), (40, 30, 1, {"nrc": {"train_mod": 4}})])
def test_few_paths_in_many_waves(krr, gpu, w, h, spp, more):
    """Frames of fewer paths than the launch has lanes are spread over more
    waves with fewer lanes each.  Launches that fill their waves trace the
    same paths: those over a ray queue (wavefront_depths 1) and, with the
    radiance cache, those held to few blocks ("occupancy")."""
    print(f"case: field {w}x{h} {spp} spp {more}", flush=True)
    s = krr.Scene(icosphere_scene(count=64, level=2, res=(w, h)))
    params = dict({"spp": spp, "max_depth": 8, "refill_lanes": 8}, **more)
    out = []
    for p in (params, dict(params, **({"occupancy": 0.01} if "nrc" in more else {"wavefront_depths": 1}))):
        wf = krr.WavefrontPathTracer(p)
        wf.set_scene(s)
        wf.resize(w, h)
        film = gpu.DeviceBuffer(w * h * 16)
        wf.begin_frame(s.camera(0), 1)
        wf.render(film.ptr, 0)
        st = wf.stats()
        out.append((film.to_numpy(np.float32, (h, w, 4)), st["closest_rays"], st["shadow_rays"], wf.to_json()["launch_in_force"]["lanes"]))
        wf.close()
    (a, ca, sa, lanes), (b, cb, sb, full) = out
    assert lanes < 64 and full == 64
    assert ca == cb and sa == sb
    assert np.array_equal(a, b)
