"""Shapes of the persistent launch ("launch_in_force"): blocks, lanes of a wave
that take up paths, samples of a pixel per launch, entries of a lane's
traversal stack in LDS."""
import numpy as np
import pytest

from conftest import CORNELL, icosphere_scene

pytestmark = pytest.mark.gpu


def _frame(krr, gpu, scene, w, h, params, frame_index=3):
    """Film, launch shape and counters of one frame."""
    wf = krr.WavefrontPathTracer(params)
    wf.set_scene(scene)
    wf.resize(w, h)
    film = gpu.DeviceBuffer(w * h * 16)
    wf.begin_frame(scene.camera(0), frame_index)
    wf.render(film.ptr, 0)
    stats = wf.stats()
    out = film.to_numpy(np.float32, (h, w, 4))
    launch = wf.to_json()["launch_in_force"]
    wf.close()
    return out, launch, stats


@pytest.mark.parametrize("scene,spp,more", [("cornell", 257, {}), ("cornell", 300, {"legacy_spp_accumulate": True}), ("field", 256, {"refill_lanes": 8}),
                                            ("field", 513, {"refill_lanes": 8})])
def test_launches_run_a_bounded_number_of_samples(krr, gpu, scene, spp, more):
    """A launch runs at most 256 samples of a pixel; the next one goes on with
    the pixel's sampler and sum, so the film is that of a launch per sample."""
    print(f"case: {scene} 31x17 {spp} spp {more}", flush=True)
    s = krr.Scene(CORNELL if scene == "cornell" else icosphere_scene(count=64, level=2, res=(31, 17)))
    params = dict({"spp": spp, "max_depth": 4}, **more)
    a, la, sa = _frame(krr, gpu, s, 31, 17, params)
    b, _, sb = _frame(krr, gpu, s, 31, 17, dict(params, wavefront_depths=1))
    assert la["samples"] == min(spp, 256)
    assert sa["closest_launches"] == -(-spp // 256)
    assert sa["closest_rays"] == sb["closest_rays"] and sa["shadow_rays"] == sb["shadow_rays"]
    assert np.array_equal(a, b)


def test_views_run_a_bounded_number_of_samples(krr, gpu):
    print("case: views, 260 spp", flush=True)
    s = krr.Scene(icosphere_scene(count=64, level=2, res=(31, 17)))
    a, _, sa = _frame(krr, gpu, s, 31, 17, {"spp": 260, "max_depth": 4})
    for graph in (True, False):
        wf = krr.WavefrontPathTracer({"spp": 260, "max_depth": 4, "graph": graph})
        wf.set_scene(s)
        film = gpu.DeviceBuffer(31 * 17 * 16)
        wf.set_views([(s.camera(0), 31, 17, film.ptr)])
        for _ in range(3):  # replays
            wf.render_views(3, 0)
            gpu.synchronize()
            assert np.array_equal(a, film.to_numpy(np.float32, (17, 31, 4)))
        st = wf.stats()
        assert st["closest_launches"] == 2 and st["closest_rays"] == sa["closest_rays"]
        assert wf.to_json()["launch_in_force"]["samples"] == 256
        wf.close()


@pytest.mark.parametrize("entries", [0, 1, 2, 3, 4, 16, 96])
def test_stack_entries_in_lds_are_the_setting(krr, gpu, entries):
    """stack_lds_entries of each lane are kept in LDS, or all that the tree
    needs (three per level and four)."""
    print(f"case: stack_lds_entries={entries}", flush=True)
    s = krr.Scene(icosphere_scene(count=64, level=2, res=(32, 32)))
    accel = krr.Accel(s.desc)
    need = 3 * accel.info()["max_depth"] + 4
    accel.close()
    _, launch, _ = _frame(krr, gpu, s, 32, 32, {"spp": 1, "max_depth": 3, "stack_lds_entries": entries})
    print(launch, "needed", need, flush=True)
    assert launch["stack_lds_entries"] == min(entries, need)


@pytest.mark.parametrize("scene,refill,media,half", [("cornell", 0, False, True), ("cornell", 8, False, False), ("field", 0, False, False),
                                                     ("field", 8, False, False), ("field", 0, True, False)])
@pytest.mark.parametrize("w,h", [(64, 48), (131, 77)])
def test_lanes_that_take_up_paths(krr, gpu, scene, refill, media, half, w, h):
    """Small frames take the fewest lanes per wave that hold their paths in the
    resident waves, or in half of them for small trees without refill or media."""
    print(f"case: {scene} refill={refill} media={media} {w}x{h}", flush=True)
    s = krr.Scene(CORNELL if scene == "cornell" else icosphere_scene(count=64, level=2, res=(w, h), media=media, grid_res=16))
    params = {"spp": 1, "max_depth": 2, "refill_lanes": refill, "trace_block_size": 128}
    _, full, _ = _frame(krr, gpu, s, 1024, 768, params)
    _, small, _ = _frame(krr, gpu, s, w, h, params)
    assert full["lanes"] == 64  # more paths than lanes: every resident block
    waves = full["blocks"] * 2 // (2 if half else 1)
    lanes = 64
    while lanes > 1 and waves * (lanes // 2) >= w * h:
        lanes //= 2
    print("full", full, "small", small, flush=True)
    assert small["lanes"] == lanes and small["blocks"] == -(-w * h // (2 * lanes))


@pytest.mark.parametrize("more,dense_from", [({}, 3.0), ({"occupancy": 0.5}, 1.5), ({"node_format": "quantized"}, None)])
def test_four_waves_per_simd_for_many_paths(krr, gpu, more, dense_from):
    """The refill launch's 4-wave form takes frames of three times the paths it
    has lanes, on as many lanes as the device and "occupancy" give it, over 2 MB
    of nodes as they are read (18,000 nodes: not when quantised)."""
    import ctypes as C
    print(f"case: waves per SIMD {more}", flush=True)
    cus = C.c_int()
    f = gpu.runtime().hipDeviceGetAttribute
    gpu.check(f(C.byref(cus), 63, 0))  # hipDeviceAttributeMultiprocessorCount
    lanes, share = cus.value * 1024, more.get("occupancy", 1.0)
    s = krr.Scene(icosphere_scene(count=110, level=2, res=(64, 64)))
    accel = krr.Accel(s.desc)
    nodes = accel.info()["nodes"]
    accel.close()
    assert 1 << 14 <= nodes < 1 << 15
    params = dict({"spp": 1, "max_depth": 1, "trace_block_size": 64, "refill_lanes": 8}, **more)
    for paths, dense in ((3 * lanes, True), (3 * lanes - 64, dense_from != 3.0), (3 * lanes // 2, dense_from == 1.5), (3 * lanes // 2 - 64, False)):
        _, launch, _ = _frame(krr, gpu, s, 64, paths // 64, params)
        waves = launch["blocks"] / (cus.value * 4 * share)  # per SIMD
        print(paths, launch, waves, flush=True)
        assert waves == (4 if dense and dense_from else 3)
