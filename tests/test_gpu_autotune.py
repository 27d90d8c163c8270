"""The autotuner's trials are the launches that frames make.

A frame of few paths spreads them over many waves with few lanes each, and a
pixel's samples run one after the other in one launch; a trial that filled its
waves, or traced one sample, would time another launch than the one its
settings are kept for.
"""
import numpy as np
import pytest

from conftest import CORNELL, icosphere_scene

pytestmark = pytest.mark.gpu


def _tracer(krr, gpu, scene, w, h, views, params):
    wf = krr.WavefrontPathTracer(params)
    wf.set_scene(scene)
    film = gpu.DeviceBuffer(w * h * 16)
    cam = scene.camera(0)
    if views:
        wf.set_views([(cam, w, h, film.ptr)])
    else:
        wf.resize(w, h)

    def frame():
        if views:
            wf.render_views(2, 0)
        else:
            wf.begin_frame(cam, 2)
            wf.render(film.ptr, 0)
        gpu.synchronize()
        return film.to_numpy(np.float32, (h, w, 4))

    return wf, frame


@pytest.mark.parametrize("scene,views,more", [
    ("field", False, {}), ("field", True, {}), ("cornell", False, {}), ("media", False, {"max_depth": 6}), ("field", False, {"wavefront_depths": 2}),
    ("field", False, {"nrc": {"train_mod": 4, "batch": 1024}})])
def test_trials_launch_what_frames_launch(krr, gpu, scene, views, more):
    print(f"case: autotune {scene} views={views} {more}", flush=True)
    w, h, spp = 93, 61, 3
    s = krr.Scene(CORNELL if scene == "cornell" else icosphere_scene(count=64, level=2, res=(w, h), media=scene == "media", grid_res=32))
    wf, frame = _tracer(krr, gpu, s, w, h, views, dict({"spp": spp, "max_depth": 5}, **more))
    before = frame()
    rep = wf.autotune(trial_paths=w * h * spp)
    after = frame()
    launch = wf.to_json()["launch_in_force"]
    print("best", rep["best"], "frame", launch, flush=True)
    best = next(c for c in rep["candidates"] if c == rep["best"])
    if "nrc" in more:  # the frame's own kernel has another size: its lanes may differ, not its one sample per launch
        assert best["launch"]["samples"] == launch["samples"] == 1
    else:
        assert best["launch"] == launch
        assert launch["samples"] == (1 if "wavefront_depths" in more else spp)
        assert np.array_equal(before, after)
    wf.close()


@pytest.mark.parametrize("views", [False, True])
def test_short_trials_keep_the_frames_shape(krr, gpu, views):
    """Trials of fewer paths than the frame has keep its kernel, blocks and
    lanes, and trace the samples that fit."""
    print(f"case: autotune short trials views={views}", flush=True)
    w, h, spp = 640, 400, 2
    s = krr.Scene(icosphere_scene(count=64, level=2, res=(w, h)))
    wf, frame = _tracer(krr, gpu, s, w, h, views, {"spp": spp, "max_depth": 5})
    frame()
    rep = wf.autotune(trial_paths=5000)
    frame()
    launch = wf.to_json()["launch_in_force"]
    print("best", rep["best"], "frame", launch, flush=True)
    assert rep["best"]["launch"] == dict(launch, samples=1) and launch["samples"] == spp
    wf.close()
