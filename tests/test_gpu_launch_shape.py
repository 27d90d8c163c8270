"""Shapes of the persistent launch ("launch_in_force"): blocks, lanes of a wave
that take up paths, samples of a pixel per launch."""
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


@pytest.mark.parametrize("w,h", [(5, 3), (64, 48), (301, 200)])
def test_queue_launches_are_no_larger_than_the_queue(krr, gpu, w, h):
    """Rays of a queue fill waves, so a launch over one needs a block per
    trace_block_size rays; camera paths of a small frame take more."""
    print(f"case: queue launch {w}x{h}", flush=True)
    s = krr.Scene(icosphere_scene(count=64, level=2, res=(w, h)))
    params = {"spp": 2, "max_depth": 5, "trace_block_size": 128}
    a, la, _ = _frame(krr, gpu, s, w, h, dict(params, wavefront_depths=1))
    b, lb, _ = _frame(krr, gpu, s, w, h, params)
    print("queue", la, "camera", lb, flush=True)
    assert la == {"blocks": (w * h + 127) // 128, "lanes": 64, "samples": 1}
    assert lb["blocks"] > la["blocks"] and lb["lanes"] < 64 and lb["samples"] == 2
    assert np.array_equal(a, b)
