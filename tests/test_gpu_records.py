"""Per-triangle and per-light records that the shading kernels read.

Scenes of generated meshes around the block sizes the records are made in,
with and without vertex normals, no light, one or many emissive triangles
(normals agreeing with the winding and against it), beside an infinite light:
both integrators against the oracle.
"""
import numpy as np
import pytest

from conftest import icosphere_scene
from test_gpu_megakernel import mk_render
from test_gpu_render import assert_images_match, gpu_render

pytestmark = pytest.mark.gpu


def _scene(krr, n, lights, flip, sky):
    rng = np.random.default_rng(n + lights)

    def mesh(k, lo, hi, size, normals, **more):
        c = lo + (hi - lo) * rng.random((k, 1, 3))
        p = (c + size * (rng.random((k, 3, 3)) - 0.5)).reshape(-1, 3)
        m = {"type": "mesh", "material": 0, "positions": p.round(4).reshape(-1).tolist(), "indices": list(range(3 * k)), **more}
        if normals is not None:
            m["normals"] = np.tile(normals, (3 * k, 1)).reshape(-1).tolist()
        return m

    lo, hi = np.array([-1.0, 0.0, -1.0]), np.array([1.0, 1.5, 1.0])
    model = [mesh(n - n // 2, lo, hi, 0.5, None)]
    if n // 2:
        model.append(mesh(n // 2, lo, hi, 0.5, np.array([0.1, 0.9, 0.2]), material=1))
    if lights:
        model.append(mesh(lights, np.array([-1.0, 1.8, -1.0]), np.array([1.0, 2.2, 1.0]), 0.6, np.array([0.0, 1.0 if flip else -1.0, 0.0]),
                          emission=[6.0, 5.0, 4.0]))
    cfg = {"model": model, "materials": [{"bsdf": "diffuse", "params": {"diffuse": [0.7, 0.6, 0.5]}},
                                         {"bsdf": "conductor", "params": {"diffuse": [0.9, 0.8, 0.7], "roughness": 0.3}}],
           "camera": {"eye": [0.0, 1.0, 3.5], "target": [0.0, 0.8, 0.0]}}
    if sky:
        cfg["environment"] = {"tint": [0.3, 0.4, 0.5], "scale": 1.0}
    return krr.Scene(cfg)


@pytest.mark.parametrize("n,lights,flip,sky", [(1, 1, False, False), (2, 0, False, True), (255, 2, False, True), (256, 63, True, False),
                                               (257, 64, False, False), (700, 65, True, True)])
def test_records_match_oracle(krr, oracle, gpu, n, lights, flip, sky):
    print(f"case: {n} triangles, {lights} lights, flip={flip}, sky={sky}", flush=True)
    s = _scene(krr, n, lights, flip, sky)
    g, gs = gpu_render(krr, gpu, s, 40, 30, {"spp": 2, "max_depth": 6}, frame_index=2)
    o, os_ = oracle.render(s.desc, s.camera(0), 40, 30, 2, spp=2, max_depth=6)
    assert gs["closest_rays"] == os_["closest_rays"] and gs["shadow_rays"] == os_["shadow_rays"]
    assert_images_match(g, o)
    g, gs = mk_render(krr, gpu, s, 40, 30, {"spp": 2, "max_depth": 6}, frame_index=2)
    o, os_ = oracle.render_megakernel(s.desc, s.camera(0), 40, 30, 2, spp=2, max_depth=6)
    assert gs["closest_rays"] == os_["closest_rays"] and gs["shadow_rays"] == os_["shadow_rays"]
    assert_images_match(g, o)


def _free_bytes(gpu):
    import ctypes as C
    free, total = C.c_size_t(), C.c_size_t()
    gpu.synchronize()
    gpu.check(gpu.runtime().hipMemGetInfo(C.byref(free), C.byref(total)))
    return free.value


@pytest.mark.parametrize("media", [False, True])
def test_triangle_records_only_where_they_are_read(krr, gpu, tmp_path, media):
    """Scenes with texture lookups build hits from the vertex arrays: without
    media nothing reads a triangle's record, and none is kept (96 bytes each,
    of 328 K triangles)."""
    print(f"case: device memory of a scene under an image environment, media={media}", flush=True)
    np.save(tmp_path / "sky.npy", np.ones((4, 8, 3), np.float32))
    cfg = icosphere_scene(count=256, level=3, res=(32, 32), media=media, grid_res=16)
    used = []
    for textured in (False, True, False, True):  # the first of a kind may also pay for the runtime's own memory
        s = krr.Scene(dict(cfg, environment={"image": str(tmp_path / "sky.npy")}) if textured else cfg)
        wf = krr.WavefrontPathTracer({"spp": 1, "max_depth": 3})
        before = _free_bytes(gpu)
        wf.set_scene(s)
        used.append(before - _free_bytes(gpu))
        wf.close()
    records = 96 * s.n_triangles
    print("bytes without / with textures", used[2:], "records", records, flush=True)
    if media:
        assert used[3] >= used[2]
    else:
        assert used[3] < used[2] - 0.8 * records
