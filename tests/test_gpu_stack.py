"""The traversal stack at every split between LDS and the overflow area.

A node visit pushes up to three children at once; pushes and pops that cross
the LDS part's end take another path.  The closest hit does not depend on
where an entry is kept, so hits, visibility and frames must be equal bit for
bit whatever "stack_lds_entries" is: none, fewer than one push, one push, a
few, more than the tree needs.
"""
import numpy as np
import pytest

from conftest import icosphere_scene
from test_gpu_render import gpu_render
from test_gpu_trace import _assert_same_hits, _gpu_closest, _rays_towards_triangles

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def field(krr, oracle):
    s = krr.Scene(icosphere_scene(count=128, level=2, res=(64, 64)))
    pos, idx, _ = s.arrays()
    rays = _rays_towards_triangles(pos, idx, 12345, np.random.default_rng(5), np.array([-0.5, 0.0, -0.5]), np.array([1.5, 1.7, 1.5]), jitter=0.05)
    rays[::3, 3] = 0.7
    return s, rays, oracle.trace_closest(s.desc, rays), oracle.trace_any(s.desc, rays)


@pytest.mark.parametrize("nodes", ["float", "quantized"])
@pytest.mark.parametrize("entries", [0, 1, 2, 3, 4, 5, 7, 96])
def test_hits_do_not_depend_on_stack_split(krr, gpu, field, entries, nodes):
    print(f"case: stack_lds_entries={entries} {nodes} nodes, 12345 rays", flush=True)
    s, rays, closest, visible = field
    g, vis, _ = _gpu_closest(krr, gpu, s, rays, {"stack_lds_entries": entries, "node_format": nodes})
    _assert_same_hits(g, closest)
    assert np.array_equal(vis, visible)


@pytest.mark.parametrize("entries,more", [(0, {}), (1, {"refill_lanes": 0}), (4, {"refill_lanes": 16, "leaf_share": 0}), (3, {"lds_nodes": 64}),
                                          (5, {"wavefront_depths": 2}), (2, {"node_format": "quantized", "trace_block_size": 256})])
def test_frames_do_not_depend_on_stack_split(krr, gpu, field, entries, more):
    print(f"case: frame with stack_lds_entries={entries} {more}", flush=True)
    s = field[0]
    params = {"spp": 2, "max_depth": 8, "rr_min_depth": 3, "refill_lanes": 8}
    a, sa = gpu_render(krr, gpu, s, 131, 77, dict(params, **dict(more, stack_lds_entries=entries)))
    b, sb = gpu_render(krr, gpu, s, 131, 77, dict(params, stack_lds_entries=96))
    assert sa["closest_rays"] == sb["closest_rays"] and sa["shadow_rays"] == sb["shadow_rays"]
    assert np.array_equal(a, b)
