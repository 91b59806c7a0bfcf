"""Builds that one workgroup holds (2 to 2048 primitives: its sort, hierarchy
and collapse take one launch each) against the oracle, bit for bit, at the
edges of waves, of the sort's padding and of the range: the staged build, the
allocation-free build and the instance level."""
import numpy as np
import pytest

import scene_util as U
from mufflon_amd import scenes as S

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 63, 64, 65, 127, 129, 1023, 1025, 2047, 2048, 2049]


def _mesh(n, copies):
    v, t = S.random_triangle_soup(n, seed=n)
    # every `copies` triangles share one centroid, and with it the Morton code
    return v, np.ascontiguousarray(t[(np.arange(n) // copies) * copies])


@pytest.mark.parametrize("copies", [1, 7])
@pytest.mark.parametrize("n", SIZES)
def test_small_build_matches_oracle(hip_ctx, oracle, n, copies):
    v, t = _mesh(n, copies)
    print("small build n=%d copies=%d" % (n, copies), flush=True)
    want = oracle.lbvh_build_tris(v, t, None)
    lod = hip_ctx.lod_create(v, t)
    got = hip_ctx.lbvh_build_stages(lod, n, want["bbox"])
    for k in ("unsorted_keys", "sorted_keys", "sorted_ids", "parents", "offsets"):
        assert np.array_equal(got[k], want[k]), k
    nint, nodes, ids = hip_ctx.lbvh_get(lod, n)
    assert nint == want["num_internal"]
    assert np.array_equal(nodes, want["nodes"]) and np.array_equal(ids, want["sorted_ids"])
    dv, dt = hip_ctx.to_device(v), hip_ctx.to_device(t)
    dn, di = hip_ctx.alloc(64 * n), hip_ctx.alloc(4 * n)
    assert hip_ctx.lbvh_build_noalloc(dv.ptr, len(v), dt.ptr, n, want["bbox"], dn.ptr, di.ptr) == nint
    assert np.array_equal(dn.download(np.uint8, 64 * nint), nodes)
    assert np.array_equal(di.download(np.int32, n), ids)


@pytest.mark.parametrize("n", [2, 65, 2048, 2049])
def test_small_instance_level_matches_oracle(hip_ctx, oracle, n):
    geoms, rng = U.small_lods(3)
    lods = []
    for v, t in geoms:
        lods.append(hip_ctx.lod_create(v, t))
        hip_ctx.lbvh_build(lods[-1])
    boxes = np.stack([oracle.vertex_box(v) for v, _ in geoms])
    il = rng.integers(0, len(geoms), n).astype(np.int32)
    w = U.random_transforms(n, 4, spread=50.0)
    print("small instance level n=%d" % n, flush=True)
    sc = hip_ctx.scene_create(np.array(lods, np.int32)[il], w)
    box, nint, nodes, ids = hip_ctx.scene_get(sc, n)
    want = oracle.lbvh_build_instances(w, boxes, il, box)
    assert nint == want["num_internal"]
    assert np.array_equal(nodes, want["nodes"]) and np.array_equal(ids, want["sorted_ids"])
