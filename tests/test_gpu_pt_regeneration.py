"""Path regeneration of the megakernel: the iterations of a call run in one
launch, lanes of a wave take pixels in 8x8 tiles (all 64 lanes, or fewer for
small images), and further pixels come from a queue where the image exceeds
the resident waves. Every split of the work gives the same bits: one launch,
one launch per iteration and the wavefront kernels, at image sizes around the
tile and at one past the resident lanes."""
import numpy as np
import pytest

import pt_util as P
from mufflon_amd import hip
from mufflon_amd import scenes as S

pytestmark = pytest.mark.gpu


def _image(ctx, pt, calls):
    ctx.pt_reset(pt)
    for n in calls:
        ctx.pt_iterate(pt, n)
    return ctx.pt_target(pt, hip.TARGET_RADIANCE), ctx.pt_target(pt, hip.TARGET_HIT_ID)


@pytest.mark.parametrize("width,height", [(1, 1), (7, 9), (64, 8), (65, 33), (1023, 401)])
def test_launch_shapes_agree(hip_ctx, width, height):
    c = S.cornell_box(8, 16, width, height)
    print("pt regeneration %dx%d" % (width, height), flush=True)
    pt = P.gpu_pt(hip_ctx, c, seed=5, max_path_length=5, nee_count=1)
    one = _image(hip_ctx, pt, [3])
    each = _image(hip_ctx, pt, [1, 1, 1])
    hip_ctx.pt_set_mode(pt, hip.PT_WAVEFRONT)
    wave = _image(hip_ctx, pt, [3])
    hip_ctx.pt_set_mode(pt, hip.PT_MEGAKERNEL)
    for other in (each, wave):
        assert np.array_equal(one[0].view(np.uint32), other[0].view(np.uint32))
        assert np.array_equal(one[1], other[1])
    assert np.isfinite(one[0]).all() and (width * height < 64 or one[0].max() > 0)


def test_calls_of_more_than_one_launch(hip_ctx):
    """A call of more than 2^26 paths is split into launches: five iterations of a
    4096x4096 image run as four and one, with the bits of one launch each."""
    c = S.cornell_box(4, 8, 4096, 4096)
    print("pt regeneration 4096x4096 x 5", flush=True)
    pt = P.gpu_pt(hip_ctx, c, seed=5, max_path_length=1, nee_count=0)
    one = _image(hip_ctx, pt, [5])
    each = _image(hip_ctx, pt, [1] * 5)
    assert np.array_equal(one[0].view(np.uint32), each[0].view(np.uint32))
    assert np.array_equal(one[1], each[1])
    assert one[0].max() > 0


@pytest.mark.parametrize("depth,nee", [(0, 1), (1, 1), (4, 0), (4, 3)])
def test_depths_and_estimates(hip_ctx, oracle, depth, nee):
    c = S.cornell_box(8, 16, 37, 21)
    print("pt regeneration depth %d nee %d" % (depth, nee), flush=True)
    pt = P.gpu_pt(hip_ctx, c, seed=2, max_path_length=depth, nee_count=nee)
    rad, hit = _image(hip_ctx, pt, [4])
    ps = P.oracle_pt_scene(oracle, c, hip_ctx.pt_light_tree(pt))
    o_rad, o_hit, _ = oracle.pt_render(ps, 2, 0, depth, nee, 4)
    assert np.array_equal(hit, o_hit)
    assert not (np.abs(rad - o_rad) > 1e-4 * np.abs(o_rad) + 1e-6).any()
