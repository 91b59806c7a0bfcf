"""The light tracer runs the iterations of a call in one launch, each into a
splat image of its own, and in as many launches as the splat images' bound
asks for. Every split gives the same sums, up to the order of its float
atomics: one call, one call per iteration, at image sizes below a wave, around
a tile, and where nine iterations need a second launch."""
import numpy as np
import pytest

import pt_util as P
from mufflon_amd import hip
from mufflon_amd import scenes as S

pytestmark = pytest.mark.gpu


def _targets(ctx, pt, calls):
    ctx.lighttracer_reset(pt, variance=True)
    for n in calls:
        ctx.lighttracer_iterate(pt, n, density=True)
    return [ctx.lighttracer_target(pt, hip.LT_RADIANCE), ctx.lighttracer_target(pt, hip.LT_DENSITY),
            ctx.lighttracer_target(pt, hip.LT_RADIANCE, variance=True)]


@pytest.mark.parametrize("width,height,iterations", [(1, 1, 5), (7, 9, 3), (65, 33, 3), (1023, 401, 9)])
def test_launch_shapes_agree(hip_ctx, width, height, iterations):
    c = S.cornell_box(8, 16, width, height)
    print("light tracer regeneration %dx%d, %d iterations" % (width, height, iterations), flush=True)
    pt = P.gpu_pt(hip_ctx, c, seed=5, max_path_length=4)
    one = _targets(hip_ctx, pt, [iterations])
    each = _targets(hip_ctx, pt, [1] * iterations)
    for a, b in zip(one, each):
        # the same positive terms in another order: a pixel takes at most a few
        # thousand of them, each rounding 2^-24 of the sum
        assert np.abs(a - b).max() <= 1e-4 * max(float(np.abs(a).max()), 1e-30)
    assert one[0].max() > 0 or width * height == 1
