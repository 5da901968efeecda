"""Rays with zero, infinite and NaN components through the 8-wide nodes against
the binary ones."""
import numpy as np
import pytest

from luz_amd import api
from tests.helpers import random_rays

pytestmark = pytest.mark.gpu


def _hits(ctx, tlas, rays, n):
    out = ctx.to_device(np.full(n + 64, 7, np.uint8))
    ctx.trace_rays(tlas, rays, n, out)
    got = out.download(np.uint8, n + 64)
    assert (got[n:] == 7).all()      # nothing written past the last ray
    return got[:n]


def test_special_rays_meet_the_same_triangles_in_both_trees(ctx):
    """Zero, negative-zero, infinite, denormal and NaN components: any-hit results of
    the 8-wide tree equal the binary tree's."""
    rng = np.random.default_rng(11)
    rays = random_rays(rng, 60000, (0, 0, 0), 50.0, 100.0)
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-40, -1e-40, 1e30], np.float32)
    k = np.arange(len(rays))
    rays[k, 4 + k % 3] = special[rng.integers(0, 2, len(k))]             # axis-parallel planes
    odd = k % 2 == 1
    rays[odd, 4 + (k[odd] + 1) % 3] = 0.0                               # axis-parallel rays
    weird = k % 5 == 0
    rays[weird, rng.integers(0, 8, weird.sum())] = special[rng.integers(0, len(special), weird.sum())]
    nan = k % 50 == 7
    rays[nan, 3] = np.nan                                               # NaN tmin, half of them on NaN rays
    rays[k % 100 == 7, 4:7] = np.nan
    rays = rays[~(np.abs(rays[:, 4:7]) < 1e-30).all(1)]                 # a direction of zero is no ray
    got = []
    wide = api.Context(0)
    wide.set_precision(api.PRECISION_WIDE)
    for c in (ctx, wide):
        s = api.HostScene(api.SCENE_SPHERES, 0)
        g = api.GPUScene(c, s)
        got.append(_hits(c, g.tlas, c.to_device(rays), len(rays)))
        g.close()
    wide.close()
    print(f"{int(got[0].sum())} of {len(rays)} rays hit", flush=True)
    assert 0 < got[0].sum() < len(rays)
    np.testing.assert_array_equal(got[1], got[0])
