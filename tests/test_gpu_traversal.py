"""Traversal launches at the edges of their dispatch: ray counts around the
chunks that waves are dealt and claim, and rays with zero, infinite and NaN
components through the 8-wide nodes against the binary ones."""
import numpy as np
import pytest

from luz_amd import api
from tests.helpers import oracle_scene, random_rays

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def cube(ctx):
    s = api.HostScene(api.SCENE_CUBE, 0)
    g = api.GPUScene(ctx, s)
    rays = random_rays(np.random.default_rng(3), 1 << 19, (0, 0.5, 0), 2.0, 20.0)
    want, _ = oracle_scene(s).any_hit(rays)
    yield g, ctx.to_device(rays), want
    g.close()


def _hits(ctx, tlas, rays, n):
    out = ctx.to_device(np.full(n + 64, 7, np.uint8))
    ctx.trace_rays(tlas, rays, n, out)
    got = out.download(np.uint8, n + 64)
    assert (got[n:] == 7).all()      # nothing written past the last ray
    return got[:n]


@pytest.mark.parametrize("groups", [0, 1])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 255, 256, 257, 4097, 98303, 393217, 1 << 19])
def test_ray_counts_around_chunks(ctx, cube, n, groups):
    # one workgroup per CU (256 groups) claims chunks from 65,536 x 4 rays on
    g, rays, want = cube
    if groups:
        ctx.set_trace_config(groups_per_cu=groups)
    got = _hits(ctx, g.tlas, rays, n)
    ctx.set_trace_config(groups_per_cu=6)
    np.testing.assert_array_equal(got, want[:n])


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
