"""Traversal launches at the edges of their dispatch: ray counts around the
chunks that waves are dealt and claim, and rays with zero, infinite and NaN
components through the 8-wide nodes against the binary ones."""
import numpy as np
import pytest

from luz_amd import api
from oracle import oracle as orc
from tests.helpers import oracle_scene, random_rays, scaled_instances

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


@pytest.mark.parametrize("stack", [8, 32])
@pytest.mark.parametrize("n", [1, 786432, 786433, 1 << 20])
def test_ray_counts_around_chunks_of_other_stacks(ctx, cube, n, stack):
    # 32 entries leave three workgroups a CU (dealt up to 786,432 rays), 8 five
    g, rays, want = cube
    two = np.tile(rays.download(np.float32, (1 << 19, 8)), (2, 1))
    ctx.set_trace_config(stack_entries=stack)
    got = _hits(ctx, g.tlas, ctx.to_device(two), n)
    ctx.set_trace_config(stack_entries=16)
    np.testing.assert_array_equal(got, np.tile(want, 2)[:n])


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


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("size", [(1, 1), (64, 1), (65, 3), (131, 77)])
@pytest.mark.parametrize("lights", ["axis", "at_pixel", "near"])
def test_culled_pixels_change_no_count(ctx, size, lights, wide):
    """Culling by pixel keeps every count, on 102 instances (both words of a
    candidate mask) with whole, partial and single-pixel groups: a directional
    light along an axis (segments without extent in two axes), a point light at a
    pixel's own position, and one just off the surface with a large radius; AO
    rays far shorter and longer than the distance between instances."""
    W, H = size
    c = api.Context(0) if wide else ctx
    if wide:
        c.set_precision(api.PRECISION_WIDE)
    s = api.HostScene(api.SCENE_SPHERES, 0)
    g = api.GPUScene(c, s)
    _, _, cam = s.camera()
    o2w, mesh, mats = s.nodes()
    moved = o2w.copy()
    moved[:, 3::4] += np.float32([7.0, 5.0, 3.0])
    o2w, mesh = np.concatenate([o2w, moved]), np.concatenate([mesh, mesh])
    tlas = c.create_tlas(len(mesh))
    tlas.build([api.make_instance(g.blas(int(m)), o2w[i], i) for i, m in enumerate(mesh)])
    o = oracle_scene(s)
    o.set_instances(o2w, mesh)
    gd = api.GBufferDevice(c, W, H)
    c.primary_gbuffer(tlas, cam, mats + mats, gd.desc())
    gbuf = gd.download()
    covered = np.flatnonzero(gbuf["normal"].reshape(H * W, -1)[:, :3].any(1))
    sb = s.pack()
    if len(covered):
        p = gbuf["position"].reshape(H * W, -1)[covered[len(covered) // 2], :3]
        for l in range(sb.num_lights):
            light = sb.lights[l]
            if lights == "axis":
                light.type = api.LIGHT_DIRECTIONAL
                light.direction[:] = [(0.0, -1.0, 0.0), (1.0, 0.0, 0.0), (0.0, 0.0, -1.0)][l % 3]
            else:
                light.type = api.LIGHT_POINT
                off = 0.0 if lights == "at_pixel" else 0.02
                light.position[:] = [float(v) + off for v in p]
                light.radius = 0.5 if lights == "near" else 0.0
    nl = sb.num_lights
    for ao_max in (1 / 16, 4.0):
        sb.ao_max = ao_max
        want_sh, want_ao, _ = o.trace_visibility(gbuf, W, H, sb)
        dsh, dao = c.buffer(nl * W * H), c.buffer(W * H)
        print(f"{W}x{H} {lights} wide {wide} AO {ao_max}: {len(covered)} pixels", flush=True)
        c.trace_visibility(tlas, gd.desc(), sb, dsh, dao)
        np.testing.assert_array_equal(dsh.download(np.uint8, (nl, W * H)), want_sh)
        np.testing.assert_array_equal(dao.download(np.uint8, W * H), want_ao)
    tlas.destroy()
    g.close()
    if wide:
        c.close()


@pytest.mark.parametrize("copies", [1, 2, 3])
@pytest.mark.parametrize("size", [(1, 1), (9, 7), (131, 77)])
def test_closest_hits_of_tiles_match_oracle(ctx, size, copies):
    """Primary rays of whole and partial 8x8 tiles on 51, 102 and 153 instances (one
    and two words of candidates, and the walk from the TLAS root), from the scene's
    camera and from inside an instance's box along an axis (directions of both signs
    and zero components in one tile): the G-buffer bit for bit."""
    W, H = size
    s = api.HostScene(api.SCENE_SPHERES, 0)
    g = api.GPUScene(ctx, s)
    o2w, mesh, mats = s.nodes()
    n = len(mesh)
    all_o2w = np.concatenate([o2w] * copies)
    for c in range(1, copies):
        all_o2w[c * n:(c + 1) * n, 3::4] += np.float32([7.0, 5.0, 3.0]) * c
    all_mesh = np.concatenate([mesh] * copies)
    tlas = ctx.create_tlas(n * copies)
    tlas.build([api.make_instance(g.blas(int(m)), all_o2w[i], i) for i, m in enumerate(all_mesh)])
    o = oracle_scene(s)
    o.set_instances(all_o2w, all_mesh)
    _, _, cam = s.camera()
    hit = 0
    for inside in (False, True):
        if inside:
            cam.eye[:] = [float(v) for v in o2w[1, 3::4]]
            cam.forward[:], cam.right[:], cam.up[:] = (0.0, 0.0, 1.0), (1.0, 0.0, 0.0), (0.0, 1.0, 0.0)
        gd = api.GBufferDevice(ctx, W, H)
        print(f"{W}x{H}, {n * copies} instances, inside {inside}", flush=True)
        ctx.primary_gbuffer(tlas, cam, mats * copies, gd.desc())
        got, want = gd.download(), o.primary_gbuffer(cam, mats * copies, W, H)
        for k in ("position", "normal"):
            np.testing.assert_array_equal(got[k].view(np.uint32), want[k].view(np.uint32), err_msg=k)
        for k in ("albedo", "material", "emission"):
            np.testing.assert_array_equal(got[k], want[k], err_msg=k)
        hit += int((got["normal"] != 0).any())
    assert hit
    tlas.destroy()
    g.close()


def _unrotated(c, size=1.0):
    """Five sphere meshes (vertices times `size`) in 40 instances of several scales
    without rotation, so that a ray's zero and tiny components reach the object
    space; returns GPU scene, TLAS and oracle scene."""
    s = api.HostScene(api.SCENE_SPHERES, 0)
    rng = np.random.default_rng(17)
    xyz = rng.uniform(-6, 6, (40, 3)) * size
    o2w = scaled_instances(xyz, rng.choice([0.5, 1.0, 2.0], 40))
    mesh = np.arange(40, dtype=np.uint32) % 5
    o = orc.OracleScene()
    blas = []
    for m in range(5):
        v, idx = s.mesh(m)
        v = v.copy()
        v[:, :3] *= np.float32(size)
        o.add_mesh(v, idx)
        blas.append(c.create_blas(c.to_device(v), 48, len(v), c.to_device(idx), len(idx)))
    o.set_instances(o2w, mesh)
    tlas = c.create_tlas(40)
    tlas.build([api.make_instance(blas[m], o2w[i], i) for i, m in enumerate(mesh)])
    return blas, tlas, o


def _both_trees(ctx, rays, size=1.0):
    wide = api.Context(0)
    wide.set_precision(api.PRECISION_WIDE)
    got = []
    for c in (ctx, wide):
        blas, tlas, o = _unrotated(c, size)
        got.append(_hits(c, tlas, c.to_device(rays), len(rays)))
        tlas.destroy()
        for b in blas:
            b.destroy()
    wide.close()
    return got[0], got[1], o


@pytest.mark.parametrize("size, smallest", [(1.0, -40), (1000.0, -36)])
def test_tiny_direction_components_lose_no_hit(ctx, size, smallest):
    """Direction components from 1e-40 to 1e-18 of both signs on one or two axes, origins
    inside the boxes: the reciprocal of such a component is finite while a node's plane
    distances come near the largest float."""
    rng = np.random.default_rng(5)
    n = 60000
    rays = random_rays(rng, n, (0, 0, 0), 7.0 * size, 20.0 * size)
    tiny = np.float32(10.0) ** rng.uniform(smallest, -18, (n, 2)) * rng.choice([-1.0, 1.0], (n, 2))
    k = np.arange(n)
    rays[k, 4 + k % 3] = tiny[:, 0].astype(np.float32)
    two = k % 4 == 0
    rays[two, 4 + (k[two] + 1) % 3] = tiny[two, 1].astype(np.float32)
    plain, wide, o = _both_trees(ctx, rays, size)
    want, _ = o.any_hit(rays)
    print(f"size {size}: {int(want.sum())} of {n} rays hit, 8-wide {int(wide.sum())}", flush=True)
    assert 0 < want.sum() < n
    np.testing.assert_array_equal(plain, want)
    np.testing.assert_array_equal(wide, want)


def test_ranges_that_are_no_numbers_meet_the_same_triangles_in_both_trees(ctx):
    """NaN and infinite range ends, on ordinary rays and on rays with a NaN component
    (whose box tests compare NaN with NaN: a miss)."""
    rng = np.random.default_rng(23)
    n = 40000
    rays = random_rays(rng, n, (0, 0, 0), 7.0, 20.0)
    ends = np.array([np.nan, np.inf, -np.inf], np.float32)
    k = np.arange(n)
    rays[k, np.where(k % 2, 3, 7)] = ends[rng.integers(0, 3, n)]
    both = k % 5 == 0
    rays[both, 3], rays[both, 7] = ends[rng.integers(0, 3, both.sum())], ends[rng.integers(0, 3, both.sum())]
    nan = k % 3 == 0
    rays[nan, np.array([0, 1, 2, 4, 5, 6])[rng.integers(0, 6, nan.sum())]] = np.nan
    rays[nan & (k % 2 == 0), 4] *= -1       # NaNs of both signs
    plain, wide, _ = _both_trees(ctx, rays)
    print(f"{int(plain.sum())} of {n} rays hit, 8-wide {int(wide.sum())}", flush=True)
    assert 0 < plain.sum() < n
    np.testing.assert_array_equal(wide, plain)


def test_timings_after_ray_queries_count_their_rays(ctx):
    """A ray query or an unculled call after a culled one reports its own traced rays."""
    W, H = 160, 90
    s = api.HostScene(api.SCENE_SPHERES, 0)
    g = api.GPUScene(ctx, s)
    _, _, cam = s.camera()
    _, _, mats = s.nodes()
    gd = api.GBufferDevice(ctx, W, H)
    ctx.primary_gbuffer(g.tlas, cam, mats, gd.desc())
    sb = s.pack()
    sh, ao = ctx.buffer(sb.num_lights * W * H), ctx.buffer(W * H)
    rays = random_rays(np.random.default_rng(1), 777, (0, 0.5, 0), 2.0)
    for _ in range(2):
        ctx.trace_visibility(g.tlas, gd.desc(), sb, sh, ao)
        t = ctx.timings()
        assert 0 < t.traced_rays < t.rays      # culled
        assert ctx.timings().traced_rays == t.traced_rays
        _hits(ctx, g.tlas, ctx.to_device(rays), len(rays))
        t = ctx.timings()
        assert (t.rays, t.traced_rays) == (777, 777)
    g.close()


@pytest.mark.parametrize("ao", [(-3.0, 0.5), (-0.5, 0.25), (-2.0, -0.5), (-4.0, 4.0)])
def test_culling_keeps_ao_ranges_behind_the_surface(ctx, ao):
    """AO ranges that start behind the origin, further than they reach ahead of it: the
    culled counts equal the unculled ones and the oracle's."""
    W, H = 96, 64
    s = api.HostScene(api.SCENE_SPHERES, 0)
    g = api.GPUScene(ctx, s)
    _, _, cam = s.camera()
    _, _, mats = s.nodes()
    gd = api.GBufferDevice(ctx, W, H)
    ctx.primary_gbuffer(g.tlas, cam, mats, gd.desc())
    sb = s.pack()
    sb.ao_min, sb.ao_max, sb.ao_num_samples = *ao, 8
    want_sh, want_ao, _ = oracle_scene(s).trace_visibility(gd.download(), W, H, sb)
    nl = sb.num_lights
    for cull in (False, True):
        ctx.set_group_culling(cull)
        dsh, dao = ctx.buffer(nl * W * H), ctx.buffer(W * H)
        ctx.trace_visibility(g.tlas, gd.desc(), sb, dsh, dao)
        np.testing.assert_array_equal(dao.download(np.uint8, W * H), want_ao, err_msg=f"culled {cull}")
        np.testing.assert_array_equal(dsh.download(np.uint8, (nl, W * H)), want_sh)
    g.close()


@pytest.mark.parametrize("far", [10.0, 1e18, 1e37, np.finfo(np.float32).max])
def test_culling_keeps_an_instance_with_a_far_vertex(ctx, far):
    """A box that reaches far, up to past the largest float (its padded bound is
    infinite): rays still meet the triangle beside the pixels."""
    W = H = 24
    verts = np.zeros((6, 12), np.float32)
    verts[:3, :3] = [(-1, 0.5, -1), (1, 0.5, -1), (0, 0.5, 1)]            # a roof over the pixels
    verts[3:, :3] = [(5, 5, 5), (6, far, 5), (5, 5, 6)]
    idx = np.arange(6, dtype=np.uint32)
    blas = ctx.create_blas(ctx.to_device(verts), 48, 6, ctx.to_device(idx), 6)
    tlas = ctx.create_tlas(1)
    tlas.build([api.make_instance(blas, np.eye(3, 4, dtype=np.float32).reshape(12), 0)])
    gd = api.GBufferDevice(ctx, W, H)
    gbuf = gd.download()
    y, x = np.mgrid[0:H, 0:W].astype(np.float32) / W - 0.5
    gbuf["position"] = np.stack([x, 0 * x, y], -1).reshape(gbuf["position"].shape).astype(np.float32)
    gbuf["normal"] = np.broadcast_to(np.float32([0, 1, 0]), gbuf["normal"].shape).copy()
    gd.upload(gbuf)
    sb = api.HostScene(api.SCENE_CUBE, 0).pack()
    sb.ao_min, sb.ao_max, sb.ao_num_samples = 1e-4, 2.0, 16
    got = []
    for cull in (False, True):
        ctx.set_group_culling(cull)
        dsh, dao = ctx.buffer(sb.num_lights * W * H), ctx.buffer(W * H)
        ctx.trace_visibility(tlas, gd.desc(), sb, dsh, dao)
        got.append((dsh.download(np.uint8, (sb.num_lights, W * H)), dao.download(np.uint8, W * H)))
    print(f"unoccluded AO samples: {int(got[0][1].sum())} unculled, {int(got[1][1].sum())} culled", flush=True)
    assert got[0][1].sum() < 16 * W * H
    np.testing.assert_array_equal(got[1][0], got[0][0])
    np.testing.assert_array_equal(got[1][1], got[0][1])
    tlas.destroy()
    blas.destroy()
