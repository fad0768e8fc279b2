"""The automatic traversal (triangle tree) against the kernel that tests every
candidate (traversal_prefilter 1, itself checked against the oracle): equal
records, bit for bit, at the sizes where the tree's construction and the
quads' remainders can go wrong, and for rays and scenes outside the ordinary."""
import dataclasses

import numpy as np
import pytest

from rsh_amd import queries

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def engine(rsh):
    e = rsh.Engine(0)
    yield e
    e.close()


def make_scene(rsh, tris, per_object):
    """A scene of the given [T, 3, 3] vertices, per_object consecutive triangles each."""
    T = len(tris)
    v = np.zeros((T, 3, 4), np.float32)
    v[:, :, :3] = tris
    n = np.cross(tris[:, 1] - tris[:, 0], tris[:, 2] - tris[:, 0])
    n /= np.maximum(np.linalg.norm(n, axis=1, keepdims=True), 1e-12)
    nrm = np.zeros((T, 3, 4), np.float32)
    nrm[:, :, :3] = n[:, None]
    spheres = []
    for a in range(0, T, per_object):
        b = min(a + per_object, T) - 1
        p = tris[a:b + 1].reshape(-1, 3).astype(np.float64)
        c = (p.min(0) + p.max(0)) / 2
        spheres.append([*c, np.linalg.norm(p - c, axis=1).max() * 1.0001 + 1e-4, a, b])
    base = rsh.scenes.config0_scene()
    lo, hi = tris.reshape(-1, 3).min(0), tris.reshape(-1, 3).max(0)
    return dataclasses.replace(base, tri_pos=v.reshape(-1, 4), tri_nrm=nrm.reshape(-1, 4),
                               tri_mat=np.zeros(3 * T, np.int32), object_spheres=np.asarray(spheres, np.float32),
                               bounds_min=lo - 1.0, bounds_max=hi + 1.0)


def soup(rng, T, spread=100.0, size=5.0):
    c = rng.uniform(50.0, 50.0 + spread, (T, 1, 3))
    return (c + rng.normal(0.0, size, (T, 3, 3))).astype(np.float32)


def rays_at(rng, sc, n):
    o = rng.uniform(sc.bounds_min, sc.bounds_max, (n, 3))
    t = sc.tri_pos[:, :3].reshape(-1, 3, 3).mean(1)[rng.integers(sc.triangle_total, size=n)]
    d = t + rng.normal(0.0, 1.0, (n, 3)) - o
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    return np.concatenate([o, d], 1).astype(np.float32)


def qcfg(rsh, sc, **kw):
    return dataclasses.replace(rsh.config.config0(8, 8), cell_bits=4, dir_bits=6, **kw).with_scene_bounds(sc)


def check(engine, rsh, sc, rays, **kw):
    cfg = qcfg(rsh, sc, **kw)
    engine.load_scene(sc)
    tmax = np.full(len(rays), 60.0, np.float32)
    for kind in (0, 1):
        got = engine.trace(rays, kind, cfg, tmax=tmax)
        want = engine.trace(rays, kind, dataclasses.replace(cfg, traversal_prefilter=1), tmax=tmax)
        np.testing.assert_array_equal(got, want)
    return want


@pytest.mark.parametrize("T", [1, 2, 4, 5, 8, 9, 63, 65, 513, 4099, 20011])
def test_scene_sizes(engine, rsh, T):
    rng = np.random.default_rng(T)
    sc = make_scene(rsh, soup(rng, T), 7)
    check(engine, rsh, sc, rays_at(rng, sc, 1501))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 64, 65, 1025])
def test_ray_counts(engine, rsh, n):
    rng = np.random.default_rng(n)
    sc = make_scene(rsh, soup(rng, 777), 50)
    check(engine, rsh, sc, rays_at(rng, sc, n))


@pytest.mark.parametrize("variant", [dict(algorithm=1), dict(hit_mode=1), dict(depth=1), dict(depth=3, branch=4),
                                     dict(depth=4, leaf=4, branch=3), dict(leaf=32, branch=2), dict(key_mode=0),
                                     dict(triangle_batch=512), dict(cone_mode=0)])
def test_options(engine, rsh, variant):
    rng = np.random.default_rng(3)
    sc = make_scene(rsh, soup(rng, 3001), 64)
    check(engine, rsh, sc, rays_at(rng, sc, 2003), **variant)


def test_scenes_outside_the_ordinary(engine, rsh):
    rng = np.random.default_rng(5)
    one = soup(rng, 1)
    flat = soup(rng, 600)
    flat[:, :, 1] = 70.0                                     # a flat scene box
    sliver = soup(rng, 600)
    sliver[:, 2] = sliver[:, 1] + 1e-3                       # no reliable plane
    point = soup(rng, 600)
    point[::3, 1] = point[::3, 0]                            # triangles without area
    # nested triangles about one corner, each half the size of the one before:
    # the deepest tree the codes allow, every box on the way of the rays
    s = 0.5 ** np.repeat(np.arange(9), 40)[:, None, None]
    nested = (50.0 + 100.0 * s * (np.asarray([[0.1, 0.1, 0.1], [1.0, 0.1, 0.2], [0.1, 1.0, 0.3]])
                                  + 0.01 * rng.random((360, 3, 3)))).astype(np.float32)
    for tris in (np.repeat(one, 3000, 0), flat, sliver, point, nested):
        sc = make_scene(rsh, tris, 30)
        check(engine, rsh, sc, rays_at(rng, sc, 700))


def test_rays_outside_the_ordinary(engine, rsh):
    """Long, short, axis-parallel, zero and non-finite rays among ordinary ones."""
    rng = np.random.default_rng(6)
    sc = make_scene(rsh, soup(rng, 400), 40)
    rays = rays_at(rng, sc, 640)
    rays[0:64, 3:] *= 1e6
    rays[64:128, 3:] *= 1e-4
    rays[128:192, 3:] = np.eye(3, dtype=np.float32)[rng.integers(3, size=64)]
    rays[192:256, 3:] = -np.eye(3, dtype=np.float32)[rng.integers(3, size=64)]
    rays[256:264, 3:] = 0.0
    rays[264:272, 3:] = np.nan
    rays[272:280, 3] = np.inf
    rays[280:288, 0] = np.nan
    rays[288:296, 1] = -np.inf
    rays[296:304, 3:] *= 1e-20
    rays[304:312, 3:] *= 1e20
    rays[312:320, :3] *= 1e16
    check(engine, rsh, sc, rays)


def test_moved_objects(engine, rsh):
    """The tree follows the objects: a frame after an update equals the frame
    of the exhaustive kernel on the same engine."""
    sc = rsh.scenes.config1_scene(boxes=120)
    cam = rsh.scenes.config1_camera(97, 61)
    cfg = rsh.config.config1(97, 61).with_scene_bounds(sc)
    engine.load_scene(sc)
    K = sc.object_total
    rng = np.random.default_rng(8)
    for _ in range(2):
        m = np.tile(np.eye(4, dtype=np.float32), (K, 1, 1))
        n, s = m.copy(), m.copy()
        m[1:, :3, 3] = rng.uniform(-20.0, 20.0, (K - 1, 3))
        engine.update_objects(m, n, s)
        engine.render(cam, cfg, flags=engine.KEEP_PASSES)
        got = [engine.pass_hits(i) for i in range(engine.stats.pass_count)]
        engine.render(cam, dataclasses.replace(cfg, traversal_prefilter=1), flags=engine.KEEP_PASSES)
        assert len(got) == engine.stats.pass_count
        for i, g in enumerate(got):
            np.testing.assert_array_equal(g, engine.pass_hits(i))


def test_serving_mix_on_the_soup(engine, rsh):
    """Overlapping triangles: the tree's longest paths."""
    sc = rsh.scenes.soup_scene(triangles=30_000)
    for mix in (queries.PRIMARY, queries.DIFFUSE):
        rays, _, _ = queries.make_query(sc, mix, 5003, np.random.default_rng(9))
        check(engine, rsh, sc, rays)


@pytest.mark.parametrize("T", [2047, 2048, 2049, 2051, 32768, 32769])
def test_merge_groups(engine, rsh, T):
    """Around the triangles of one merging workgroup, and of the sixteen whose
    clusters the next launch takes."""
    rng = np.random.default_rng(T)
    sc = make_scene(rsh, soup(rng, T, size=2.0), 97)
    check(engine, rsh, sc, rays_at(rng, sc, 501))


@pytest.mark.parametrize("kind", ["equal", "nested", "grid", "far"])
def test_merge_orders(engine, rsh, kind):
    """Clusters that offer no clear best partner: equal triangles, each inside
    the next (one pair a round, so the rounds run out), a regular grid, and
    coordinates whose surfaces overflow."""
    rng = np.random.default_rng(3)
    T = 2300
    if kind == "equal":
        tris = np.repeat(soup(rng, 1), T, 0)
    elif kind == "nested":
        c = soup(rng, 1, size=1.0)
        mid = c.mean(1, keepdims=True)
        tris = mid + (c - mid) * (1.006 ** np.arange(T))[:, None, None] * 1e-2
    elif kind == "grid":
        g = np.stack(np.meshgrid(np.arange(48), np.arange(48), indexing="ij"), -1).reshape(-1, 2)[:T]
        base = np.concatenate([g, np.zeros((T, 1))], 1)[:, None] * 2.0 + 50.0
        tris = base + np.array([[0, 0, 0], [2, 0, 0], [0, 2, 0]])[None]
    else:
        tris = soup(rng, T)
        tris[::3] *= 1e15
    sc = make_scene(rsh, tris.astype(np.float32), 50)
    check(engine, rsh, sc, rays_at(rng, sc, 501))


@pytest.mark.parametrize("n", [32767, 32768, 32769])
def test_wave_and_quad(engine, rsh, n):
    """A wave per ray up to 32768 rays and a quad per ray beyond: scenes and
    rays outside the ordinary on both sides of the line."""
    rng = np.random.default_rng(n)
    s = 0.5 ** np.repeat(np.arange(9), 40)[:, None, None]
    nested = (50.0 + 100.0 * s * (np.asarray([[0.1, 0.1, 0.1], [1.0, 0.1, 0.2], [0.1, 1.0, 0.3]])
                                  + 0.01 * rng.random((360, 3, 3)))).astype(np.float32)
    for tris in (soup(rng, 513), nested, np.repeat(soup(rng, 1), 300, 0)):
        sc = make_scene(rsh, tris, 30)
        rays = rays_at(rng, sc, n)
        rays[0:64, 3:] *= 1e6
        rays[128:192, 3:] = np.eye(3, dtype=np.float32)[rng.integers(3, size=64)]
        rays[256:264, 3:] = 0.0
        rays[264:272, 3:] = np.nan
        rays[280:288, 0] = np.nan
        rays[296:304, 3:] *= 1e-20
        rays[312:320, :3] *= 1e16
        check(engine, rsh, sc, rays)
        if len(tris) == 513:
            check(engine, rsh, sc, rays, hit_mode=1)
            check(engine, rsh, sc, rays, algorithm=1)


def test_wave_stack_full(engine, rsh):
    """Equal boxes by the thousand: a ray's stack fills and it takes every
    triangle in turn."""
    rng = np.random.default_rng(4)
    sc = make_scene(rsh, np.repeat(soup(rng, 1), 20_000, 0), 500)
    rays = rays_at(rng, sc, 64)
    rays[:32, 3:] = (sc.tri_pos[:3, :3].mean(0) - rays[:32, :3])
    check(engine, rsh, sc, rays)


@pytest.mark.parametrize("w,h", [(127, 129), (128, 128), (145, 113)])
def test_wave_camera_passes(engine, rsh, w, h):
    """Camera passes on both sides of their line (16384 rays)."""
    sc = rsh.scenes.config0_scene()
    cfg = rsh.config.config0(w, h).with_scene_bounds(sc)
    engine.load_scene(sc)
    cam = rsh.scenes.config0_camera(w, h)
    engine.render(cam, cfg, flags=engine.KEEP_PASSES)
    got = [engine.pass_hits(i) for i in range(engine.stats.pass_count)]
    engine.render(cam, dataclasses.replace(cfg, traversal_prefilter=1), flags=engine.KEEP_PASSES)
    for i, g in enumerate(got):
        np.testing.assert_array_equal(g, engine.pass_hits(i))


def tiles(n):
    """A floor of n x n tiles of one unit, two triangles each."""
    g = np.stack(np.meshgrid(np.arange(n), np.arange(n), indexing="ij"), -1).reshape(-1, 1, 2).astype(np.float64)
    g = np.insert(g, 1, 0.0, axis=2)
    return np.concatenate([g + np.array([[0, 0, 0], [1, 0, 0], [0, 0, 1]]),
                           g + np.array([[1, 0, 1], [0, 0, 1], [1, 0, 0]])])


@pytest.mark.parametrize("n", [1501, 32783])
@pytest.mark.parametrize("away", [0.0, 2e4, 3e5, 1e6, 1e9])
def test_scenes_far_from_the_origin(engine, rsh, n, away):
    """Small scenes and their rays translated, for the wave and the quad kernel.
    The reference is the kernel with the pre-tests (traversal_prefilter 2): that
    far out a triangle's sphere, rounded to its coordinates, need not hold the
    triangle, and the pre-tests take it at its word, as the tree does."""
    rng = np.random.default_rng(int(away))
    for tris in (tiles(10), soup(rng, 400, spread=10.0, size=1.0) - 50.0, soup(rng, 2000, spread=100.0)):
        sc = make_scene(rsh, (tris + away * np.array([1.0, -0.7, 0.4])).astype(np.float32), 50)
        rays = rays_at(rng, sc, n)
        cfg = qcfg(rsh, sc)
        engine.load_scene(sc)
        tmax = np.full(n, 60.0, np.float32)
        for kind in (0, 1):
            got = engine.trace(rays, kind, cfg, tmax=tmax)
            want = engine.trace(rays, kind, dataclasses.replace(cfg, traversal_prefilter=2), tmax=tmax)
            np.testing.assert_array_equal(got, want)
            if away <= 3e5:
                assert (want != (np.uint64(0xFFFFFFFFFFFFFFFF) if kind == 0 else 0)).sum() > n // 10


# Both traversal kernels at sizes of either's choosing (rsh_selfcheck_tree_walk):
# above, passes of up to 32768 rays walk a wave per ray only.
QUAD, WAVE, NO_TREE = 1, 2, 3


@pytest.fixture
def walk(engine):
    def use(kernel, small_stack=False):
        assert engine.L.rsh_selfcheck_tree_walk(engine.h, kernel, int(small_stack)) == 0
    yield use
    use(0)


@pytest.mark.parametrize("T", [1, 2, 4, 5, 8, 9, 63, 65, 513, 2047, 2049, 4099, 32769])
def test_quad_scene_sizes(engine, rsh, walk, T):
    rng = np.random.default_rng(T)
    walk(QUAD)
    sc = make_scene(rsh, soup(rng, T, size=2.0), 7)
    check(engine, rsh, sc, rays_at(rng, sc, 1501))


@pytest.mark.parametrize("n", [1, 3, 15, 16, 17, 31, 64, 65, 1025, 1040])
def test_quad_ray_counts(engine, rsh, walk, n):
    rng = np.random.default_rng(n)
    sc = make_scene(rsh, soup(rng, 777), 50)
    walk(QUAD)
    check(engine, rsh, sc, rays_at(rng, sc, n))


@pytest.mark.parametrize("kernel,n", [(QUAD, 2003), (WAVE, 40_001)])
@pytest.mark.parametrize("variant", [dict(algorithm=1), dict(hit_mode=1), dict(depth=1), dict(depth=3, branch=4),
                                     dict(depth=4, leaf=4, branch=3), dict(leaf=32, branch=2), dict(key_mode=0),
                                     dict(triangle_batch=512), dict(cone_mode=0)])
def test_options_in_both_kernels(engine, rsh, walk, kernel, n, variant):
    rng = np.random.default_rng(3)
    sc = make_scene(rsh, soup(rng, 3001), 64)
    walk(kernel)
    check(engine, rsh, sc, rays_at(rng, sc, n), **variant)


@pytest.mark.parametrize("kernel", [QUAD, WAVE])
def test_outside_the_ordinary_in_both_kernels(engine, rsh, walk, kernel):
    walk(kernel)
    test_scenes_outside_the_ordinary(engine, rsh)
    test_rays_outside_the_ordinary(engine, rsh)
    for kind in ("equal", "nested", "grid", "far"):
        test_merge_orders(engine, rsh, kind)
    test_serving_mix_on_the_soup(engine, rsh)
    test_moved_objects(engine, rsh)


@pytest.mark.parametrize("kernel", [QUAD, WAVE])
@pytest.mark.parametrize("variant", [dict(), dict(hit_mode=1), dict(algorithm=1)])
def test_full_stacks(engine, rsh, walk, kernel, variant):
    """Stacks of a few entries.  In the scene of equal triangles every box of
    the tree is the same, so a ray that meets one meets all, and three levels
    (more than 64 triangles) fill either stack: it then takes every triangle in
    turn.  The others fill it for some rays."""
    rng = np.random.default_rng(4)
    one = soup(rng, 1)
    for tris in (np.repeat(one, 300, 0), soup(rng, 3001), soup(rng, 400, size=30.0)):
        sc = make_scene(rsh, tris, 50)
        rays = rays_at(rng, sc, 1003)
        rays[:64, 3:] = sc.tri_pos[:3, :3].mean(0) - rays[:64, :3]      # through the first triangle
        walk(kernel, small_stack=True)
        want = check(engine, rsh, sc, rays, **variant)
        if len(tris) == 300:
            assert want[:64].any()
    walk(kernel, small_stack=True)
    test_moved_objects(engine, rsh)


def test_frames_without_the_tree(engine, rsh, walk):
    """A scene too large for the tree: the automatic traversal's other kernels
    (front-to-back camera pass, work list, ray masks) on the full-size atrium
    frame, against the tree's frame."""
    sc = rsh.scenes.config2_scene()
    cfg = rsh.config.config2().with_scene_bounds(sc)
    cam = rsh.scenes.config2_camera(cfg.width, cfg.height)
    engine.load_scene(sc)
    engine.render(cam, cfg, flags=engine.KEEP_PASSES)
    modes = list(engine.stats.pass_mode[:engine.stats.pass_count])
    got = [engine.pass_hits(i) for i in range(engine.stats.pass_count)]
    px = engine.pixels()
    walk(NO_TREE)
    engine.render(cam, cfg, flags=engine.KEEP_PASSES)
    assert modes == [3] * len(modes) and 3 not in engine.stats.pass_mode[:engine.stats.pass_count]
    np.testing.assert_array_equal(px, engine.pixels())
    for i, g in enumerate(got):
        np.testing.assert_array_equal(g, engine.pass_hits(i))
    check(engine, rsh, rsh.scenes.soup_scene(triangles=5000),
          queries.make_query(rsh.scenes.soup_scene(triangles=5000), queries.DIFFUSE, 5003, np.random.default_rng(1))[0])


@pytest.mark.parametrize("n", [131_071, 131_072, 131_073])
def test_wave_limit_of_overlapping_scenes(engine, rsh, n):
    """Where a line through the scene meets many triangles' boxes, passes of up to 131072
    rays walk a wave per ray."""
    rng = np.random.default_rng(n)
    sc = make_scene(rsh, soup(rng, 2000, size=30.0), 50)
    check(engine, rsh, sc, rays_at(rng, sc, n))


def query_ms(engine, rsh, rays, cfg):
    import time
    dev = rsh.DeviceArray.from_host(rays)
    out, desc = rsh.DeviceArray((len(rays),), np.uint64), rsh.config_desc(cfg)
    times = []
    for _ in range(9):
        t = time.perf_counter()
        assert engine.L.rsh_engine_trace(engine.h, dev.ptr, None, None, len(rays), 0, rsh.C.byref(desc), out.ptr, 0,
                                         None) == 0
        times.append(time.perf_counter() - t)
    return 1e3 * float(np.median(times))


@pytest.mark.parametrize("scene,n", [("soup", 33_000), ("soup_of_10k", 33_000), ("large", 33_000), ("large", 100_000)])
def test_overlapping_scenes_are_no_slower_than_without_the_tree(engine, rsh, walk, scene, n):
    """Rays that meet hundreds of overlapping triangles: measured at 0.45 to
    0.6 of the time of the kernels that test every candidate; with a quad a ray
    from 32769 rays on they took 1.1 to 2 times as long."""
    rng = np.random.default_rng(n)
    if scene == "large":
        sc = make_scene(rsh, soup(rng, 2000, size=30.0), 100)
        rays = rays_at(rng, sc, n)
    else:
        sc = rsh.scenes.soup_scene(triangles=100_000 if scene == "soup" else 10_000)
        rays = queries.make_query(sc, queries.PRIMARY if scene == "soup" else queries.DIFFUSE, n, rng)[0]
    engine.load_scene(sc)
    cfg = qcfg(rsh, sc)
    tree = query_ms(engine, rsh, rays, cfg)
    walk(NO_TREE)
    assert tree < query_ms(engine, rsh, rays, cfg)


def frame_ms(engine, cam, cfg, flags):
    import time
    times = []
    for _ in range(20):
        t = time.perf_counter()
        engine.render(cam, cfg, flags=flags)
        times.append(time.perf_counter() - t)
    return 1e3 * min(times)


def test_a_frames_shadow_rays_keep_a_quad_each(engine, rsh, walk):
    """90,000 of them in a 512x512 frame of the soup: they end at the first
    occluder, so a wave each is the slower by 13 % of the frame."""
    sc = rsh.scenes.soup_scene()
    engine.load_scene(sc)
    cfg = dataclasses.replace(rsh.config.config0(512, 512), bounces=0, bounce_shadows=0).with_scene_bounds(sc)
    cam = rsh.scenes.random_view(np.random.default_rng(1), 512, 512)
    auto = frame_ms(engine, cam, cfg, 0)
    assert 60_000 < engine.stats.pass_rays[1] < 131_072
    walk(QUAD)
    assert auto < 1.06 * frame_ms(engine, cam, cfg, 0)


@pytest.mark.parametrize("kernel", [0, QUAD, WAVE])
def test_captured_frames_in_both_kernels(engine, rsh, walk, kernel):
    """Frames replayed from a graph keep their sizes on the device: fewer rays
    than the launches cover, and other cameras than the captured one."""
    sc = rsh.scenes.config1_scene(boxes=120)
    engine.load_scene(sc)
    w, h = 71, 53
    cfg = dataclasses.replace(rsh.config.config1(w, h), bounces=2, bounce_shadows=1).with_scene_bounds(sc)
    rng = np.random.default_rng(2)
    cams = [rsh.scenes.random_view(rng, w, h) for _ in range(4)]
    want = []
    for cam in cams:
        engine.render(cam, dataclasses.replace(cfg, traversal_prefilter=1))
        want.append(engine.pixels())
    walk(kernel)
    for i in (0, 0, 1, 2, 3, 0):
        engine.render(cams[i], cfg, flags=engine.GRAPH)
        np.testing.assert_array_equal(engine.pixels(), want[i])
    assert engine.stats.graph_replayed


@pytest.mark.parametrize("bounces,shadows", [(0, 0), (2, 1)])
def test_small_captured_frames_are_no_slower_than_without_the_tree(engine, rsh, walk, bounces, shadows):
    """Measured at a third of the time without the tree; with a quad a ray they
    took 1.3 times as long."""
    sc = rsh.scenes.soup_scene()
    engine.load_scene(sc)
    cfg = dataclasses.replace(rsh.config.config0(64, 64), bounces=bounces, bounce_shadows=shadows).with_scene_bounds(sc)
    cam = rsh.scenes.random_view(np.random.default_rng(3), 64, 64)
    tree = frame_ms(engine, cam, cfg, engine.GRAPH)
    walk(NO_TREE)
    assert tree < frame_ms(engine, cam, cfg, engine.GRAPH)


def test_large_camera_passes_of_overlapping_scenes(engine, rsh, walk):
    """Their camera pass takes the kernels that share candidates among
    neighbours (mode 1 or 2), the others the tree (3): the same hits, eager and
    replayed, and no slower than without the tree (measured at 0.84, replayed
    0.95; with the tree for every pass 1.45)."""
    sc = rsh.scenes.soup_scene()
    cfg = rsh.config.config0(1024, 1024).with_scene_bounds(sc)
    cam = rsh.scenes.random_view(np.random.default_rng(1), 1024, 1024)
    engine.load_scene(sc)
    engine.render(cam, cfg, flags=engine.KEEP_PASSES)
    modes = list(engine.stats.pass_mode[:engine.stats.pass_count])
    assert modes[0] in (1, 2) and set(modes[1:]) == {3}
    got, px = [engine.pass_hits(i) for i in range(len(modes))], engine.pixels()
    for _ in range(3):
        engine.render(cam, cfg, flags=engine.GRAPH)
        np.testing.assert_array_equal(engine.pixels(), px)
    auto = [frame_ms(engine, cam, cfg, fl) for fl in (0, engine.GRAPH)]
    walk(QUAD)
    engine.render(cam, cfg, flags=engine.KEEP_PASSES)
    assert list(engine.stats.pass_mode[:len(modes)]) == [3] * len(modes)
    for i, g in enumerate(got):
        np.testing.assert_array_equal(g, engine.pass_hits(i))
    walk(NO_TREE)
    for ms, fl in zip(auto, (0, engine.GRAPH)):
        assert ms < 1.1 * frame_ms(engine, cam, cfg, fl)


@pytest.mark.parametrize("scene", ["config0", "config1", "config2"])
def test_camera_passes_of_other_scenes_keep_the_tree(engine, rsh, scene):
    sc = getattr(rsh.scenes, scene + "_scene")()
    cfg = rsh.config.config0(1920, 1080).with_scene_bounds(sc)
    engine.load_scene(sc)
    engine.render(getattr(rsh.scenes, scene + "_camera")(1920, 1080), cfg)
    assert set(engine.stats.pass_mode[:engine.stats.pass_count]) == {3}


def test_overlap_is_measured_again_after_an_update(engine, rsh):
    """Objects pulled apart, and put back: the camera pass's kernels follow."""
    sc = rsh.scenes.soup_scene()
    cfg = rsh.config.config0(1024, 1024).with_scene_bounds(sc)
    cam = rsh.scenes.random_view(np.random.default_rng(1), 1024, 1024)
    engine.load_scene(sc)
    K = sc.object_total
    eye = np.tile(np.eye(4, dtype=np.float32), (K, 1, 1))
    apart = eye.copy()
    apart[:, :3, 3] = np.random.default_rng(2).uniform(-5e4, 5e4, (K, 3))
    for m, tree in ((apart, True), (eye, False)):
        engine.update_objects(m, eye, eye)
        engine.render(cam, cfg)
        assert (engine.stats.pass_mode[0] == 3) == tree
        px = engine.pixels()
        engine.render(cam, dataclasses.replace(cfg, traversal_prefilter=2))
        np.testing.assert_array_equal(engine.pixels(), px)


def test_tree_given_back_for_memory(rsh):
    """Frames, queries, replays and object updates on an engine that has given
    back the tree's construction buffers, and then the tree: the same results,
    and the next load builds it again."""
    sc = rsh.scenes.config1_scene(boxes=120)
    cam = rsh.scenes.config1_camera(97, 61)
    cfg = rsh.config.config1(97, 61).with_scene_bounds(sc)
    K = sc.object_total
    rng = np.random.default_rng(8)
    eye = np.tile(np.eye(4, dtype=np.float32), (K, 1, 1))
    moves = []
    for _ in range(3):
        m = eye.copy()
        m[1:, :3, 3] = rng.uniform(-20.0, 20.0, (K - 1, 3))
        moves.append(m)
    rays = rays_at(rng, sc, 501)
    steps = [None, moves[0], None, moves[1], moves[2]]

    def results(e, m):
        if m is not None:
            e.update_objects(m, eye, eye)
        e.render(cam, cfg)
        out = [e.pixels()]
        mode = e.stats.pass_mode[0]
        for _ in range(2):
            e.render(cam, cfg, flags=e.GRAPH)
            out.append(e.pixels())
        return out + [e.trace(rays, 0, cfg)], mode

    e, ref = rsh.Engine(0), rsh.Engine(0)
    try:
        e.load_scene(sc)
        ref.load_scene(sc)
        # the construction buffers after the first step (an update takes them
        # again), both parts after the second
        for i, m in enumerate(steps):
            got, mode = results(e, m)
            want, _ = results(ref, m)
            for g, w in zip(got, want):
                np.testing.assert_array_equal(g, w)
            assert (mode == 3) == (i < 2), (i, mode)
            if i == 0:
                assert e.L.rsh_selfcheck_give_back(e.h) == 0
            elif i == 1:
                assert e.L.rsh_selfcheck_give_back(e.h) == 0
                assert e.L.rsh_selfcheck_give_back(e.h) == 0
                assert e.L.rsh_selfcheck_give_back(e.h) != 0
        e.load_scene(sc)
        assert results(e, None)[1] == 3
    finally:
        e.close()
        ref.close()
