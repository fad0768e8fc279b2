"""Sorting a pass's rays directly against sorting its packets, and the sort's
small tiles: the same order, at the edges of the tiles and of the rule that
picks between the two."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTERS = ("pass_rays", "pass_chunks", "pass_pairs_top", "pass_pairs_leaf", "pass_ray_tests")


def counters(st):
    return {f: list(getattr(st, f)) for f in COUNTERS}


@pytest.mark.parametrize("n", [1, 1023, 1024, 1025, 8 * 1024, 8 * 1024 + 1, 128 * 1024, 128 * 1024 + 1])
@pytest.mark.parametrize("bits", [8, 27, 32])
def test_sort_tiles(rsh, n, bits):
    L = rsh.lib()
    rng = np.random.default_rng(n + bits)
    keys = rng.integers(0, 1 << bits, n, dtype=np.uint64).astype(np.uint32)
    keys[: n // 3] = keys[0]            # one long run: a digit that fills whole tiles
    vals = np.arange(n, dtype=np.uint32)
    dk, dv = rsh.DeviceArray.from_host(keys), rsh.DeviceArray.from_host(vals)
    ok, ov = rsh.DeviceArray((n,), np.uint32), rsh.DeviceArray((n,), np.uint32)
    L.rsh_sort_pairs(dk.ptr, dv.ptr, n, bits, ok.ptr, ov.ptr)
    assert L.rsh_compat_status() == 0, L.rsh_compat_error()
    order = np.argsort(keys, kind="stable")
    np.testing.assert_array_equal(ok.download(), keys[order])
    np.testing.assert_array_equal(ov.download(), vals[order])


@pytest.mark.parametrize("n,runs", [(1, 1), (4097, 50), (1 << 20, 300), ((1 << 20) + 1, 300), ((1 << 20) + 1, 1 << 20)])
def test_rays_and_packets(rsh, n, runs):
    """A query's pair and test counts (functions of the sorted order) with the
    rays sorted (where the rule says so) and with its packets sorted (the order
    read-back, bit 6), and equal results."""
    sc = rsh.scenes.config0_scene()
    cfg = dataclasses.replace(rsh.config.config0(8, 8), cell_bits=4, dir_bits=8).with_scene_bounds(sc)
    rng = np.random.default_rng(n + runs)
    o = rng.uniform(sc.bounds_min, sc.bounds_max, (runs, 3))
    d = rng.normal(size=(runs, 3))
    rays = np.repeat(np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1), -(-n // runs), 0)[:n]
    rays = rays.astype(np.float32)
    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        a = e.trace(rays, 0, cfg, flags=2)
        ca = counters(e.stats)
        b = e.trace(rays, 0, cfg, flags=2 | 64)
        assert ca == counters(e.stats)
        assert ca["pass_rays"][0] == n
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(e.trace(rays, 0, cfg), b)
    finally:
        e.close()


def test_frame_passes(rsh):
    """The passes of a frame, whose slots are only partly live."""
    sc = rsh.scenes.config0_scene()
    cfg = rsh.config.config0(203, 149).with_scene_bounds(sc)
    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        cam = rsh.scenes.config0_camera(203, 149)
        ca = counters(e.render(cam, cfg, flags=2))
        pa = e.pixels()
        assert ca == counters(e.render(cam, cfg, flags=2 | 64))
        np.testing.assert_array_equal(pa, e.pixels())
    finally:
        e.close()


@pytest.mark.parametrize("leaf,branch", [(8, 8), (4, 1), (2, 256), (64, 8), (16, 2), (8, 3)])
def test_levels(rsh, oracle, leaf, branch):
    """Records and both hierarchy levels in one launch (fan-outs whose product
    divides 512; the last pair takes a launch a level), at ray counts about the
    block's 512, against the oracle bit for bit."""
    sc = rsh.scenes.config0_scene()
    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        for w, h in ((2, 1), (3, 3), (9, 7), (73, 7), (64, 8), (27, 19), (41, 25)):
            cfg = dataclasses.replace(rsh.config.config0(w, h), leaf=leaf, branch=branch).with_scene_bounds(sc)
            cam = rsh.scenes.config0_camera(w, h)
            e.render(cam, cfg, flags=e.KEEP_ORDER)
            ofr = oracle.render(sc, cam, cfg, keep_order=True, keep_hits=False)
            for i, op in enumerate(ofr.passes):
                assert e.stats.pass_rays[i] == op["rays"]
                if op["rays"]:
                    g = e.pass_order(i)["nodes"]
                    np.testing.assert_array_equal(g.view(np.uint32), op["nodes"][:len(g)].view(np.uint32),
                                                  err_msg=f"{w}x{h}, pass {i}")
    finally:
        e.close()


@pytest.mark.parametrize("n", [1, 2, 63, 65, 1023, 1025, 4095, 4096, 4097, 8192, 8193, 16383, 16384, 16385])
@pytest.mark.parametrize("bits", [(4, 8), (3, 4), (4, 9)])
def test_small_passes(rsh, n, bits):
    """Passes sorted by one workgroup, at its sizes' edges: the pair and test
    counts of the packets' path, and equal results; few and many equal keys."""
    sc = rsh.scenes.config0_scene()
    cell, dirs = bits
    cfg = dataclasses.replace(rsh.config.config0(8, 8), cell_bits=cell, dir_bits=dirs).with_scene_bounds(sc)
    rng = np.random.default_rng(n)
    o = rng.uniform(sc.bounds_min, sc.bounds_max, (n, 3))
    d = rng.normal(size=(n, 3))
    rays = np.concatenate([o, d / np.linalg.norm(d, axis=1, keepdims=True)], 1).astype(np.float32)
    rays[: n // 2] = rays[0]
    tmax = np.full(n, 60.0, np.float32)
    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        for kind in (0, 1):
            a = e.trace(rays, kind, cfg, tmax=tmax, flags=2)
            ca = counters(e.stats)
            b = e.trace(rays, kind, cfg, tmax=tmax, flags=2 | 64)
            assert ca == counters(e.stats)
            np.testing.assert_array_equal(a, b)
    finally:
        e.close()


@pytest.mark.parametrize("w,h", [(1, 1), (31, 33), (64, 64), (127, 129), (128, 128)])
def test_small_frames(rsh, w, h):
    """Frames whose shadow and reflection passes (partly live) fit one workgroup."""
    sc = rsh.scenes.config0_scene()
    cfg = rsh.config.config0(w, h).with_scene_bounds(sc)
    cam = rsh.scenes.config0_camera(w, h)
    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        ca = counters(e.render(cam, cfg, flags=2))
        pa = e.pixels()
        assert ca == counters(e.render(cam, cfg, flags=2 | 64))
        np.testing.assert_array_equal(pa, e.pixels())
        e.render(cam, cfg)
        np.testing.assert_array_equal(pa, e.pixels())
    finally:
        e.close()


@pytest.mark.parametrize("w,h", [(2048, 1024), (2045, 1025), (2049, 1024), (1025, 1023)])
def test_levels_of_large_passes(rsh, w, h):
    """Camera passes about the 2^21 rays up to which both levels come from one
    launch: the nodes of a hierarchy of three levels, made with a launch each,
    start with the same two."""
    sc = rsh.scenes.config0_scene()
    cam = rsh.scenes.config0_camera(w, h)
    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        nodes = []
        for depth in (2, 3):
            cfg = dataclasses.replace(rsh.config.config0(w, h), depth=depth, bounces=0).with_scene_bounds(sc)
            e.render(cam, cfg, flags=e.KEEP_ORDER)
            nodes.append(e.pass_order(0)["nodes"].view(np.uint32))
        n0 = -(-w * h // 8)
        assert len(nodes[0]) == 2 * (n0 + -(-n0 // 8)) < len(nodes[1])
        np.testing.assert_array_equal(nodes[0], nodes[1][:len(nodes[0])])
    finally:
        e.close()
