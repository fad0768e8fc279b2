"""The trimming stage's compaction and the inclusive scan of the warm-up stage,
staged through LDS, at the edges of a tile of 4096."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 4095, 4096, 4097, 8191, 12289])
@pytest.mark.parametrize("live", [0.0, 0.03, 0.6, 1.0])
def test_trim(rsh, n, live):
    L = rsh.lib()
    rng = np.random.default_rng(n)
    flags = (rng.random(n) >= live).astype(np.uint32)
    keys, vals = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32), rng.permutation(n).astype(np.uint32)
    df, dk, dv = (rsh.DeviceArray.from_host(a) for a in (flags, keys, vals))
    scan = rsh.DeviceArray((n,), np.uint32)
    ok, ov = rsh.DeviceArray.from_host(np.full(n + 1, 7, np.uint32)), rsh.DeviceArray.from_host(np.full(n + 1, 7, np.uint32))
    total = C.c_uint32(99)
    L.RayTrimmingWrapper(dk.ptr, dv.ptr, n, 1, 1, df.ptr, scan.ptr, ok.ptr, ov.ptr, C.byref(total))
    assert L.rsh_compat_status() == 0, L.rsh_compat_error()
    keep = flags == 0
    m = int(keep.sum())
    assert total.value == m
    np.testing.assert_array_equal(ok.download()[:m], keys[keep])
    np.testing.assert_array_equal(ov.download()[:m], vals[keep])
    assert (ok.download()[m:] == 7).all() and (ov.download()[m:] == 7).all()


GUARD = 0xA5A5A5A5


def guarded(rsh, n):
    return rsh.DeviceArray.from_host(np.full(n + 64, GUARD, np.uint32))


def read(dev, n):
    out = dev.download()
    assert (out[n:] == GUARD).all()
    return out[:n]


EDGES = [1, 2, 15, 16, 17, 255, 256, 4095, 4096, 4097, 8191, 8193, 12289, 131073]


@pytest.mark.parametrize("n", EDGES)
@pytest.mark.parametrize("tri", [1, 3])
def test_inclusive_scan(rsh, n, tri):
    """The warm-up stage's scan of its flags.  One object of `tri` triangles, at
    a node's flag their count where it meets the node (a cone of half pi does,
    a line that passes 50 units off does not)."""
    rng = np.random.default_rng(n + tri)
    meets = rng.random(n) < 0.6
    nodes = np.zeros((n, 2, 4), np.float32)
    nodes[:, 1] = (1.0, 0.0, 0.0, 0.0)
    nodes[meets, 1, 3] = np.float32(np.float32(3.1415927) / np.float32(2.0))
    sphere = np.array([[0.0, 50.0, 0.0], [1e-3, 0.0, tri - 1]], np.float32)
    total = n * tri
    flags, scan, hits, thits = (guarded(rsh, total) for _ in range(4))
    pos = rsh.DeviceArray.from_host(np.zeros((3 * tri, 4), np.float32))
    h, sph = rsh.DeviceArray.from_host(nodes), rsh.DeviceArray.from_host(sphere)
    ctx = rsh.Context(0)
    try:
        ctx.configure(1, 1, 1, 0)
        count, room = C.c_uint32(0), C.c_uint32(total)
        ctx.stage("hierarchy_traversal_warmup", None, h.ptr, sph.ptr, pos.ptr, 1, n, tri, 0, flags.ptr, scan.ptr,
                  hits.ptr, thits.ptr, C.byref(count), C.byref(room))
    finally:
        ctx.close()
    want = np.zeros((n, tri), np.uint32)
    want[:, 0] = meets * tri
    np.testing.assert_array_equal(read(scan, total), np.cumsum(want.ravel(), dtype=np.uint32))
    for b in (flags, hits, thits):
        read(b, total)


@pytest.mark.parametrize("n", EDGES)
def test_exclusive_scan(rsh, n):
    """The decompression stage's scan of its chunk sizes, their number on the
    device (a count on the host takes one workgroup up to 131072)."""
    rng = np.random.default_rng(n)
    sizes = rng.integers(1, 6, n).astype(np.uint32)
    bases = (np.cumsum(sizes) - sizes).astype(np.uint32)
    order = rng.permutation(n).astype(np.uint32)
    N = int(sizes.sum())
    keys, vals = rng.integers(0, 1 << 32, N, dtype=np.uint64).astype(np.uint32), rng.permutation(N).astype(np.uint32)
    d = [rsh.DeviceArray.from_host(a) for a in (bases, sizes, keys[bases[order]], order, keys, vals)]
    total = rsh.DeviceArray.from_host(np.array([n], np.uint32))
    skeleton, scan, ok, ov = guarded(rsh, n), guarded(rsh, n), guarded(rsh, N), guarded(rsh, N)
    ctx = rsh.Context(0)
    try:
        ctx.configure(1, 2, 8, 0)
        ctx.stage("ray_decompression", None, *[x.ptr for x in d], skeleton.ptr, scan.ptr, n, total.ptr, ok.ptr, ov.ptr)
    finally:
        ctx.close()
    np.testing.assert_array_equal(read(skeleton, n), sizes[order])
    np.testing.assert_array_equal(read(scan, n), np.cumsum(sizes[order]) - sizes[order])
    rays = np.concatenate([np.arange(bases[k], bases[k] + sizes[k]) for k in order])
    np.testing.assert_array_equal(read(ok, N), keys[rays])
    np.testing.assert_array_equal(read(ov, N), vals[rays])
