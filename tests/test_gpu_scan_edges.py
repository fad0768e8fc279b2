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
