"""The surface records' read-back (colours from the material tables) against
the oracle's planes, also after another scene was loaded, and frames whose
pixels miss."""
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (37, 29), (64, 48)])
def test_read_back(rsh, oracle, w, h):
    sc = rsh.scenes.config0_scene()
    # part of the view looks out of the room
    keep = slice(0, 3 * int(sc.object_spheres[0][5] + 1))
    part = dataclasses.replace(sc, tri_pos=sc.tri_pos[keep], tri_nrm=sc.tri_nrm[keep], tri_mat=sc.tri_mat[keep],
                               object_spheres=sc.object_spheres[:1])
    cam = rsh.scenes.config0_camera(w, h)
    e = rsh.Engine(0)
    try:
        for s in (sc, part, sc):
            cfg = rsh.config.config0(w, h).with_scene_bounds(s)
            e.load_scene(s)
            e.render(cam, cfg)
            want = oracle.render(s, cam, cfg).gbuffer
            got = e.gbuffer()
            other = dataclasses.replace(s, mat_diffuse=s.mat_diffuse[::-1] * 0.5,
                                        mat_specular=s.mat_specular[::-1] * 0.25)
            e.load_scene(other)
            again = e.gbuffer()
            e.load_scene(other)
            third = e.gbuffer()
            for k in ("dif", "spec"):
                np.testing.assert_array_equal(got[k], np.asarray(want[k]).reshape(got[k].shape), err_msg=k)
            assert not got["nrm"][:, 3].view(np.uint32).any()
            for k in ("pos", "nrm", "dif", "spec"):
                np.testing.assert_array_equal(again[k], got[k], err_msg=k)
                np.testing.assert_array_equal(third[k], got[k], err_msg=k)
    finally:
        e.close()


def test_only_a_completed_frames_records_are_read(rsh):
    """A read-back without a frame's records behind it is refused: before any
    frame, past the frame's pixels, and after a larger query has reallocated
    the buffers.  A query that leaves them in place leaves them readable, and a
    replayed frame writes them as an eager one does."""
    sc = rsh.scenes.config0_scene()
    cfg = rsh.config.config0(48, 32).with_scene_bounds(sc)
    cam = rsh.scenes.config0_camera(48, 32)
    rng = np.random.default_rng(0)

    def query(n):
        rays = np.concatenate([rng.uniform(sc.bounds_min, sc.bounds_max, (n, 3)), rng.normal(size=(n, 3))], 1)
        e.trace(rays.astype(np.float32), 0, cfg)

    def read(n, planes=("dif", "spec", "pos", "nrm")):
        out = {k: np.empty((max(n, 1), 4), np.float32) for k in planes}
        ptr = [out[k].ctypes.data_as(rsh.PF) if k in planes else None for k in ("dif", "spec", "pos", "nrm")]
        rc = e.L.rsh_engine_read_gbuffer(e.h, *ptr, n)
        assert rc in (0, 1), rc                      # RSH_OK, RSH_INVALID_ARG
        return out if rc == 0 else None

    e = rsh.Engine(0)
    try:
        e.load_scene(sc)
        query(100)
        assert read(0) is not None                   # nothing asked for, nothing read
        for planes in (("pos",), ("nrm",), ("dif",), ("spec",)):
            assert read(1, planes) is None
        e.render(cam, cfg)
        want = e.gbuffer()
        query(48 * 32)                               # fits: the records stand
        got = read(48 * 32)
        for k, v in want.items():
            np.testing.assert_array_equal(got[k], v, err_msg=k)
        big, bcam = rsh.config.config0(96, 64).with_scene_bounds(sc), rsh.scenes.config0_camera(96, 64)
        e.render(bcam, big)
        e.render(cam, cfg)
        query(96 * 64)
        assert read(48 * 32) is not None and read(48 * 32 + 1) is None
        query(96 * 64 + 1)                           # reallocates the buffers
        assert read(1) is None
        e.load_scene(sc)
        assert read(1) is None
        for _ in range(3):                           # captured, then replayed
            e.render(cam, cfg, flags=e.GRAPH)
            for k, v in e.gbuffer().items():
                np.testing.assert_array_equal(v, want[k], err_msg=k)
    finally:
        e.close()
