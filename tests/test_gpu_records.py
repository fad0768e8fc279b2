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
