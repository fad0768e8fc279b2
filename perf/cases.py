"""The work this library is timed on: frames, batches of views, ray queries,
served requests and the drop-in stages, each through its public entry point
(``rsh_amd.Engine``, ``rsh_amd.server.Server``, ``rsh_amd.Context`` and the C
ABI of include/rsh.h for rays that already lie on the device).

Scenes are the repository's own generators and stay resident, as a renderer
keeps its assets; what changes with the seed is what changes from call to call
in use: the camera, the object transforms, the rays and the requests.  Every
output is whole numbers (pixels, hit records, occlusion flags, ray counts).
"""
from __future__ import annotations

import ctypes
import dataclasses
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ray-tracer_amd"))

import rsh_amd  # noqa: E402
from rsh_amd import config as cf  # noqa: E402
from rsh_amd import queries, scenes, serving  # noqa: E402
from rsh_amd.server import Server  # noqa: E402

SCENES = {"plain": scenes.config0_scene, "office": scenes.config1_scene, "atrium": scenes.config2_scene,
          "soup": scenes.soup_scene}
TRIANGLES = {"plain": 2060, "office": 30012, "atrium": 262604, "soup": 100000}
LIGHTS = {"plain": 1, "office": 2, "atrium": 1, "soup": 1}
MIX = {"primary": queries.PRIMARY, "shadow": queries.SHADOW, "diffuse": queries.DIFFUSE}
SERVED = ("plain", "office", "atrium", "soup")


@functools.lru_cache(maxsize=None)
def scene(name):
    return SCENES[name]()


def listed():
    return [
        # the smallest frame: a thumbnail or preview, the size of the smoke frame (launches and waits)
        frame("frame_plain_64", "plain", 64, 64, bounces=1, bounce_shadows=0),
        # the plain 512 x 512 frame, one shadow pass and one mirror bounce: the reference's window size
        frame("frame_plain_512", "plain", 512, 512, bounces=1, bounce_shadows=0),
        # the office-scale frame: two lights, two gated bounces with shadows at every hit
        frame("frame_office_1024", "office", 1024, 1024, bounces=2, bounce_shadows=1),
        # the headline frame: the 262k-triangle atrium at 1080p, three bounces and shadows
        frame("frame_atrium_1080p", "atrium", 1920, 1080, bounces=3, bounce_shadows=1),
        # soft shadows (16 shadow rays a slot) at a ragged window size
        frame("frame_office_soft_ragged", "office", 701, 499, bounces=1, bounce_shadows=1, soft=True),
        # an animated scene: every object moves before every frame
        frame("frame_atrium_moving_720p", "atrium", 1280, 720, bounces=2, bounce_shadows=1, moving=True),
        # a batch of random square views in one call, replayed from its graph as a render loop does
        dict(name="views_office_16", kind="views", scene="office", views=16, lo=128, hi=1024),
        # a picking or visibility probe from host code: a thousand rays from and to host arrays
        query("query_host_primary_1k", "office", "primary", 1000, host=True),
        # an occlusion batch of rays that a simulation holds on the device, odd count
        query("query_shadow_100k", "atrium", "shadow", 100_003),
        # one bounce of a path tracer or a light-map bake: a million spread-out rays on the device
        query("query_diffuse_1m", "atrium", "diffuse", 1 << 20),
        # a burst of requests of mixed sizes and kinds against four resident scenes, host to host
        dict(name="serve_burst_24", kind="serve", requests=24, lo=1000, hi=400_000),
        # the reference's own stages driven one by one at its window size (shadow pass, one bounce)
        dict(name="stages_plain_512", kind="stages", side=512),
    ]


def frame(name, scene_name, width, height, bounces, bounce_shadows, algorithm=cf.CRSH, key=cf.KEY_OCT, soft=False,
          moving=False):
    return dict(name=name, kind="frame", scene=scene_name, width=width, height=height, bounces=bounces,
                bounce_shadows=bounce_shadows, algorithm=algorithm, key=key, soft=soft, moving=moving)


def query(name, scene_name, mix, rays, host=False):
    return dict(name=name, kind="query", scene=scene_name, mix=mix, rays=rays, host=host)


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ranges: any size from the smallest listed
    to the largest, any scene, and the options callers set (reference keys,
    the unsorted RAH hierarchy where its cost allows, soft shadows, moving
    objects)."""
    kind = rng.choice(["frame", "frame", "frame", "query", "query", "query", "views", "serve", "stages"])
    if kind == "frame":
        name = rng.choice(["plain", "office", "atrium"])
        algorithm = cf.RAH if name == "plain" and rng.random() < 0.3 else cf.CRSH
        soft = rng.random() < 0.2
        pixels = log_int(rng, 64 * 64, (640 * 480) if soft else 1920 * 1080)
        aspect = rng.uniform(0.7, 1.9)
        width = max(16, int(round(math.sqrt(pixels * aspect))))
        c = frame("", name, width, max(16, pixels // width), rng.randint(0, 3 if name == "atrium" else 2),
                  rng.randint(0, 1), algorithm, cf.KEY_REF if rng.random() < 0.2 else cf.KEY_OCT, soft,
                  rng.random() < 0.2)
    elif kind == "query":
        name = rng.choice(SERVED)
        mix = rng.choice(["primary", "shadow", "diffuse"])
        host = rng.random() < 0.35
        c = query("", name, mix, log_int(rng, 500, 100_000 if host else 1 << 20), host)
    elif kind == "views":
        lo = log_int(rng, 64, 256)
        c = dict(name="", kind="views", scene=rng.choice(["plain", "office"]), views=rng.randint(2, 16), lo=lo,
                 hi=rng.randint(lo, 1024))
    elif kind == "serve":
        c = dict(name="", kind="serve", requests=rng.randint(4, 24), lo=1000, hi=log_int(rng, 4000, 400_000))
    else:
        c = dict(name="", kind="stages", side=log_int(rng, 48, 512))
    c.pop("name")
    return c


def walked(name, width, height, rng):
    """The scene's own camera a few steps along a walk."""
    eye, target = {"plain": ((0.5, 0.5, 0.05), (0.5, 0.5, 1.0)), "office": ((0.5, 0.5, 0.02), (0.5, 0.45, 1.0)),
                   "atrium": ((0.5, 0.35, 0.01), (0.5, 0.3, 1.0))}[name]
    eye = np.asarray(eye) + rng.uniform(-1.0, 1.0, 3) * (0.03, 0.03, 0.005)
    target = np.asarray(target) + rng.uniform(-0.08, 0.08, 3)
    return scenes.camera_basis(scenes.world(eye), scenes.world(target), (0, 1, 0), 60.0, width, height)


def transforms(sc, rng):
    """Every object but the room turned about y and shifted a little about its
    centre: model, normal and scale matrices."""
    K = sc.object_total
    model = np.tile(np.eye(4, dtype=np.float32), (K, 1, 1))
    normal, scale = model.copy(), model.copy()
    a = rng.uniform(-0.2, 0.2, K)
    a[0] = 0.0
    shift = rng.uniform(-0.4, 0.4, (K, 3))
    shift[0] = 0.0
    c, s = np.cos(a), np.sin(a)
    R = np.zeros((K, 3, 3))
    R[:, 0, 0], R[:, 0, 2], R[:, 1, 1], R[:, 2, 0], R[:, 2, 2] = c, s, 1.0, -s, c
    centre = sc.object_spheres[:, :3].astype(np.float64)
    model[:, :3, :3] = normal[:, :3, :3] = R
    model[:, :3, 3] = centre + shift - np.einsum("kij,kj->ki", R, centre)
    return model.reshape(K, 16), normal.reshape(K, 16), scale.reshape(K, 16)


def frame_config(case):
    c = cf.FrameConfig(width=case["width"], height=case["height"], algorithm=case["algorithm"], key_mode=case["key"],
                       bounces=case["bounces"], bounce_shadows=case["bounce_shadows"],
                       soft_shadows=int(case["soft"]))
    return c.with_scene_bounds(scene(case["scene"])) if case["key"] == cf.KEY_OCT else c


def prepare(case, seed):
    return {"frame": prepare_frame, "views": prepare_views, "query": prepare_query, "serve": prepare_serve,
            "stages": prepare_stages}[case["kind"]](case, np.random.default_rng(seed))


def run(state):
    return state["run"](state)


def engine_with(name):
    e = rsh_amd.Engine(0)
    e.load_scene(scene(name))
    return e


# ------------------------------------------------------------------ frames --
def prepare_frame(case, rng):
    sc = scene(case["scene"])
    return dict(run=run_frame, engine=engine_with(case["scene"]), cfg=frame_config(case),
                camera=walked(case["scene"], case["width"], case["height"], rng),
                image=pinned_image(case["width"] * case["height"]),
                moved=transforms(sc, rng) if case["moving"] else None)


def pinned_image(pixels):
    """A page-locked image buffer of the caller's, filled by each frame."""
    return torch.empty(pixels, dtype=torch.int32, pin_memory=True)


def read_image(e, image):
    rc = e.L.rsh_engine_read_pixels(e.h, ctypes.cast(image.data_ptr(), rsh_amd.PU), image.numel())
    if rc != 0:
        raise rsh_amd.RshError(e.L.rsh_last_error(e.h).decode())
    return image


def run_frame(s):
    e = s["engine"]
    if s["moved"] is not None:
        e.update_objects(*s["moved"])
    st = e.render(s["camera"], s["cfg"])
    return {"pixels": read_image(e, s["image"]), "rays": list(st.pass_rays[:st.pass_count])}


def prepare_views(case, rng):
    sc = scene(case["scene"])
    sides = np.random.default_rng(case["views"]).integers(case["lo"], case["hi"] + 1, case["views"])
    views = [(scenes.random_view(rng, int(n), int(n)), int(n), int(n)) for n in sides]
    base = cf.config1() if case["scene"] == "office" else cf.config0()
    cfg = dataclasses.replace(base, cell_bits=4, dir_bits=6, segment_shift=26).with_scene_bounds(sc)
    return dict(run=run_views, engine=engine_with(case["scene"]), cfg=cfg, views=views,
                image=pinned_image(sum(w * h for _, w, h in views)))


def run_views(s):
    e = s["engine"]
    st = e.render_views(s["views"], s["cfg"], flags=e.GRAPH)
    return {"pixels": read_image(e, s["image"]), "rays": int(st.rays_total)}


# ----------------------------------------------------------------- queries --
def prepare_query(case, rng):
    sc = scene(case["scene"])
    rays, tmax, kind = queries.make_query(sc, MIX[case["mix"]], case["rays"], rng)
    s = dict(run=run_host_query if case["host"] else run_device_query, engine=engine_with(case["scene"]),
             cfg=serving.query_config(sc), kind=kind, rays=rays, tmax=tmax)
    if not case["host"]:
        s["rays"] = torch.from_numpy(rays).cuda()
        s["tmax"] = torch.from_numpy(tmax).cuda() if tmax is not None else None
        s["out"] = torch.empty(case["rays"], dtype=torch.int32 if kind == 1 else torch.int64, device="cuda")
        s["desc"] = rsh_amd.config_desc(s["cfg"])
        torch.cuda.synchronize()
    return s


def run_host_query(s):
    return s["engine"].trace(s["rays"], s["kind"], s["cfg"], tmax=s["tmax"])


def run_device_query(s):
    e = s["engine"]
    rc = e.L.rsh_engine_trace(e.h, s["rays"].data_ptr(), s["tmax"].data_ptr() if s["tmax"] is not None else None, None,
                              s["rays"].shape[0], s["kind"], ctypes.byref(s["desc"]), s["out"].data_ptr(), 0, None)
    if rc != 0:
        raise rsh_amd.RshError(e.L.rsh_last_error(e.h).decode())
    return s["out"]


def prepare_serve(case, rng):
    server = Server(0, hbm_budget=16 << 30)
    sids = [server.add_scene(scene(n), serving.query_config(scene(n))) for n in SERVED]
    requests = []
    shapes = np.random.default_rng(case["requests"])      # the case's own: scene, kind and size of each request
    for _ in range(case["requests"]):
        k = int(shapes.integers(len(SERVED)))
        mix = int(shapes.choice(serving.MIX[0], p=serving.MIX[1]))
        n = int(np.exp(shapes.uniform(np.log(case["lo"]), np.log(case["hi"]))))
        rays, tmax, kind = queries.make_query(scene(SERVED[k]), mix, n, rng)
        out = torch.empty(n, dtype=torch.int32 if kind == 1 else torch.int64, pin_memory=True).numpy()
        requests.append((sids[k], torch.from_numpy(rays).pin_memory().numpy(), kind,
                         torch.from_numpy(tmax).pin_memory().numpy() if tmax is not None else None,
                         out.view(np.uint32 if kind == 1 else np.uint64)))
    return dict(run=run_serve, server=server, requests=requests)


def run_serve(s):
    server = s["server"]
    ids = [server.submit(sid, rays, kind, tmax, out=out) for sid, rays, kind, tmax, out in s["requests"]]
    return [server.wait(i)[0] for i in ids]


# ------------------------------------------------------------------ stages --
SUB, BATCH = 8, 5000        # the reference's subdivision and triangle batch


def prepare_stages(case, rng):
    """The buffers of the reference's frame driver (main.cpp:1400-1497), its
    raster G-buffer taken from an engine frame."""
    sc, side = scene("plain"), case["side"]
    cam = walked("plain", side, side, rng)
    e = engine_with("plain")
    e.render(cam, cf.config0(side, side).with_scene_bounds(sc))
    g = {k: torch.from_numpy(v).cuda() for k, v in e.gbuffer().items()}
    e.close()
    S, T, K = side * side, sc.triangle_total, sc.object_total
    n0 = (S + SUB - 1) // SUB
    b = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in dict(
        pos=sc.tri_pos, nrm=sc.tri_nrm, obj=np.repeat(sc.triangle_object(), 3).astype(np.int32),
        mat=sc.tri_mat.astype(np.int32), mdif=sc.mat_diffuse, mspec=sc.mat_specular,
        sph=sc.object_spheres.reshape(2 * K, 3), lpos=sc.light_pos, lcol=sc.light_col, lint=sc.light_int).items()}
    pairs = max(n0 // 2, 1) * 10000
    for k in ("flags", "scan", "hits", "thits"):
        b[k] = torch.empty(pairs, dtype=torch.int32, device="cuda")
    for k in ("pkeys", "pvals", "skeys", "svals", "bases", "sizes", "ckeys", "cvals", "sckeys", "scvals", "records",
              "pixels"):
        b[k] = torch.zeros(S, dtype=torch.int32, device="cuda")
    b["rays"] = torch.zeros((2 * S, 3), dtype=torch.float32, device="cuda")
    b["hier"] = torch.zeros((2 * (n0 + (n0 + SUB - 1) // SUB), 4), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    p = {k: v.data_ptr() for k, v in {**b, **{"g" + k: v for k, v in g.items()}}.items()}
    ctx = rsh_amd.Context(0)
    ctx.configure(1, 2, SUB, cf.CRSH)
    ctx.set_gbuffer(p["gdif"], p["gspec"], p["gpos"], p["gnrm"], side, side)
    ctx.set_scene(p["pos"], p["nrm"], p["obj"], p["mat"], T, p["mdif"], p["mspec"], sc.mat_diffuse.shape[0], p["sph"], K,
                  p["lpos"], p["lcol"], p["lint"], sc.light_total)
    ctx.stage("memory_preparation", None, side, side, pairs)
    return dict(run=run_stages, ctx=ctx, b=b, g=g, p=p, side=side, T=T, K=K, pairs=pairs, lights=sc.light_total,
                eye=rsh_amd.Float3(*[float(v) for v in cam.eye]))


def run_stages(s):
    """The reference's frame loop (main.cpp:1234-1303) with one bounce."""
    stage, p, side = s["ctx"].stage, s["p"], s["side"]
    u = ctypes.c_uint32

    def cast():
        n, c = u(0), u(0)
        stage("ray_trimming", None, p["pkeys"], p["pvals"], side, side, 1, p["flags"], p["scan"], p["skeys"],
              p["svals"], ctypes.byref(n), None)
        stage("ray_compression", None, p["skeys"], p["svals"], n.value, None, p["flags"], p["scan"], p["bases"],
              p["sizes"], p["ckeys"], p["cvals"], ctypes.byref(c), None)
        stage("ray_sorting", None, p["ckeys"], p["cvals"], c.value, None, p["sckeys"], p["scvals"])
        stage("ray_decompression", None, p["bases"], p["sizes"], p["sckeys"], p["scvals"], p["skeys"], p["svals"],
              p["flags"], p["scan"], c.value, None, p["pkeys"], p["pvals"])
        stage("hierarchy_creation", None, p["rays"], p["pkeys"], p["pvals"], n.value, None, 0.0, 0.0, p["hier"])
        return n.value

    def traverse(n, name, *more):
        for off in range(0, s["T"], BATCH):
            batch, hits, room = min(BATCH, s["T"] - off), u(0), u(s["pairs"])
            stage("hierarchy_traversal_warmup", None, p["hier"], p["sph"], p["pos"], s["K"], n, batch, off, p["flags"],
                  p["scan"], p["hits"], p["thits"], ctypes.byref(hits), ctypes.byref(room))
            stage("hierarchy_traversal", None, p["hier"], p["pos"], n, batch, off, p["flags"], p["scan"], p["hits"],
                  p["thits"], ctypes.byref(hits), ctypes.byref(room))
            stage(name, None, p["rays"], p["pkeys"], p["pvals"], p["thits"], p["pos"], hits.value, n, off, side, side,
                  *more, s["eye"], p["records"])

    stage("shadow_ray_creation", None, side, side, 1, p["rays"], p["flags"], p["pkeys"], p["pvals"])
    shadow_rays = cast()
    stage("shadow_ray_preparation", None, side, side, 1, p["records"])
    traverse(shadow_rays, "shadow_ray_intersection")
    stage("shadow_ray_coloring", None, side, side, s["lights"], s["eye"], p["records"], p["pixels"])
    stage("reflection_ray_creation", None, side, side, s["eye"], p["rays"], p["flags"], p["pkeys"], p["pvals"])
    mirror_rays = cast()
    stage("reflection_ray_preparation", None, side, side, p["records"])
    traverse(mirror_rays, "reflection_ray_intersection", 1)
    stage("reflection_ray_coloring", None, p["pos"], p["nrm"], side, side, s["lights"], s["eye"], False, p["records"],
          p["rays"], p["flags"], p["pkeys"], p["pvals"], p["pixels"])
    return {"pixels": s["b"]["pixels"], "records": s["b"]["records"], "rays": [shadow_rays, mirror_rays]}


# -------------------------------------------------------------------- work --
RAY_BYTES, TEST_FLOPS, TRIANGLE_BYTES = 24, 46, 48 + 48 + 12   # a ray; one exact test; positions, normals, materials


def work(case):
    """Inputs read once, outputs written once, and one exact ray / triangle
    test per ray that is certain to be traced.  A call with fewer rays than
    triangles cannot need more triangles than it has rays."""
    kind = case["kind"]
    if kind == "frame":
        pixels, tris = case["width"] * case["height"], TRIANGLES[case["scene"]]
        rays = pixels * (1 + LIGHTS[case["scene"]] * (16 if case["soft"] else 1))
        return {"bytes": 4 * pixels + TRIANGLE_BYTES * min(tris, rays), "flops": TEST_FLOPS * rays}
    if kind == "views":
        side2 = (case["lo"] ** 2 + case["lo"] * case["hi"] + case["hi"] ** 2) / 3.0
        pixels = int(case["views"] * side2)
        rays = pixels * (1 + LIGHTS[case["scene"]])
        return {"bytes": 4 * pixels + TRIANGLE_BYTES * min(TRIANGLES[case["scene"]], rays), "flops": TEST_FLOPS * rays}
    if kind == "query":
        n = case["rays"]             # a shadow ray: its length in, 4 bytes out; another: 8 bytes out
        return {"bytes": n * (RAY_BYTES + 8) + 48 * min(n, TRIANGLES[case["scene"]]), "flops": TEST_FLOPS * n}
    if kind == "serve":
        lo, hi = case["lo"], max(case["hi"], case["lo"] + 1)
        n = int(case["requests"] * (hi - lo) / math.log(hi / lo))
        return {"bytes": n * (RAY_BYTES + 8) + 48 * min(n, sum(TRIANGLES[x] for x in SERVED)), "flops": TEST_FLOPS * n}
    pixels = case["side"] ** 2
    return {"bytes": pixels * (64 + 4 + 4) + TRIANGLE_BYTES * TRIANGLES["plain"], "flops": 2 * TEST_FLOPS * pixels}


def exact(case, seed):
    """Every output is whole numbers: nothing to compare in 64 bits."""
    return None
