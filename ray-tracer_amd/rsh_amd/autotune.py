"""Autotuner of the batched-views form.

Searches the octahedral hash split (cell bits x direction bits, at most 26
bits below the view id), the hierarchy shape (leaf size x branching factor,
depth 2), the traversal mode (the engine's per-pass rule, or one mode of the
work-list kernel for every pass) and, where a work-list kernel runs, its item
size (candidate clusters per item) by coordinate descent: each dimension in
turn, keeping the best value found so far for the others.  A candidate is timed
as the median of graph replays of the whole batch (render flag bit 3), after the
eager frame that captures it; one whose first replay takes twice the best
median is not replayed again.
Every candidate's image is compared with the starting configuration's: the
hierarchy grouping may move a culling decision for a few rays, and the
fraction of identical pixels is reported with each timing.
"""
from __future__ import annotations

import dataclasses
import time

import numpy as np

from . import RshError

HASH_SPLITS = [(4, 6), (5, 4), (3, 7), (6, 3), (2, 9)]        # 2 + 3c + 2d <= 26
# (leaf, branch) of 64 rays a top node: other shapes run the generic kernel where
# a pass does not walk the triangle tree (64-view batches 10 to 100 times slower),
# and their graphs replay for the captured cameras only
SHAPES = [(8, 8), (4, 16), (16, 4), (32, 2)]
CHUNKS = [64, 16, 256]                                        # candidate clusters per work item
PREFILTERS = [0, 2, 3]          # traversal mode: the per-pass rule; the work list with the ray pre-test, + cluster masks
TREE = 3                        # FrameStats.pass_mode of a pass that walked the triangle tree


@dataclasses.dataclass
class Trial:
    cell_bits: int
    dir_bits: int
    leaf: int
    branch: int
    traversal_chunk: int
    traversal_prefilter: int
    ms: float
    mrays: float
    same_pixels: float


def time_batch(engine, views, cfg, reps=3, stop_ms=None):
    """Median wall time (ms) of graph replays of the batch, rays per batch.
    stop_ms: no further replays after a first that takes longer."""
    st = engine.render_views(views, cfg, flags=engine.GRAPH)          # eager frame + capture
    rays = st.rays_total
    times = []
    for _ in range(reps):
        t0 = time.perf_counter()
        engine.render_views(views, cfg, flags=engine.GRAPH)
        times.append(time.perf_counter() - t0)
        if stop_ms is not None and len(times) == 1 and 1e3 * times[0] > stop_ms:
            break
    return 1e3 * float(np.median(times)), rays


def tune(engine, scene, views, base_cfg, reps=3, log=None):
    """Coordinate-descent search from base_cfg (cell grid re-fitted to the
    scene for every hash split); returns (best_cfg, [Trial])."""
    engine.render_views(views, base_cfg)
    ref = engine.pixels().copy()
    trials = []
    best = base_cfg
    best_ms = None

    def run(cfg):
        nonlocal best, best_ms
        try:
            ms, rays = time_batch(engine, views, cfg, reps, None if best_ms is None else 2.0 * best_ms)
        except RshError as err:      # e.g. a work list over capacity for a small chunk: not a candidate
            if log:
                log(f"skipped {cfg.cell_bits}/{cfg.dir_bits} {cfg.leaf}x{cfg.branch} chunk {cfg.traversal_chunk} "
                f"mode {cfg.traversal_prefilter}: {err}")
            return
        same = float((engine.pixels() == ref).mean())
        t = Trial(cfg.cell_bits, cfg.dir_bits, cfg.leaf, cfg.branch, cfg.traversal_chunk, cfg.traversal_prefilter, ms,
                  rays / ms / 1e3, same)
        trials.append(t)
        if log:
            log(t)
        if best_ms is None or ms < best_ms:
            best, best_ms = cfg, ms

    run(base_cfg)
    for c, d in HASH_SPLITS:
        if (c, d) != (best.cell_bits, best.dir_bits):
            run(dataclasses.replace(best, cell_bits=c, dir_bits=d).with_scene_bounds(scene))
    for leaf, branch in SHAPES:
        if (leaf, branch) != (best.leaf, best.branch):
            run(dataclasses.replace(best, leaf=leaf, branch=branch))
    def walks_tree():
        st = engine.render_views(views, best)
        return TREE in list(st.pass_mode)[:st.pass_count]

    # The work-list kernel's own dimensions leave the tree, so they are worth a
    # trial only in its shapes, and an item size only once the work list is ahead.
    if best.leaf * best.branch == 64 or not walks_tree():
        for pf in PREFILTERS:
            if pf != best.traversal_prefilter:
                run(dataclasses.replace(best, traversal_prefilter=pf))
        if not walks_tree():
            for ch in CHUNKS:
                if ch != best.traversal_chunk:
                    run(dataclasses.replace(best, traversal_chunk=ch))
    return best, trials
