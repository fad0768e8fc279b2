"""The batch autotuner's search against an engine of stated costs: which
candidates it times, and what it chooses."""
import dataclasses
import time
import types

import numpy as np
import pytest


class Engine:
    """Frames that take cost(cfg) milliseconds; a pass walks the tree unless a
    work-list option is asked for, and those need 64 rays a top node."""
    GRAPH = 8

    def __init__(self, cost):
        self.cost, self.calls = cost, []

    def render_views(self, views, cfg, flags=0):
        tree = cfg.traversal_prefilter == 0 and cfg.traversal_chunk == 0
        kind = "tree" if tree else "list" if cfg.leaf * cfg.branch == 64 else "generic"
        self.calls.append((kind, cfg))
        time.sleep(1e-3 * self.cost(kind, cfg))
        return types.SimpleNamespace(rays_total=1000, pass_count=2, pass_mode=[3 if tree else 1] * 2 + [0] * 8)

    def pixels(self):
        return np.zeros(4, np.uint32)


def search(rsh_amd, cost, **base):
    from rsh_amd import autotune
    sc = types.SimpleNamespace(bounds_min=np.zeros(3, np.float32), bounds_max=np.ones(3, np.float32))
    eng = Engine(cost)
    cfg = dataclasses.replace(rsh_amd.config.config0(), cell_bits=4, dir_bits=6, **base)
    best, trials = autotune.tune(eng, sc, [None], cfg)
    return eng, best, trials


def test_options_that_leave_the_tree_cost_little(rsh):
    """The work list twice and the generic kernel a hundred times as long as the
    tree: the generic kernel is never timed, the work list never more than its
    captures and one replay, and the tree keeps its options."""
    eng, best, trials = search(rsh, lambda kind, cfg: {"tree": 2.0, "list": 6.0, "generic": 200.0}[kind])
    kinds = [k for k, _ in eng.calls]
    assert "generic" not in kinds
    assert kinds.count("list") <= 4                  # two trials: a capturing frame and one replay each
    assert (best.traversal_chunk, best.traversal_prefilter) == (0, 0)
    assert len(trials) >= 10


@pytest.mark.parametrize("base", [dict(leaf=8, branch=4)])
def test_other_shapes_keep_the_tree(rsh, base):
    cost = {"tree": lambda cfg: 1.0 if (cfg.leaf, cfg.branch) == (8, 4) else 4.0}
    eng, best, _ = search(rsh, lambda kind, cfg: cost.get(kind, lambda c: 200.0)(cfg), **base)
    assert {k for k, _ in eng.calls} == {"tree"}
    assert (best.leaf, best.branch) == (8, 4)


def test_a_faster_work_list_is_found_and_its_item_size_tuned(rsh):
    def cost(kind, cfg):
        if kind == "tree":
            return 8.0
        if cfg.traversal_prefilter != 3:
            return 6.0
        return 1.0 if cfg.traversal_chunk == 16 else 3.0
    _, best, _ = search(rsh, cost)
    assert (best.traversal_prefilter, best.traversal_chunk) == (3, 16)
