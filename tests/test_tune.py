"""The granularity tuner's host side (vdttfs.tune): plan files are checked
against the workload they are applied to, and plan records round-trip."""
import json

import pytest

import vdttfs
from vdttfs import models, tune


def test_plan_records_round_trip():
    for p in [(vdttfs.PATH_BINS, 4, 2), (vdttfs.PATH_DENSE, 2, 1), (vdttfs.PATH_FUSED, 1, 8), (vdttfs.PATH_REG, 1, 10)]:
        d = tune._plan_dict(p)
        assert (tune._path_id(d["path"]), d["gather"], d["ppw"]) == p
    assert tune._plan_dict((0, 0, 0))["path"] == "none"


def test_load_plans_checks_workload(tmp_path):
    w = models.lenet5()
    plans = [None] * len(w.layers)
    plans[0] = {"path": "dense", "gather": 1, "ppw": 10}
    f = tmp_path / "p.json"
    f.write_text(json.dumps({"workload": w.name, "batch": 64, "T": w.consts.T, "plans": plans}))
    assert tune.load_plans(str(f), w, 64) == plans
    with pytest.raises(ValueError):
        tune.load_plans(str(f), w, 128)  # another batch
    with pytest.raises(ValueError):
        tune.load_plans(str(f), models.lenet5(T=32), 64)  # another window
    with pytest.raises(ValueError):
        tune.load_plans(str(f), models.vgg16(), 64)  # another network
    assert tune.load_pool_fusion(str(f), w, 64) is None  # files without a pool-fusion mode
    for name in ("off", "auto", "all"):
        f.write_text(json.dumps({"workload": w.name, "batch": 64, "T": w.consts.T, "plans": plans,
                                 "pool_fusion": name}))
        assert tune.load_pool_fusion(str(f), w, 64) == name
        assert tune.POOL_FUSION[name] in (vdttfs.POOL_FUSE_OFF, vdttfs.POOL_FUSE_AUTO, vdttfs.POOL_FUSE_ALL)
    f.write_text(json.dumps({"workload": w.name, "batch": 64, "T": w.consts.T, "plans": plans,
                             "pool_fusion": "some"}))
    with pytest.raises(ValueError):
        tune.load_pool_fusion(str(f), w, 64)


class FakeNet:
    """The tuner's view of a network with one integrating layer: a time per
    plan, None being the built-in choice."""

    def __init__(self, layers, ms):
        self.layers, self.ms, self.plans = layers, ms, {}

    def set_plan(self, layer, *plan):
        self.plans[layer] = plan or None
        if plan and plan not in self.ms:
            raise vdttfs.VdttfsError(-6, "plan")


@pytest.mark.parametrize("builtin_ms,wins", [(1.0, True), (2.0, True), (3.0, False)])
def test_builtin_choice_is_a_candidate(builtin_ms, wins):
    """A layer whose built-in time is the lowest keeps the built-in choice,
    whose kernels may have no plan of their own."""
    named = [{"plan": {"path": "fused", "gather": 2, "ppw": 1}, "ms": 2.0, "identical": True},
             {"plan": {"path": "bins", "gather": 4, "ppw": 2}, "ms": 0.5, "identical": False}]
    auto = {"plan": {"path": "fused", "gather": 2, "ppw": 1, "builtin": True}, "ms": builtin_ms, "identical": True}
    best = tune.best_candidate([auto] + named)
    assert (best is auto) == wins
    net = FakeNet([None], {(vdttfs.PATH_FUSED, 2, 1): 2.0})
    tune.apply_plans(net, [best["plan"]])
    assert net.plans[0] == (None if wins else (vdttfs.PATH_FUSED, 2, 1))
    assert tune.best_candidate([named[1]]) is None


def test_committed_vgg_plans_fit_the_benchmark():
    """configs/plans_vgg16_b256.json (tuned on MI355X, bench.py --plans) names
    a plan for exactly the integrating layers of the benchmark network."""
    import os

    w = models.vgg16()
    path = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "configs",
                        "plans_vgg16_b256.json")
    plans = tune.load_plans(path, w, 256)
    assert len(plans) == len(w.layers)
    for l, p in zip(w.layers, plans):
        integ = l.kind in (vdttfs.LAYER_CONV, vdttfs.LAYER_FC)
        assert (p is not None) == integ
        if p:
            assert p["path"] in ("bins", "dense", "fused", "reg") and p["gather"] in (1, 2, 4) and 1 <= p["ppw"] <= 64
