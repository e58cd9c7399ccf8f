"""The looked-up arguments of a one-operator call: what a call gets depends on its own parameters only (no GPU needed)."""
import itertools

import numpy as np
import pytest
import torch

from li_sparse import _pipeline

HW, TILE, FRAMES = (16, 28), (4, 8, 4), 4
NQ = _pipeline.geometry(HW, TILE, FRAMES * HW[0] * HW[1], 0, 0).nq_blk


def _plan(mode, default_ratio, p):
    n = FRAMES * HW[0] * HW[1]
    return _pipeline._call_plan(mode, torch.device("cpu"), n, 2 * n, 0, 128, HW, TILE, p, default_ratio)


def _outcome(entry, p):
    """The plan's values, None for the calls it leaves to the general route, or the type of what it raises."""
    try:
        plan = _plan(*entry, p)
    except (TypeError, ValueError) as e:
        return type(e)
    return plan if plan is None else tuple(x.tolist() if isinstance(x, torch.Tensor) else x for x in plan)


@pytest.mark.parametrize("entry", [("decode", None), ("prefill", None), ("prefill", 0.25)])
def test_a_plan_does_not_depend_on_the_calls_before_it(entry):
    """Absent keys, explicit None, equal numbers of other types, arrays: every pair in both orders as each alone."""
    base = {"topk_ratio": 0.3, "recent_protect": 2}
    params = [base] + [dict(base, **kw) for kw in (
        dict(sim_metric=None), dict(sim_metric="dot"), dict(sim_metric="cosine"), dict(topk_ratio=None),
        dict(topk_ratio=1), dict(topk_ratio=torch.tensor(0.3)), dict(recent_protect=None), dict(recent_protect=0),
        dict(recent_protect=True), dict(force_diag=None), dict(force_diag=1), dict(force_sink="yes"),
        dict(row_budget=list(range(NQ))), dict(row_budget=np.arange(NQ)), dict(row_budget=[1.5] * NQ),
        dict(row_budget=[1] * NQ), dict(row_budget=[torch.tensor(1)] * NQ), dict(row_budget=[1, 2, 3]))]
    params += [{}, {"topk_ratio": 0.3}, {"recent_protect": 2}]
    alone = []
    for p in params:
        _pipeline._CALL_PLANS.clear()
        alone.append(_outcome(entry, p))
    for (p, a), (r, b) in itertools.permutations(list(zip(params, alone)), 2):
        _pipeline._CALL_PLANS.clear()
        assert [_outcome(entry, x) for x in (p, r, p)] == [a, b, a], (p, r)


def test_changed_parameters_are_read_again():
    """A parameter object that changes in place between two calls of the same configuration."""
    def raise_ratio(x):
        x.fill_(0.6)

    def raise_first(x):
        x[0] += 2

    for name, value, change in (("topk_ratio", torch.tensor(0.3), raise_ratio),
                                ("row_budget", [torch.tensor(3) for _ in range(NQ)], raise_first),
                                ("row_budget", np.full(NQ, 3), raise_first)):
        p = {"topk_ratio": 0.3, name: value}
        before = _outcome(("decode", None), p)
        change(value)
        assert before is not None and _outcome(("decode", None), p) != before, name
    assert _outcome(("decode", None), {"recent_protect": torch.tensor(2)}) is None


def test_metric_of_an_explicit_none_is_the_plain_product():
    for first, second in itertools.permutations([{"topk_ratio": 0.3}, {"topk_ratio": 0.3, "sim_metric": None}]):
        _pipeline._CALL_PLANS.clear()
        got = {"sim_metric" in p: _plan("decode", None, p) for p in (first, second)}
        assert got[False][1][0] == _pipeline._core.METRICS["cosine"] and got[False][5] is True
        assert got[True][1][0] == _pipeline._lib.LI_METRIC_DOT and got[True][5] is False
