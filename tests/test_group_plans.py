"""Plans that a whole-group combine takes: those of its own sizes, one a rank.  The kernels read and write
where the plans say, so anything else is refused before a launch."""

import dataclasses
import types

import pytest
import torch

from moonep_amd import MoonEPCommPlan, moe


def _group(S=6, K=2, E=8, R=4, NvS=32):
    return types.SimpleNamespace(S=S, K=K, E=E, R=R, epn=E // R, NvS=NvS)


def _plans(g, stacked=True):
    """As a whole-group dispatch makes them: views of one tensor each, which the plans carry."""
    i32 = dict(dtype=torch.int32)
    dst, zero_fill = torch.arange(g.R * g.S * g.K, **i32).view(g.R, -1), torch.zeros(g.R, 2 * g.epn, 2, **i32)
    t = moe._PlanTensors(dst, zero_fill, torch.zeros(g.R, 2 * g.epn, **i32))
    plans = [MoonEPCommPlan(dst=d, experts_to_copy=torch.zeros(g.R, g.epn, **i32), zero_fill_ranges=z,
                            remote_stats=torch.zeros(2, **i32), dup_groups=torch.zeros(g.NvS, 3, **i32),
                            dup_loffs=torch.zeros(g.NvS, **i32), dup_counts=torch.zeros(2, **i32),
                            N=g.S * g.K, R=g.R, E=g.E, NvS=g.NvS, K=g.K) for d, z in zip(dst.unbind(0), zero_fill.unbind(0))]
    if stacked:
        for p in plans:
            p.dst._group_tensors = t
    return plans, t


def test_plans_of_the_group():
    g = _group()
    plans, t = _plans(g)
    assert moe._plan_tensors(g, plans) is t and moe._plan_tensors(g, tuple(plans)) is t
    other = [dataclasses.replace(p, zero_fill_ranges=p.zero_fill_ranges + 1) for p in plans]
    got = moe._plan_tensors(g, other)
    assert got.dst is t.dst and got.cu is t.cu and torch.equal(got.zero_fill, t.zero_fill + 1)
    for some in (plans[::-1], [p.clone() for p in plans], plans[:3] + plans[:1], _plans(g, stacked=False)[0]):
        got = moe._plan_tensors(g, some)
        assert got.cu is None and torch.equal(got.dst, torch.stack([p.dst for p in some]))
        assert got.zero_fill.shape == t.zero_fill.shape


@pytest.mark.parametrize("stacked", [True, False])
def test_plans_of_two_smaller_groups_behind_each_other(stacked):
    small = _group(E=8, R=4)
    plans = _plans(small, stacked)[0] + _plans(small, stacked)[0]
    with pytest.raises(AssertionError, match="plan 0 must be of"):
        moe._plan_tensors(_group(E=16, R=8), plans)


@pytest.mark.parametrize("stacked", [True, False])
@pytest.mark.parametrize("other", [dict(S=7), dict(S=4, K=3), dict(E=16), dict(NvS=48), dict(E=16, R=8)])
def test_plans_of_other_sizes(other, stacked):
    g = _group()
    plans = _plans(_group(**other), stacked)[0][:4]
    with pytest.raises(AssertionError, match="plan 0 must be of"):
        moe._plan_tensors(g, plans)
    with pytest.raises(AssertionError, match="plan 3 must be of"):
        moe._plan_tensors(g, _plans(g, stacked)[0][:3] + plans[3:])


@pytest.mark.parametrize("stacked", [True, False])
def test_more_or_fewer_plans_than_ranks(stacked):
    g = _group()
    plans, _ = _plans(g, stacked)
    for some in ([], plans[:3], plans + plans[:1]):
        with pytest.raises(AssertionError, match="takes 4 plans"):
            moe._plan_tensors(g, some)
