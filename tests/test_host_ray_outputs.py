"""The output arrays of a traced model share no view and no version, on the
host: the first call's (a plan's) and those a cached template binds."""
import os
import sys

import pytest
import torch

sys.path.insert(0, os.path.dirname(__file__))
from test_host_column import _ray, _random_model, _trace  # noqa: E402

import numpy as np  # noqa: E402

from temgymcore_amd import _program  # noqa: E402


def _use(a, b, c):
    """a in a graph, b and c changed in place."""
    for t in (a, b, c):
        t.fill_(0.5)
    w = torch.ones_like(a, requires_grad=True)
    loss = (a * w).sum()
    b.mul_(2)
    c.add_(w)
    loss.backward()
    assert c.requires_grad and not any(t._is_view() for t in (a, b, c))


@pytest.mark.parametrize("n", [1, 64, 257])
@pytest.mark.parametrize("column", [True, False])
def test_plan_outputs(n, column):
    model = _random_model(np.random.default_rng(3), 5)
    tr, sym, out = _trace(_ray(n=n), model)
    plan = _program.build_plan(tr, out, sym_in=sym if column else None)
    assert (plan.column is not None) == column
    _use(plan.out_ray.x, plan.out_ray.y, plan.out_ray.dx)


@pytest.mark.parametrize("n", [1, 64, 257])
def test_bound_outputs(n):
    model = _random_model(np.random.default_rng(3), 5)
    ray = _ray(n=n)
    tr, sym, out = _trace(ray, model)
    leaves = []
    _program._structure_key((tuple(model), ray), leaves, {})
    tpl = _program._PlanTemplate(_program.build_plan(tr, out, sym_in=sym), leaves)
    _, got, _ = tpl.bind(leaves, None)
    _use(got.x, got.y, got.dx)


@pytest.mark.parametrize("shape,row", [((0,), None), ((7,), 8), ((8,), 8), ((), None), ((2, 3), None), ((2, 3), 8)])
def test_arrays(shape, row):
    got = _program._arrays(3, shape, torch.float64, torch.device("cpu"), row)
    assert [tuple(t.shape) for t in got] == [shape] * 3 and all(t.is_contiguous() for t in got)
    for k, t in enumerate(got):
        t.fill_(k)
    assert all((t == k).all() for k, t in enumerate(got))
    if len(shape) == 1 and shape[0] > 1:
        assert got[1].data_ptr() - got[0].data_ptr() == 8 * (row or shape[0])
