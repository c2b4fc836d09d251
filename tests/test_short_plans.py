"""The plans of short lists through the three named functions: which ones the bounded cache keeps.
On the CPU: the walk over the list is told that host tensors are on a GPU, and prepare() is its plan."""

import threading
from collections import OrderedDict

import pytest
import torch

from torchft_amd import quantization as q


@pytest.fixture
def match(monkeypatch):
    if q._pylist is None:
        pytest.skip("torchft_amd._pylist cannot be built here")
    made = []

    class Pylist:
        @staticmethod
        def describe(tensors, most):
            key, _, pointers = q_pylist.describe(tensors, most)
            return key, 0, pointers

    def prepare(tensors, ws):
        made.append(tuple(tensors[0].shape))
        return type("Bucket", (), {"plan": q._plan_for(tensors[0].dtype, ws, tuple(t.size() for t in tensors),
                                                       tuple(t.stride() for t in tensors))})

    q_pylist = q._pylist
    monkeypatch.setattr(q, "_pylist", Pylist)
    monkeypatch.setattr(q, "prepare", prepare)
    monkeypatch.setattr(q, "_plan_cache", OrderedDict())
    monkeypatch.setattr(q, "_short_plans", {})
    monkeypatch.setattr(q, "_plan_cache_tensors", 0)
    monkeypatch.setattr(q, "_PLAN_CACHE_SIZE", 8)
    return lambda n: q._match_short_list([torch.empty(2, n)], 2), made


def test_a_plan_in_use_outlives_many_that_come_once(match):
    match, made = match
    for n in range(1, 100):
        match(n)
        match(1000)
        match(2000)
    assert made.count((2, 1000)) == made.count((2, 2000)) == 1 and len(made) == 99 + 2
    assert len(q._plan_cache) == 8 and len(q._short_plans) <= 8
    assert set(q._short_plans.values()) <= set(q._plan_cache.values())
    # all of them in use: the newest stays, one of the others goes
    for _ in range(3):
        for n in range(200, 208):
            match(n)
    plan = match(300)[0]
    assert plan.cached and match(300)[0] is plan and len(q._plan_cache) == 8


def test_a_plan_that_the_cache_has_let_go_is_not_entered(match, monkeypatch):
    match, _ = match
    prepare = q.prepare

    def prepare_slowly(tensors, ws):   # as if other threads had made plans in the meantime
        bucket = prepare(tensors, ws)
        for n in range(3000, 3020):
            q._plan_for(torch.float32, 2, (torch.Size((2, n)),), ((n, 1),))
        return bucket

    monkeypatch.setattr(q, "prepare", prepare_slowly)
    plan, _, _ = match(77)
    assert not plan.cached and not q._short_plans


def test_threads(match):
    match, _ = match
    bad = []

    def run(k):
        for i in range(300):
            n = (i * (k + 1)) % 23 + 1
            plan = match(n)[0]
            if list(plan.shapes) != [2, n]:
                bad.append(n)

    threads = [threading.Thread(target=run, args=(k,)) for k in range(6)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad and len(q._plan_cache) <= 8
    assert set(q._short_plans.values()) <= set(q._plan_cache.values())
    assert q._plan_cache_tensors == len(q._plan_cache)
