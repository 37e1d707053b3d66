"""How long host plans live (no GPU: the work lists are built on the host and put on the CPU here)."""

import gc
import weakref

import torch

from hackaton_amd import attention as att

CPU = torch.device("cpu")


def _plan_of(lengths, hq=12, hkv=2):
    return att._plan(att._cu_seqlens(lengths, CPU), hq, hkv)


def test_plans_of_33_batches_are_built_once():
    """A program that cycles through 33 lists of lengths gets every plan of the first cycle back in
    the second, whether its cu_seqlens come from the host lengths or are its own tensor."""
    batches = [[100 + i, 50, 7] for i in range(33)]
    plans = [_plan_of(lengths) for lengths in batches]
    assert all(_plan_of(lengths) is plan for lengths, plan in zip(batches, plans))
    own = torch.tensor([0, 100, 150, 157], dtype=torch.int32)
    assert att._plan(own, 12, 2) is plans[0]


def test_plan_cache_is_bounded():
    for i in range(80):
        _plan_of([200 + i, 31])
    assert len(att._CU_SEQLENS) <= 17
    assert att._host_plan.cache_info().currsize <= 33


def test_plans_of_a_captured_graph_are_kept(monkeypatch):
    """The work lists of a call under graph capture outlive every cache and autograd node: the
    graph's kernels hold their addresses. They go when the program says so."""
    monkeypatch.setattr(att, "_capturing", lambda: True, raising=False)
    lists = []
    for make in (lambda: att._cu_seqlens([300, 41], CPU),
                 lambda: torch.tensor([0, 301, 342], dtype=torch.int32)):
        plan = att._plan(make(), 12, 2)
        lists += [weakref.ref(plan.fwd_items), weakref.ref(plan.bwd_items),
                  weakref.ref(plan.partial_bwd()[0])]
    del plan
    monkeypatch.setattr(att, "_capturing", lambda: False, raising=False)
    for i in range(80):
        _plan_of([300 + i, 42])
    gc.collect()
    assert all(items() is not None for items in lists)
    att.release_captured_plans()
    gc.collect()
    assert all(items() is None for items in lists)
