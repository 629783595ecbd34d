"""Handing requests back while something fails: the arena keeps every slot and range until all of it is queued, so a
retire that raised can be repeated, and nothing admitted later shares a range with particles still in the set.

Bar: the repeated retire's results bit-exact against the same requests stepped alone."""

import pytest
import torch

import serve
from test_gpu_serve import alone, make_templates, same

pytestmark = pytest.mark.gpu

STEPS = 2


def arena_with(tpls):
    arena = serve.FempicArena(max_cells=5000, max_nodes=2000, max_particles=40000, max_overlay=10000, max_insts=4)
    slots = [arena.admit(t) for t in tpls]
    for _ in range(STEPS):
        arena.step()
    return arena, slots


def owned(arena):
    return (sorted(arena.res), sorted(arena.slots_free), list(arena.cells.free), list(arena.nodes.free),
            list(arena.ovl.free), arena.dropping, arena.size)


def fail_at(monkeypatch, where, call):
    """The call-th (from 0) pinned allocation, or copy_batch, raises."""
    n = [0]
    if where == "pin":
        real, target, name = torch.empty, torch, "empty"
        hit = lambda a, kw: kw.get("pin_memory", False)
    else:
        real, target, name = serve.copy_batch, serve, "copy_batch"
        hit = lambda a, kw: True

    def f(*a, **kw):
        if hit(a, kw):
            n[0] += 1
            if n[0] == call + 1:
                raise MemoryError("no more of it")
        return real(*a, **kw)

    monkeypatch.setattr(target, name, f)


@pytest.mark.parametrize("where,call", [("pin", 0), ("pin", 5), ("pin", 9), ("copy", 0), ("copy", 1)])
def test_a_retire_that_raised_can_be_repeated(monkeypatch, where, call):
    tpls = make_templates([(3, 4000), (4, 9000), (2, 700)], seed=64)
    arena, slots = arena_with(tpls)
    before = owned(arena)
    with monkeypatch.context() as m:
        fail_at(m, where, call)
        with pytest.raises(MemoryError):
            arena.retire(slots[:2])
    assert owned(arena) == before
    for res, tpl in zip(arena.retire(slots[:2]), tpls):
        assert same(res, alone(tpl, STEPS))
    late = make_templates([(3, 1500)], seed=65)[0]
    slot = arena.admit(late)  # into the ranges given back
    arena.step()
    for res, tpl, steps in zip(arena.retire([slots[2], slot]), (tpls[2], late), (STEPS + 1, 1)):
        assert same(res, alone(tpl, steps))


def test_a_slot_listed_twice_is_refused():
    tpls = make_templates([(3, 4000), (2, 700)], seed=66)
    arena, slots = arena_with(tpls)
    before = owned(arena)
    with pytest.raises(KeyError):
        arena.retire([slots[0], slots[1], slots[0]])
    assert owned(arena) == before
    for res, tpl in zip(arena.retire(slots), tpls):
        assert same(res, alone(tpl, STEPS))
