"""A clone's copies are launched with the object's own device current, whichever device the caller has current (the copy
itself is stood in for: no GPU is needed)."""

import types

import pytest
import torch

import oppx


@pytest.mark.parametrize("dev,switched", [("cuda:1", True), ("cuda:0", False), ("cuda", False)])  # the current one is 0
def test_clone_launches_on_its_own_device(monkeypatch, dev, switched):
    dev = torch.device(dev)
    inside, launched = [], []

    class Device:
        def __init__(self, dev):
            self.dev = dev

        def __enter__(self):
            inside.append(self.dev)

        def __exit__(self, *exc):
            inside.pop()

    shim = types.SimpleNamespace(empty_like=torch.empty_like, contiguous_format=torch.contiguous_format,
                                 cuda=types.SimpleNamespace(device=Device, current_device=lambda: 0))
    monkeypatch.setattr(oppx, "copy_batch", lambda jobs, stream, max_blocks=0: launched.append((list(inside), len(jobs))))
    monkeypatch.setattr(oppx.FempicDevice, "_rebind", lambda self: None)
    monkeypatch.setattr(oppx, "raw_stream", lambda dev: ("stream", inside[-1] if inside else None))
    g = object.__new__(oppx.FempicDevice)
    g.torch, g.dev, g.pending, g.staged = shim, dev, False, False
    for name in ("pos", "vel", "lc", "p2c", "counters", "hole_bits", "charge", "hops", "work", "scratch"):
        setattr(g, name, torch.zeros(8, dtype=torch.int32))
    h = g.clone()
    assert h.dev == g.dev and h.pos.data_ptr() != g.pos.data_ptr()
    assert launched == [([dev] if switched else [], 8)]
