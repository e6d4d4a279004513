"""Host-side guarantees of the launch helpers: what they allocate, keep and
refuse.  No kernel is launched (CPU-only)."""

import weakref

import torch

from srswa import _lib

CPU = torch.device("cpu")


def test_scratch_belongs_to_one_call(monkeypatch):
    """Two calls in flight on one stream (host threads, a captured graph and an
    eager call) must not get one buffer, and none is kept after its call."""
    monkeypatch.setattr(_lib, "stream_ptr", lambda device: 0)
    a, b = _lib.scratch(CPU, 4096), _lib.scratch(CPU, 4096)
    assert a.numel() >= 4096 and a.data_ptr() % 16 == 0
    assert a.data_ptr() != b.data_ptr()
    kept = weakref.ref(a)
    del a
    assert kept() is None
    assert _lib.scratch(CPU, 0) is None
