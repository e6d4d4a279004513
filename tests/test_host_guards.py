"""Host-side guarantees of the launch helpers: what they allocate, keep and
refuse.  No kernel is launched (CPU-only)."""

import ctypes
import warnings
import weakref

import pytest
import torch

from srswa import _lib, dash_train, ops

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


def test_stream_of_a_host_device_is_refused(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda idx: 0, raising=False)
    for device in (CPU, torch.device("meta"), torch.zeros(1, device="cpu:0").device, torch.zeros(1, device="meta:0").device):
        with pytest.raises(ValueError, match="Expected a cuda device"):
            _lib.stream_ptr(device)
    assert _lib.stream_ptr(torch.device("cuda")) == 0 and _lib.stream_ptr(torch.device("cuda", 0)) == 0


def test_host_tensors_reach_no_launch(monkeypatch):
    """The launchers without a check of their own refuse host tensors through
    the stream they ask for, before the library is called."""
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda idx: 0, raising=False)
    launched = []

    class Lib:
        def __getattr__(self, name):
            return lambda *a: launched.append(name) or 0

    monkeypatch.setattr(_lib, "lib", Lib)
    prior, cand = torch.rand(4, 8), torch.ones(4, 8, dtype=torch.bool)
    with pytest.raises(ValueError, match="Expected a cuda device"):
        dash_train.select_forward(prior, cand, 2, 1e-4, 1.0)
    with pytest.raises(ValueError, match="Expected a cuda device"):
        dash_train.route_backward(prior, prior, cand, 1.0)
    assert launched == []


def test_backward_bias_must_cover_the_query_rows(monkeypatch):
    """A bias (and ids) of fewer rows than the queries would be read past its end."""
    monkeypatch.setattr(ops, "_require_cuda", lambda *ts: None)
    B, T, H, D, S = 1, 64, 2, 64, 3
    q, lse = torch.zeros(B, T, H, D), torch.zeros(B, T, H)
    for rows in (T // 2, T + 1):
        ids, bias = torch.zeros(B, 1, rows, S, dtype=torch.int32), torch.zeros(B, rows, S)
        with pytest.raises(RuntimeError, match="expand"):
            ops.gather_bwd(q, q, q, q, lse, q, ids, block_size=64, local_window=64, scale=1.0, bias=bias)


@pytest.mark.parametrize("shape", [(5,), (1, 5), (3, 5), (3, 1)])
def test_sample_starts_broadcast(shape):
    """Positions of one row, or of one column, stand for all of them, without
    torch's warning of a resized output."""
    pos = torch.arange(15).view(3, 5)[:shape[0] if len(shape) == 2 else 1, :shape[-1]].reshape(shape)
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        seg = ops._seg_from_positions(pos, 5, 9, CPU)
    assert seg.dtype == torch.int32
    assert torch.equal(seg.long(), torch.arange(4, 9)[None] - pos)


@pytest.mark.parametrize("rows", [(4,), (1, 4), (3, 4)])
def test_forward_reads_sample_starts_of_every_sequence(monkeypatch, rows):
    """The kernel reads seg [B, T] by its strides: one row given for three
    sequences must not be read past its end."""
    seen = []

    class Lib:
        def srswa_gather_fwd_workspace(self, a):
            return 0

        def srswa_gather_fwd_ws(self, a, ws, nws, stream):
            f = a._obj
            raw = (ctypes.c_int32 * (2 * f.seg_sb + f.T)).from_address(f.seg)
            seen.append(torch.tensor([[raw[b * f.seg_sb + t] for t in range(f.T)] for b in range(f.B)]))
            return 0

    monkeypatch.setattr(ops, "_require_cuda", lambda *ts: None)
    monkeypatch.setattr(_lib, "stream_ptr", lambda device: 0)
    monkeypatch.setattr(_lib, "lib", Lib)
    B, T, H, D = 3, 4, 2, 64
    q = torch.zeros(B, T, H, D)
    seg = torch.arange(torch.Size(rows).numel()).view(rows)
    ops.gather_fwd(q, q, q, torch.zeros(B, 1, T, 2, dtype=torch.int32), block_size=64, local_window=64, scale=1.0, seg=seg)
    assert torch.equal(seen[0].long(), seg.expand(B, T))
