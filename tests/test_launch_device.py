"""Launches happen with the tensors' device current and on its stream, whatever device the
caller has current (on the CPU: tensors, streams and the library call are stand-ins)."""
from __future__ import annotations

import contextlib

import pytest
import torch


class _OnGpu1:
    """What an op reads of a contiguous tensor on the second GPU."""
    device = torch.device("cuda", 1)
    is_cuda = True

    def __init__(self, *shape, dtype=torch.float16):
        self.shape, self.dtype = torch.Size(shape), dtype

    def dim(self):
        return len(self.shape)

    def numel(self):
        return self.shape.numel()

    def stride(self, *i):
        return 1

    def data_ptr(self):
        return 4096

    def contiguous(self):
        return self

    def is_contiguous(self):
        return True

    reshape = view = lambda self, *a: self


def _i32(*shape):
    return _OnGpu1(*shape, dtype=torch.int32)


CALLS = {
    "ivakv_rms_norm": lambda o, h: o.rms_norm(h(4, 64), h(64), 1e-6),
    "ivakv_swiglu": lambda o, h: o.swiglu(h(4, 64), h(4, 64)),
    "ivakv_linear_rows": lambda o, h: o.linear_rows(h(4, 64), (h(32, 64),)),
    "ivakv_chunk_slots": lambda o, h: o.chunk_slots(_i32(2, 4), _i32(2), 3),
    "ivakv_append": lambda o, h: o.kv_append(h(3, 2, 64), h(3, 2, 64), h(8, 2, 8, 16, 8), h(8, 2, 64, 16), _i32(3)),
    "ivakv_gather": lambda o, h: o.kv_gather(h(8, 2, 8, 16, 8), h(8, 2, 64, 16), _i32(2, 4), _i32(2)),
}


@pytest.mark.parametrize("current", [0, 1])
@pytest.mark.parametrize("entry", CALLS)
def test_launch_enters_the_tensors_device(iva, monkeypatch, entry, current):
    ops, state, seen = iva.ops, {"current": current}, []

    @contextlib.contextmanager
    def enter(dev):
        before, state["current"] = state["current"], dev.index
        yield
        state["current"] = before

    monkeypatch.setattr(torch.cuda, "device", enter)
    monkeypatch.setattr(torch.cuda, "current_device", lambda: state["current"])
    monkeypatch.setattr(ops, "_current_device", lambda: state["current"], raising=False)
    monkeypatch.setattr(ops, "_raw_stream", lambda index: 100 + index)
    monkeypatch.setattr(torch, "empty", lambda *a, **k: _OnGpu1(4))
    monkeypatch.setattr(torch, "empty_like", lambda t: t)
    monkeypatch.setitem(ops._abi._FUNCS, entry,
                        lambda *a: seen.append((entry, state["current"], a[-1])) or ops._abi.OK)
    CALLS[entry](ops, _OnGpu1)
    assert seen == [(entry, 1, 101)]
    assert state["current"] == current
