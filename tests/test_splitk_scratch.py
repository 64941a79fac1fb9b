"""Split-K slabs: one buffer per device and slot, and one of its own for work on another stream."""
import contextlib
import threading
import types

import pytest
import torch

from xotorch_support_jetson_amd.ops import linear as L
from xotorch_support_jetson_amd.train import autograd_ops as A

CPU = torch.device("cpu")


@pytest.fixture(autouse=True)
def no_capture(monkeypatch):
  monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def test_side_work_has_slabs_of_its_own():
  s = L._Scratch()
  main, second = s.splitk(CPU, 8), s.splitk(CPU, 8, slot=1)
  with s.apart("dw"):
    side = s.splitk(CPU, 8)
    with s.apart("other"):
      assert s.splitk(CPU, 8) is not side
    assert s.splitk(CPU, 8) is side
    got = []
    t = threading.Thread(target=lambda: got.append(s.splitk(CPU, 8)))  # (the calling thread's work alone)
    t.start()
    t.join()
    assert got[0] is main
  assert len({x.data_ptr() for x in (main, second, side)}) == 3
  with pytest.raises(ValueError), s.apart("dw"):
    raise ValueError
  assert s.splitk(CPU, 8) is main


def test_weight_gradients_on_the_side_stream_leave_the_main_slabs_alone(monkeypatch):
  """The backward's own GEMMs run beside them, in the same slot."""
  stream = types.SimpleNamespace(wait_stream=lambda other: None)
  monkeypatch.setattr(A, "DW_STREAM", True)
  monkeypatch.setattr(A, "_dw_stream", lambda dev: stream)
  monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: stream)
  monkeypatch.setattr(torch.cuda, "stream", lambda st: contextlib.nullcontext())
  monkeypatch.setattr(L, "scratch", L._Scratch())
  taken = []
  monkeypatch.setattr(A, "_dw", lambda dy, x, acc: taken.append(L.scratch.splitk(CPU, 8)))
  t = types.SimpleNamespace(is_cuda=True, device=CPU, record_stream=lambda st: None)
  A.own_dw(t, t, types.SimpleNamespace(cb=None))
  assert taken[0] is not L.scratch.splitk(CPU, 8)
