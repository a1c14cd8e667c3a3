"""Which tensors rptunnel.autograd hands to the library's stream-ordered calls: those on the
ring's own GPU, of a potential that lives there; and on which GPU those calls are made.  No GPU
needed: the choice is made from the tensor's device and the ring's alone."""
import contextlib
from types import SimpleNamespace

import pytest
import torch

from rptunnel import autograd


@pytest.mark.parametrize("device,spec,stream", [("cuda:0", True, False), ("cuda:1", True, True),
                                                ("cuda:2", True, False), ("cuda:1", False, False),
                                                ("cpu", True, False)])
def test_route_by_device(device, spec, stream):
    ring = SimpleNamespace(device=1, pes=SimpleNamespace(spec=object() if spec else None))
    dev = torch.device(device)
    x = SimpleNamespace(is_cuda=dev.type == "cuda", device=dev)
    assert autograd._on_device(ring, x) is stream


@pytest.mark.parametrize("current", [0, 1])
def test_calls_are_made_with_the_tensors_gpu_current(monkeypatch, current):
    """A default stream has the same handle on every GPU: it means the current one's."""
    state = {"current": current, "calls": []}

    @contextlib.contextmanager
    def device(d):
        before, state["current"] = state["current"], d.index
        yield
        state["current"] = before

    monkeypatch.setattr(torch.cuda, "current_device", lambda: state["current"])
    monkeypatch.setattr(torch.cuda, "device", device)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: SimpleNamespace(cuda_stream=0))
    lib = SimpleNamespace(rp_x=lambda h, p, s: state["calls"].append((state["current"], h, p.value)) or 0)
    monkeypatch.setattr(autograd.L, "lib", lambda: lib)
    like = SimpleNamespace(device=torch.device("cuda", 1))
    autograd._call("rp_x", SimpleNamespace(h="ring"), like, SimpleNamespace(data_ptr=lambda: 64))
    assert state == {"current": current, "calls": [(1, "ring", 64)]}
