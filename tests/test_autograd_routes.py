"""Which tensors rptunnel.autograd hands to the library's stream-ordered calls: those on the
ring's own GPU, of a potential that lives there.  No GPU needed: the choice is made from the
tensor's device and the ring's alone."""
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
