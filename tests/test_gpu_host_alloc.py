"""Results that the native operators allocate: what sees torch's factory calls sees them, and they are ordinary tensors."""
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu


class _Factories(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = 0

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen += "empty" in str(func)
        return func(*args, **(kwargs or {}))


def test_allocations(ct, dev):
    x = torch.randn((40, 256), device=dev)
    with _Factories() as m:
        ct.block_quantize(x, 32)
    assert m.seen == 2
    with torch.inference_mode():
        q, s = ct.block_quantize(x, 32)
    assert q.is_inference() and s.is_inference()
    q, s = ct.block_quantize(x, 32)
    assert not q.is_inference() and not q.requires_grad and q.is_contiguous() and q.device == dev
    assert q.untyped_storage().nbytes() == 40 * 256 and s.untyped_storage().nbytes() == 40 * 8
    torch.use_deterministic_algorithms(True)
    try:
        q2, s2 = ct.block_quantize(x, 32)
    finally:
        torch.use_deterministic_algorithms(False)
    assert torch.equal(q2.view(torch.uint8), q.view(torch.uint8)) and torch.equal(s2.view(torch.uint8), s.view(torch.uint8))
