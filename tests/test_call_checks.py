"""What the wrappers refuse or leave to the stock operators, on the CPU: the tensors claim to be on the GPU and the
library is a stand-in, so that a call which would hand raw pointers to a kernel shows itself instead."""
import pytest
import torch

from qwen3_moe_fused import _lib
from qwen3_moe_fused.kernels import routing


class LibraryCalled(Exception):
    pass


class _StandIn:
    def __getattr__(self, name):
        raise LibraryCalled(name)


@pytest.fixture
def no_kernels(monkeypatch):
    monkeypatch.setattr(torch.Tensor, "is_cuda", True)
    monkeypatch.setattr(_lib, "lib", lambda: _StandIn())
    monkeypatch.setattr(_lib, "stream", lambda: 0)


def _bf16(*shape):
    return torch.ones(shape, dtype=torch.bfloat16)


@pytest.mark.parametrize("grad", [False, True])
@pytest.mark.parametrize("width", [64, 192])
def test_router_refuses_rows_of_another_width(no_kernels, width, grad):
    w = _bf16(8, 128).requires_grad_(grad)
    with pytest.raises(LibraryCalled):  # the stand-in is where a call of the right width goes
        routing.router_linear(_bf16(4, 128), w)
    x = _bf16(4, width)
    with pytest.raises(RuntimeError, match="cannot be multiplied"):
        out = routing.router_linear(x, w)
        torch.nn.functional.linear(x, w) if out is None else out
