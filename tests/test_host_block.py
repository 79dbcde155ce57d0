"""What the native MoE block takes in place of the modules' own operations, decided on the
host: the tests run on CPU and meta tensors (no GPU needed)."""
import pytest
import torch

from ponyexl3_amd import _lib

D, E, TOKENS = 64, 12, 3


def _gate(device="cpu", dtype=torch.float16, **kw):
    return torch.nn.Linear(D, E, bias=False, device=device, dtype=dtype, **kw).requires_grad_(False)


def _x(device="cpu"):
    return torch.zeros((1, TOKENS, D), dtype=torch.float16, device=device)


def test_gate_weight_is_read_on_its_own_device_only():
    """A weight on another device than x goes through torch, which refuses it; its address
    means nothing to a kernel on x's device."""
    host = _lib.host()
    gate = _gate()
    assert host.plain_gate_weight(gate, _x()).data_ptr() == gate.weight.data_ptr()
    assert host.plain_gate_weight(gate, _x("meta")) is None
    assert host.plain_gate_weight(_gate("meta"), _x()) is None
    assert host.plain_gate_weight(_gate(dtype=torch.float32), _x()) is None
    assert host.plain_gate_weight(torch.nn.Linear(D, E, dtype=torch.float16), _x()) is None  # bias


def test_logits_are_read_on_their_own_device_only():
    host = _lib.host()
    ok = torch.zeros((1, TOKENS, E), dtype=torch.float16)
    assert host.usable_logits(ok, _x(), 0) and host.usable_logits(ok[..., :1].contiguous(), _x(), 1)
    assert not host.usable_logits(ok, _x("meta"), 0)
    assert not host.usable_logits(ok.to("meta"), _x(), 0)
    assert not host.usable_logits(ok.bfloat16(), _x(), 0)
    assert not host.usable_logits(ok[..., :5], _x(), 0)  # not contiguous
    assert not host.usable_logits(ok, _x(), 1)
