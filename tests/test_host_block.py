"""What the native MoE block takes in place of the modules' own operations, decided on the
host: the tests run on CPU and meta tensors (no GPU needed)."""
import pytest
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
    odd = torch.zeros(TOKENS * D + 8, dtype=torch.float16)[3:3 + TOKENS * D].view(1, TOKENS, D)
    assert odd.is_contiguous() and host.plain_gate_weight(gate, odd) is None  # not 16-byte aligned
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


def _block(shared=False):
    from ponyexl3_amd import EXL3MoEBlock, EXL3SwitchGLU

    e, d, h, k = 3, 128, 128, 2
    z = lambda *s: torch.zeros(s, dtype=torch.float16)
    t = lambda *s: torch.zeros(s, dtype=torch.int16)
    switch = EXL3SwitchGLU(gu_trellis=t(8, e * 2 * 8, 32), gu_suh=z(e, 2, d), gu_svh=z(e, 2 * h),
                           dn_trellis=t(8, e * 8, 32), dn_suh=z(e, h), dn_svh=z(e, d), k=k, cb=0)
    lin = lambda n: torch.nn.Linear(d, n, bias=False)
    return EXL3MoEBlock(lin(e - shared), lin(1) if shared else None, switch, 1)


def _hook(*args, **kw):
    return None


@pytest.mark.parametrize("change", [
    lambda b, m: m.setattr(b, "route", b.route),
    lambda b, m: m.setattr(b, "_select", b._select),
    lambda b, m: m.setattr(b.switch_mlp, "forward", b.switch_mlp.forward),
    lambda b, m: m.setattr(type(b), "route", lambda self, x: None),
    lambda b, m: m.setattr(type(b.switch_mlp), "forward", lambda self, x, i: None),
    lambda b, m: m.setattr("ponyexl3_amd.moe.route_topk", lambda *a: None),
    lambda b, m: m.setattr("ponyexl3_amd.moe.combine_experts", lambda *a: None),
    lambda b, m: m.setattr(torch.nn.Linear, "forward", lambda self, x: x),
    lambda b, m: setattr(b.switch_mlp, "__class__", type("Sub", (type(b.switch_mlp),), {})),
    lambda b, m: b.switch_mlp.register_forward_hook(_hook),
    lambda b, m: b.switch_mlp.register_full_backward_hook(_hook),
    lambda b, m: _nn().register_module_forward_hook(_hook),
    lambda b, m: _nn().register_module_forward_pre_hook(_hook),
    lambda b, m: _nn().register_module_full_backward_hook(_hook),
])
def test_block_does_not_pass_by_what_a_caller_changed(change, monkeypatch):
    """Replaced methods and functions, hooks on the experts and hooks on all modules are
    reached through the modules; without them the native block stands in."""
    block = _block()
    assert block._is_as_defined(block.switch_mlp)
    handle = change(block, monkeypatch)
    try:
        assert not block._is_as_defined(block.switch_mlp)
    finally:
        if hasattr(handle, "remove"):
            handle.remove()


def _nn():
    import torch.nn.modules.module as m

    return m


def test_gates_are_called_in_order():
    """The router's gate first, then the shared expert's, as their side effects may show."""
    block, seen = _block(shared=True), []
    block.gate.register_forward_hook(lambda *a: seen.append("gate"))
    block.shared_expert_gate.register_forward_hook(lambda *a: seen.append("shared"))
    block.route(torch.zeros((1, 2, 128)))
    assert seen == ["gate", "shared"]


@pytest.mark.parametrize("hook", ["register_forward_hook", "register_forward_pre_hook",
                                  "register_full_backward_hook", "register_full_backward_pre_hook"])
def test_hooked_gate_is_called(hook):
    gate = _gate()
    handle = getattr(gate, hook)(_hook)
    assert _lib.host().plain_gate_weight(gate, _x()) is None
    handle.remove()
    assert _lib.host().plain_gate_weight(gate, _x()) is not None
    gate.forward = gate.forward
    assert _lib.host().plain_gate_weight(gate, _x()) is None


class _Sub(torch.Tensor):
    pass


def _dual(t):
    return torch.autograd.forward_ad.make_dual(t, torch.ones_like(t))


def test_values_with_a_meaning_of_their_own_go_through_torch():
    """Subclasses and forward-mode tangents: in the gate's weight and in logits."""
    host = _lib.host()
    gate = _gate()
    logits = torch.zeros((1, TOKENS, E), dtype=torch.float16)
    assert not host.usable_logits(logits.as_subclass(_Sub), _x(), 0)
    assert not host.usable_logits(logits.clone().requires_grad_(), _x(), 0)
    gate._parameters["weight"] = gate.weight.detach().as_subclass(_Sub)
    assert host.plain_gate_weight(gate, _x()) is None
    with torch.autograd.forward_ad.dual_level():
        assert not host.usable_logits(_dual(logits), _x(), 0)
        gate._parameters["weight"] = _dual(_gate().weight)
        assert host.plain_gate_weight(gate, _x()) is None
    assert host.usable_logits(logits, _x(), 0)


def test_watched_operations():
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    host = _lib.host()

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    assert not host.operations_watched()
    for mode in (Function(), Dispatch()):
        with mode:
            assert host.operations_watched()
    torch.set_autocast_enabled("cuda", True)  # (the context manager needs a GPU)
    try:
        assert host.operations_watched()
    finally:
        torch.set_autocast_enabled("cuda", False)
    with torch.device("cpu"):  # only where new tensors go
        assert not host.operations_watched()
        with Function():
            assert host.operations_watched()
    inside = []
    torch.func.vmap(lambda v: inside.append(host.operations_watched()) or v)(torch.zeros(2))
    torch.jit.trace(lambda v: inside.append(host.operations_watched()) or v + 1, torch.zeros(2), check_trace=False)
    assert inside == [True, True]
    assert not host.operations_watched()


def test_layers_and_experts_off_the_gpu_are_refused():
    """A module whose weights are in host memory must not hand their address to a kernel,
    whatever the input's device: the modules' calls say so before anything is launched."""
    from ponyexl3_amd import EXL3Linear, FusedEXL3Group, make_exl3_layer

    layers = [make_exl3_layer(k=4, in_features=128, out_features=128, seed=i, key=str(i)) for i in range(2)]
    x = torch.zeros((1, 128), dtype=torch.float16)
    with pytest.raises(ValueError, match="trellis must live on the GPU"):
        EXL3Linear(layers[0], "cpu")(x)
    with pytest.raises(ValueError, match="trellis must live on the GPU"):
        FusedEXL3Group(layers, "cpu").forward_all(x)
    with pytest.raises(ValueError, match="on the GPU"):
        _block().switch_mlp(x.view(1, 1, 128), torch.zeros((1, 1, 1), dtype=torch.int32))
    with pytest.raises(ValueError, match="16\\*K"):
        _lib.host().Linear(torch.zeros((8, 8, 48), dtype=torch.int16), 4, 0, None, None, None, None, None, None)


def test_first_calls_of_two_threads_do_not_wait_for_each_other():
    """The class of a plain gate is imported on the first call; the import lets other threads
    run, which then make their first call."""
    import subprocess
    import sys
    import textwrap

    from conftest import ROOT

    code = textwrap.dedent("""
        import builtins, threading, time
        import torch
        from ponyexl3_amd import _lib
        host, plain = _lib.host(), builtins.__import__
        def slow(name, *a, **kw):
            if name == "torch.nn":
                time.sleep(0.3)
            return plain(name, *a, **kw)
        gate = torch.nn.Linear(64, 8, bias=False, dtype=torch.float16)
        x, got = torch.zeros((1, 2, 64), dtype=torch.float16), []
        builtins.__import__ = slow
        threads = [threading.Thread(target=lambda: got.append(host.plain_gate_weight(gate, x))) for _ in range(3)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(got) == 3 and all(w is not None for w in got)
    """)
    subprocess.run([sys.executable, "-c", code], check=True, timeout=60, cwd=ROOT)
