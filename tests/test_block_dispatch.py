"""The block's operators under what PyTorch lays over a call -- tracers, dispatch modes -- without a GPU (on
meta tensors, whose backward the engine runs on the host): every route to the kernels is an operator that
these see."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode

from torchllmtuner_amd import ops

T, D, E, K, F = 40, 384, 8, 2, 448
BF = torch.bfloat16


class Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(func.__name__.split(".")[0] if "mi355_moe" in str(func) else str(func))
        return func(*args, **(kwargs or {}))


def _call(x, gate_w, w1, w3, w2, shared=(None, None, None), gate_b=None):
    return ops.moe_block(x, gate_w, gate_b, None, w1, w3, w2, shared, K, "softmax", True, 1.0, 0, 0, 0, E, 1, True, True)


def _weights(shared, bias, dtype=BF, device="meta"):
    mk = lambda *s, dtype=dtype: torch.empty(s, dtype=dtype, device=device, requires_grad=True)
    three = (mk(192, D), mk(192, D), mk(D, 192)) if shared else (None, None, None)
    return mk(E, D, dtype=torch.float32), mk(E, F, D), mk(E, F, D), mk(E, D, F), three, mk(E, dtype=torch.float32) if bias else None


@pytest.mark.parametrize("shared,bias", [(False, False), (True, False), (False, True), (True, True)])
def test_a_dispatch_mode_sees_the_block_operators_and_not_their_allocations(shared, bias):
    gate_w, w1, w3, w2, three, gate_b = _weights(shared, bias)
    x = torch.empty(T, D, dtype=BF, device="meta", requires_grad=True)
    gout = torch.empty(T, D, dtype=BF, device="meta")
    with Names() as names:
        out, counts = _call(x, gate_w, w1, w3, w2, three, gate_b)
        out.backward(gout)
    assert [n for n in names.seen if n.startswith("moe_block")] == ["moe_block_fwd", "moe_block_bwd"], names.seen
    assert not any("empty" in n for n in names.seen), names.seen
    assert (out.shape, out.dtype, counts.shape, counts.dtype) == ((T, D), BF, (E,), torch.int32)
    for t in (x, gate_w, w1, w3, w2, *three, gate_b):
        if t is not None:
            assert t.grad.shape == t.shape and t.grad.dtype == t.dtype
    with torch.no_grad(), Names() as names:
        out, counts = _call(x, gate_w, w1, w3, w2, three, gate_b)
    assert names.seen == ["moe_block"] and out.shape == (T, D)


@pytest.mark.parametrize("grad", [True, False])
def test_fake_tensors_go_through_without_a_look_at_their_memory(grad):
    with FakeTensorMode(), torch.set_grad_enabled(grad):
        x = torch.empty(T, D, dtype=BF, device="cuda", requires_grad=True)
        gate_w, w1, w3, w2, three, gate_b = _weights(True, True, device="cuda")
        for t in (x, gate_w, w1, w3, w2, *three, gate_b):
            torch._C._set_throw_on_mutable_data_ptr(t)
        out, counts = _call(x, gate_w, w1, w3, w2, three, gate_b)
        assert (out.shape, out.dtype, out.device.type, out.requires_grad) == ((T, D), BF, "cuda", grad)
        assert (counts.shape, counts.dtype, counts.device.type) == ((E,), torch.int32, "cuda")
        kept = torch.ops.mi355_moe.moe_block_fwd(x, gate_w, gate_b, None, w1, w3, w2, *three, K, 1, True, 1.0, 0, 0, 0, E, 1, True,
                                                 True, None, None, None, 0.0, None)[2]
        assert kept.dtype == torch.uint8 and kept.device.type == "cuda"


def test_a_trace_records_the_block_operators():
    gate_w, w1, w3, w2, _, _ = _weights(False, False)

    def step(x):
        x = x.detach().requires_grad_()
        out, _ = _call(x, gate_w, w1, w3, w2)
        return (out, *torch.autograd.grad(out, (x, w1), torch.ones_like(out)))

    graph = make_fx(step)(torch.empty(T, D, dtype=BF, device="meta")).graph
    targets = [str(n.target) for n in graph.nodes if n.op == "call_function"]
    assert "mi355_moe.moe_block_fwd.default" in targets and "mi355_moe.moe_block_bwd.default" in targets
    assert not any("aten.empty" in t for t in targets), targets


def test_partial_gradient_requests_reach_the_backward_operator():
    gate_w, w1, w3, w2, three, gate_b = _weights(True, True)
    for t in (gate_w, w1, three[0], three[1], three[2]):
        t.requires_grad_(False)
    x = torch.empty(T, D, dtype=BF, device="meta")
    out, _ = _call(x, gate_w, w1, w3, w2, three, gate_b)
    dw3, dgate_b = torch.autograd.grad(out, (w3, gate_b), torch.ones_like(out))
    assert dw3.shape == w3.shape and dgate_b.shape == gate_b.shape and dgate_b.dtype == torch.float32


def test_the_backward_operator_refuses_what_the_forward_did_not_keep():
    op = torch.ops.mi355_moe.moe_block_bwd
    gate_w, w1, w3, w2, _, _ = _weights(False, False)
    x = torch.empty(T, D, dtype=BF, device="meta")
    args = lambda dout, kept: (dout, x, gate_w, None, w1, w3, w2, None, None, None, kept, None, K, 1, True, 1.0, 0, E, 1,
                               True, False, True, True, False, True, False)
    with torch.no_grad():
        kept = torch.ops.mi355_moe.moe_block_fwd(x, gate_w, None, None, w1, w3, w2, None, None, None, K, 1, True, 1.0, 0,
                                                 0, 0, E, 1, True, True, None, None, None, 0.0, None)[2]
        assert [t is not None for t in op(*args(torch.empty_like(x), kept))] == [
            True, True, False, True, True, True, False, False, False]
        with pytest.raises(ValueError, match="kept"):
            op(*args(torch.empty_like(x), kept[:-256]))
        with pytest.raises(ValueError, match="gradient"):
            op(*args(torch.empty(T + 1, D, dtype=BF, device="meta"), kept))


@pytest.mark.parametrize("shared", [False, True])
def test_the_backward_has_no_derivative_and_says_so(shared):
    gate_w, w1, w3, w2, three, gate_b = _weights(shared, True)
    x = torch.empty(T, D, dtype=BF, device="meta", requires_grad=True)
    wanted = [t for t in (x, gate_w, gate_b, w1, w3, w2, *three) if t is not None]
    out, _ = _call(x, gate_w, w1, w3, w2, three, gate_b)
    grads = torch.autograd.grad(out, wanted, torch.ones_like(out), create_graph=True)  # by itself no error
    for g in grads:
        with pytest.raises(RuntimeError, match="moe_block_bwd is not implemented"):
            torch.autograd.grad(g, w1, torch.ones_like(g), retain_graph=True, allow_unused=True)
    out, _ = _call(x, gate_w, w1, w3, w2, three, gate_b)
    assert not any(g.requires_grad for g in torch.autograd.grad(out, wanted, torch.ones_like(out)))
