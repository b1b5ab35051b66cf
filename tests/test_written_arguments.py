"""What the operators write in place, autograd knows of: a backward that saved its earlier value raises (on the CPU, with stand-ins for the kernels)."""

from __future__ import annotations

import pytest
import torch

from torchllmtuner_amd import ops

T, D, E, K, F, BINS = 6, 8, 4, 2, 8, 5


@pytest.fixture
def cpu_kernels():
    """The operators on CPU tensors; as the kernels do, they write through the pointers."""
    ops.moe_block  # noqa: B018  (the operators are registered with the module)

    def add_one(*tensors):
        for t in tensors:
            if t is not None:
                t.detach().numpy()[...] += 1

    def block(*a):
        add_one(a[22], a[25], *a[26:])  # (a default at the end is not handed on)
        return a[0] * 2.0, torch.ones(E, dtype=torch.int32)

    lib = torch.library.Library("mi355_moe", "IMPL")
    lib.impl("moe_block", block, "CPU")
    lib.impl("moe_block_fwd", lambda *a: (*block(*a), torch.empty(16, dtype=torch.uint8)), "CPU")
    lib.impl("quantile_observe", lambda histogram, *a: add_one(histogram), "CPU")
    yield
    lib._destroy()


def call(grad, **stats):
    g = torch.Generator().manual_seed(0)
    n = lambda *s: torch.randn(*s, generator=g).requires_grad_(grad)
    return ops.moe_block(n(T, D), n(E, D), None, torch.zeros(E), n(E, F, D), n(E, F, D), n(E, D, F), (None, None, None), K, "softmax", True,
                         1.0, None, None, 0, E, 1, True, True, **stats)


def written(kind):
    """(the tensor, a call that writes it) for each of the arguments"""
    if kind == "observe":
        t = torch.zeros(E, BINS, dtype=torch.int64)
        return t, lambda grad: torch.ops.mi355_moe.quantile_observe(t, torch.rand(T, E), torch.rand(T), torch.zeros(E), None)
    if kind == "totals":
        t = torch.zeros(E)
        return t, lambda grad: call(grad, totals=t)
    if kind == "histogram":
        t = torch.zeros(E, BINS, dtype=torch.int64)
        return t, lambda grad: call(grad, histogram=t)
    t = torch.zeros(())
    return t, lambda grad: call(grad, aux_denominator=torch.ones(()), aux_coeff=0.1, aux_acc=t)


@pytest.mark.parametrize("kind", ["totals", "histogram", "aux_acc", "observe"])
@pytest.mark.parametrize("grad", [False, True])
def test_a_value_saved_before_the_call_is_not_used_after_it(cpu_kernels, kind, grad):
    t, run = written(kind)
    p = torch.ones(t.shape, requires_grad=True)
    loss = (p * t).sum()  # saves t for p's gradient
    run(grad)
    assert t.double().sum() == t.numel() and t._version >= 1
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        loss.backward()


def test_what_it_returns_and_the_modes_are_as_before(cpu_kernels):
    """Gradients still come through the operator, and inference tensors, which have no version, are still written."""
    t, run = written("totals")
    out, counts = run(True)
    assert out.requires_grad and not counts.requires_grad and counts.dtype is torch.int32
    with torch.inference_mode():
        run(False)
        assert t._version >= 2 and float(t[0]) == 2.0
        s = torch.zeros(E)
        call(False, totals=s)
    call(False, totals=s)
    assert float(s[0]) == 2.0
