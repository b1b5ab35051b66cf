"""Operands that do not start where an allocation would: views into flat buffers.  The operators copy such a
one to a boundary the kernels' 16-byte accesses want; the C entry points that have a form which loads
element by element take that."""

import contextlib

import pytest
import torch

from oracle import moe_ref as R
from tests.helpers import build_block, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda"


def shifted(t, elements=1):
    """The same values one element (or more) behind the start of an allocation."""
    flat = torch.empty(t.numel() + elements, dtype=t.dtype, device=DEV)
    view = flat[elements:].view(t.shape)
    view.copy_(t.detach())
    assert t.numel() == 0 or view.data_ptr() % 16 == elements * t.element_size() % 16
    return view


@pytest.mark.parametrize("in_stages", [False, True])
@pytest.mark.parametrize("dtype,T,D,E,F,shared", [
    (torch.bfloat16, 33, 384, 16, 384, None),    # folded kernels, few rows
    (torch.bfloat16, 1100, 512, 64, 448, 384),   # the 128-token gate kernels
    (torch.bfloat16, 200, 72, 17, 100, 60),      # any width, few experts' gate gradients
    (torch.float32, 65, 100, 5, 92, 64),
    (torch.float32, 129, 33, 12, 31, None)])     # strided kernels
def test_block_with_misaligned_operands_equals_the_aligned_one(dtype, T, D, E, F, shared, in_stages):
    print(f"misaligned block {dtype} T={T} D={D} E={E} F={F} shared={shared} stages={in_stages}", flush=True)
    p = make_params(E, D, F, dtype, seed=T, std=0.05, shared_F=shared)
    p.expert_bias_E = torch.linspace(-0.1, 0.1, E)
    g = torch.Generator().manual_seed(T)
    x, gout = (torch.randn(T, D, generator=g).to(dtype).to(DEV) for _ in range(2))

    def run(move):
        block = build_block(p, R.RouterSpec(E, 2, score_func="sigmoid", route_norm=True), D, F, dtype, DEV,
                            load_balance_coeff=1e-3).train()
        block.router.gate.bias = torch.nn.Parameter(torch.linspace(-1, 1, E, device=DEV))
        block.overlap_shared_experts = False
        for q in block.parameters():
            q.data = move(q.data)
        block._buffers["expert_bias_E"] = move(block.expert_bias_E)
        if in_stages:
            block.router.register_forward_hook(lambda *a: None)
        xin = move(x).requires_grad_()
        out = block(xin)
        out.backward(move(gout))
        with torch.no_grad():
            plain = block.eval()(xin)
        return [out.detach(), plain, xin.grad, block.tokens_per_expert_E] + [q.grad for q in block.parameters()]

    for i, (a, b) in enumerate(zip(run(shifted), run(lambda t: t))):
        assert torch.equal(a, b), f"tensor {i} differs by {float((a.float() - b.float()).abs().max())}"


@pytest.mark.parametrize("dtype,D,F,shared", [(torch.bfloat16, 384, 448, 128), (torch.float32, 68, 36, 60)])
def test_what_the_backward_reads_may_come_back_from_a_hook_anywhere(dtype, D, F, shared):
    print(f"saved-tensor hooks {dtype} D={D}", flush=True)
    p = make_params(16, D, F, dtype, seed=2, std=0.05, shared_F=shared)
    g = torch.Generator().manual_seed(3)
    x, gout = (torch.randn(70, D, generator=g).to(dtype).to(DEV) for _ in range(2))

    def run(hooks):
        block = build_block(p, R.RouterSpec(16, 2, score_func="softmax", route_norm=True), D, F, dtype, DEV).train()
        xin = x.clone().requires_grad_()
        with hooks:
            out = block(xin)
        out.backward(gout)
        return [out.detach(), xin.grad] + [q.grad for q in block.parameters()]

    away = torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: shifted(t, 3))
    want = run(contextlib.nullcontext())
    for hooks in (away, torch.autograd.graph.save_on_cpu()):
        for i, (a, b) in enumerate(zip(run(hooks), want, strict=True)):
            assert torch.equal(a, b), f"tensor {i}"
    block = build_block(p, R.RouterSpec(16, 2, score_func="softmax", route_norm=True), D, F, dtype, DEV).eval()
    with torch.inference_mode():
        assert torch.equal(block(x.clone()), want[0])


def _call(name, *args):
    from torchllmtuner_amd import _lib

    rc = getattr(_lib.load(), name)(*[a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args],
                                    torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, name)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_c_entries_of_the_experts_take_misaligned_matrices(dtype):
    """One operand off its boundary at a time, then all of them, against the aligned call (which is tested against
    fp64): another kernel, so the same sums in another order."""
    from torchllmtuner_amd import ops

    print(f"misaligned experts {dtype}", flush=True)
    counts, D, F = [33, 0, 70, 1], 68, 100
    E, R_, code = len(counts), sum(counts), 0 if dtype == torch.float32 else 1
    g = torch.Generator().manual_seed(5)
    mk = lambda *s, std=0.1: torch.randn(*s, generator=g).mul(std).to(dtype).to(DEV)
    x, dy = mk(R_, D, std=1.0), mk(R_, D, std=1.0)
    w = dict(w1=mk(E, F, D), w3=mk(E, F, D), w2=mk(E, D, F))
    plan = ops.segments_from_counts(torch.tensor(counts, dtype=torch.int32, device=DEV), R_)
    seg = [*plan.segments()]
    names = ["rows", "w1", "w3", "w2", "gate", "up", "h", "y", "dy", "dgate", "dup", "drows", "dw1", "dw3", "dw2"]

    def run(off):
        like = dict(rows=x, dy=dy, **w, gate=x.new_zeros(R_, F), up=x.new_zeros(R_, F), h=x.new_zeros(R_, F),
                    y=torch.zeros_like(x), dgate=x.new_zeros(R_, F), dup=x.new_zeros(R_, F), drows=torch.zeros_like(x),
                    **{"d" + k: torch.zeros_like(v) for k, v in w.items()})
        t = {n: shifted(v) if n in off else v for n, v in like.items()}
        _call("mi355_grouped_swiglu_fwd", t["rows"], None, R_, t["w1"], t["w3"], t["w2"], code, *seg, plan.tile_capacity, t["gate"],
              t["up"], t["h"], t["y"], E, D, F, R_)
        _call("mi355_grouped_swiglu_bwd", t["dy"], t["rows"], None, R_, t["w1"], t["w3"], t["w2"], t["gate"], t["up"], t["h"], code,
              *seg, plan.tile_capacity, t["dgate"], t["dup"], t["drows"], t["dw1"], t["dw3"], t["dw2"], E, D, F, R_)
        lin, dx, dw = (shifted(v) if "y" in off else v for v in (x.new_zeros(R_, F), torch.zeros_like(x), torch.zeros_like(w["w1"])))
        _call("mi355_grouped_linear_fwd", t["rows"], t["w1"], code, *seg, plan.tile_capacity, lin, E, D, F, R_)
        _call("mi355_grouped_linear_bwd", t["h"], t["rows"], t["w1"], code, *seg, plan.tile_capacity, dx, dw, E, D, F, R_)
        return [t[n] for n in ("gate", "up", "h", "y", "dgate", "dup", "drows", "dw1", "dw3", "dw2")] + [lin, dx, dw]

    want = run(())
    # a rounding of every intermediate to bf16 that falls the other way now and then; fp32 sums of 100 terms
    tol = 2 ** -8 if dtype == torch.bfloat16 else 2e-6
    for off in [(n,) for n in names] + [tuple(names)]:
        for i, (a, b) in enumerate(zip(run(off), want)):
            err = float((a.double() - b.double()).norm() / b.double().norm())
            assert err < tol, f"{off}: tensor {i}: {err}"


@pytest.mark.parametrize("dtype,T,D,E", [(torch.bfloat16, 300, 128, 64), (torch.bfloat16, 77, 72, 17), (torch.float32, 77, 72, 17)])
def test_c_entries_of_the_gate_take_misaligned_matrices(dtype, T, D, E):
    from torchllmtuner_amd import _lib

    print(f"misaligned gate {dtype} T={T} D={D} E={E}", flush=True)
    lib, code = _lib.load(), 0 if dtype == torch.float32 else 1
    g = torch.Generator().manual_seed(T)
    x, w, dl, add = (torch.randn(*s, generator=g).to(t).to(DEV) for s, t in (
        ((T, D), dtype), ((E, D), torch.float32), ((T, E), torch.float32), ((T, D), dtype)))
    bias = torch.randn(E, generator=g).to(DEV)
    ws = torch.empty(max(lib.mi355_router_gate_bwd_workspace_bytes(T, D, E), lib.mi355_router_gate_fwd_workspace_bytes(T, D, E)) + 16,
                     dtype=torch.uint8, device=DEV)
    logits = x.double() @ w.double().T + bias.double()
    dx, dw = dl.double() @ w.double(), dl.double().T @ x.double()
    names = ["x", "w", "dl", "add", "bias", "logits", "dx", "dw"]
    for off in [()] + [(n,) for n in names] + [tuple(names)]:
        m = lambda n, v: shifted(v) if n in off else v
        out, got_dx, got_dw = m("logits", torch.zeros_like(dl)), m("dx", torch.zeros_like(x)), m("dw", torch.zeros_like(w))
        xs, wsh, dls, adds = m("x", x), m("w", w), m("dl", dl), m("add", add)
        _call("mi355_router_gate_fwd", xs, code, wsh, 0, m("bias", bias), out, ws, T, D, E)
        _call("mi355_router_gate_add_bwd", dls, xs, code, wsh, 0, None, adds, got_dx, got_dw, ws, T, D, E)
        # fp32 sums of D, E and T terms; dx rounded to its type, added to and rounded again
        for name, got, want, tol in (("logits", out, logits, 2e-6), ("dw", got_dw, dw, 2e-6),
                                     ("dx", got_dx, dx + add.double(), 2e-6 if dtype == torch.float32 else 2 ** -8)):
            err = float((got.double() - want).norm() / want.norm())
            assert err < tol, f"{off}: {name}: {err}"
