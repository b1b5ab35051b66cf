"""The block under what PyTorch lays over a call: tracers, dispatch modes, vmap, batched gradients, weights of
a tensor subclass.  Every one of them has to see operators, and the results have to be the eager ones."""

from functools import partial

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx
from torch.utils._python_dispatch import TorchDispatchMode
from torch.utils._pytree import tree_map_only
from torch.utils.checkpoint import CheckpointPolicy, checkpoint, create_selective_checkpoint_contexts

from oracle import moe_ref as R
from tests.helpers import build_block, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda"
T, E, K = 40, 16, 2
# the folded kernels, and the other ones (fp32, off-grid widths)
SHAPES = [(torch.bfloat16, 384, 384, None), (torch.bfloat16, 384, 448, 128), (torch.float32, 68, 36, 60)]


def _block(dtype, D, F, shared, train=True):
    p = make_params(E, D, F, dtype, seed=1, std=0.05, shared_F=shared)
    return build_block(p, R.RouterSpec(E, K, score_func="softmax", route_norm=True), D, F, dtype, DEV).train(train)


def _x(seed, dtype, D):
    return torch.randn(T, D, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


def _equal(got, want):
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(got, want, strict=True)):
        assert torch.equal(a, b), f"tensor {i} differs by {float((a.detach().float() - b.detach().float()).abs().max())}"


class Names(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.seen.append(str(func))
        return func(*args, **(kwargs or {}))


def _stages(dtype):
    return "gather_experts_combine_fwd" if dtype == torch.bfloat16 else "rows_experts_combine_fwd"


@pytest.mark.parametrize("dtype,D,F,shared", SHAPES)
def test_a_traced_block_computes_what_the_block_computes(dtype, D, F, shared):
    print(f"traced {dtype} D={D} F={F} shared={shared}", flush=True)
    block = _block(dtype, D, F, shared, train=False)
    block.overlap_shared_experts = False
    with torch.no_grad():
        graph = make_fx(block)(_x(1, dtype, D))
        _equal([graph(_x(2, dtype, D))], [block(_x(2, dtype, D))])
    block.train()
    params = list(block.parameters())

    def step(x):
        x = x.detach().requires_grad_()
        out = block(x)
        return (out.detach(), *torch.autograd.grad(out, [x, *params], torch.ones_like(out)))

    graph = make_fx(step)(_x(1, dtype, D))
    counted = block.tokens_per_expert_E.clone()
    got, want = graph(_x(2, dtype, D)), step(_x(2, dtype, D))
    # With a shared expert the stages add the three input gradients in another order than the one operator: two
    # roundings on either side (unit roundoff 2^-8 for bf16, 2^-24 for fp32), of sums of about the total's size.
    order = {1} if shared else set()
    _equal([t for i, t in enumerate(got) if i not in order], [t for i, t in enumerate(want) if i not in order])
    bound = 4 * 2.0 ** (-8 if dtype == torch.bfloat16 else -24)
    assert float((got[1] - want[1]).detach().float().norm()) <= bound * float(want[1].detach().float().norm())
    assert int((block.tokens_per_expert_E - counted).sum()) == 2 * T * K  # the graph counts, and so does the step


@pytest.mark.parametrize("dtype,D,F,shared", SHAPES)
def test_the_one_operator_traces_as_operators(dtype, D, F, shared):
    """The operator itself under a tracer, with gradients: what callers of ``ops.moe_block`` get."""
    from torchllmtuner_amd import ops

    print(f"traced operator {dtype} D={D} F={F} shared={shared}", flush=True)
    block = _block(dtype, D, F, shared)
    ie, params = block.routed_experts.inner_experts, list(block.parameters())
    three = block._shared_weights(dtype)

    def step(x):
        x = x.detach().requires_grad_()
        out, counts = ops.moe_block(x, block.router.gate.weight, None, None, ie.w1_EFD, ie.w3_EFD, ie.w2_EDF, three, K,
                                    "softmax", True, 1.0, 0, 0, 0, E, 1, True, True)
        return (out.detach(), counts, *torch.autograd.grad(out, [x, *params], torch.ones_like(out)))

    graph = make_fx(step)(_x(1, dtype, D))
    for seed in (2, 3):
        _equal(graph(_x(seed, dtype, D)), step(_x(seed, dtype, D)))


def test_a_dispatch_mode_sees_the_stages_by_name():
    for dtype, D, F, shared in SHAPES:
        block, x = _block(dtype, D, F, shared), _x(1, dtype, D)
        want = block(x)
        with Names() as names:
            got = block(x)
        _equal([got], [want])
        assert any(_stages(dtype) in n for n in names.seen) and not any("moe_block" in n for n in names.seen)
        # a mode around the backward alone: one operator, none of its allocations
        out = block(x.requires_grad_())
        with Names() as names:
            out.backward(torch.ones_like(out))
        assert any("moe_block_bwd" in n for n in names.seen)
        assert not any("aten.empty" in n for n in names.seen)


def test_a_selective_checkpoint_policy_chooses_among_the_stages():
    dtype, D, F, shared = SHAPES[0]
    block, asked = _block(dtype, D, F, shared), []

    def policy(ctx, op, *args, **kwargs):
        asked.append(str(op))
        return CheckpointPolicy.MUST_SAVE if _stages(dtype) in str(op) else CheckpointPolicy.PREFER_RECOMPUTE

    grads = []
    for wrapped in (True, False):
        block.zero_grad()
        x = _x(1, dtype, D).requires_grad_()
        if wrapped:
            out = checkpoint(block, x, use_reentrant=False, context_fn=partial(create_selective_checkpoint_contexts, policy))
        else:
            out = block(x)
        out.backward(_x(2, dtype, D))
        grads.append([out, x.grad, *(p.grad.clone() for p in block.parameters())])
    assert sum(_stages(dtype) in n for n in asked) == 2  # asked in the forward and in the replay
    _equal(*grads)


def test_vmap_over_the_block_equals_a_loop():
    for dtype, D, F, shared in SHAPES:
        block = _block(dtype, D, F, shared, train=False)
        block.overlap_shared_experts = False
        x = torch.stack([_x(1, dtype, D), _x(2, dtype, D)])
        with torch.no_grad():
            _equal([torch.vmap(block)(x)], [torch.stack([block(x[0]), block(x[1])])])


def test_batched_gradients_equal_a_loop():
    for dtype, D, F, shared in SHAPES:
        block, x = _block(dtype, D, F, shared), _x(1, dtype, D).requires_grad_()
        inputs = [x, *block.parameters()]
        out = block(x)
        gouts = torch.stack([_x(2, dtype, D), _x(3, dtype, D)])
        got = torch.autograd.grad(out, inputs, gouts, is_grads_batched=True, retain_graph=True)
        each = [torch.autograd.grad(out, inputs, g, retain_graph=True) for g in gouts]
        _equal(got, [torch.stack(t) for t in zip(*each)])


class Wrapped(torch.Tensor):
    """Holds its values in another tensor and has no memory of its own."""

    __torch_function__ = torch._C._disabled_torch_function_impl

    @staticmethod
    def __new__(cls, t):
        return torch.Tensor._make_wrapper_subclass(cls, t.shape, dtype=t.dtype, device=t.device)

    def __init__(self, t):
        self.t = t

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        args, kwargs = tree_map_only(Wrapped, lambda w: w.t, (args, kwargs or {}))
        return func(*args, **kwargs)


@pytest.mark.parametrize("which", ["experts", "gate"])
def test_weights_of_a_tensor_subclass_are_unwrapped_by_their_own_rules(which):
    for dtype, D, F, _ in SHAPES:
        block = _block(dtype, D, F, None, train=False).requires_grad_(False)
        x = _x(1, dtype, D)
        want = block(x)
        ie, gate = block.routed_experts.inner_experts, block.router.gate
        for module, name in ((ie, "w1_EFD"), (ie, "w3_EFD"), (ie, "w2_EDF")) if which == "experts" else ((gate, "weight"),):
            module._parameters[name] = Wrapped(module._parameters[name].data)
        assert block._forward_as_one(x) is None
        _equal([block(x)], [want])


@pytest.mark.parametrize("which", ["experts", "gate", "gate bias", "shared"])
def test_weights_that_are_plain_attributes(which):
    """What a wrapper that owns the parameters leaves in their place: a tensor set as an attribute."""
    for dtype, D, F, _ in SHAPES:
        block = _block(dtype, D, F, 64)
        block.overlap_shared_experts = False
        gate, shared = block.router.gate, block.shared_experts
        if which == "gate bias":
            gate.bias = torch.nn.Parameter(torch.linspace(-1, 1, E, device=DEV))
        x = _x(1, dtype, D)
        want = block(x)
        for module in dict(experts=[block.routed_experts.inner_experts], gate=[gate], shared=[
                shared.gate_proj, shared.up_proj, shared.down_proj]).get(which.split()[0]):
            for name in ["bias"] if which == "gate bias" else [n for n, p in module._parameters.items() if p is not None]:
                object.__setattr__(module, name, module._parameters.pop(name).detach().requires_grad_())
        assert block._forward_as_one(x) is None
        _equal([block(x)], [want])


def test_a_gradient_penalty_raises():
    for dtype, D, F, shared in SHAPES:
        block, x = _block(dtype, D, F, shared), _x(1, dtype, D).requires_grad_()
        gout = _x(2, dtype, D)
        plain = torch.autograd.grad(block(x), x, gout)[0]
        dx, = torch.autograd.grad(block(x), x, gout, create_graph=True)
        _equal([dx], [plain])
        with pytest.raises(RuntimeError, match="moe_block_bwd is not implemented"):
            dx.float().square().sum().backward()
