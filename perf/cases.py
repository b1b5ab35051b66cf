"""The work whose time this repository answers for, as cases of plain sizes.

A case is one call of what a user's program calls: a mixture-of-experts block (``MoE`` of
``torchllmtuner_amd.moe``) going forward, or forward and backward with every gradient, or the
``rms_norm`` operator of the kernel registry.  ``listed()`` holds the cases that stand for the
range, ``draw()`` gives more of the same range.

Shapes are those of ``torchllmtuner_amd.workloads`` (the block of 2048 x 128 experts x 768, the
one-rank share of 7168 x 32 of 256 experts x 2048 with its shared expert, the small fp32 block of
256 x 8 x 512) and widths of the kind the tests draw, off the matrix-core path's 64-column grid
included.  Tokens and output gradients are N(0, 1), weights N(0, 0.02), the router weight fp32.
"""

from __future__ import annotations

import torch

from torchllmtuner_amd import kernel_registry, moe, workloads

# The block of the headline benchmark, one rank's share of the large one, and the small fp32 one.
_WIDE = dict(dim=2048, experts=128, top_k=8, hidden=768, dtype="bf16", score="softmax")
_SHARE = dict(dim=7168, experts=256, top_k=8, hidden=2048, dtype="bf16", score="sigmoid", scale=2.5, groups=8,
              limited=4, local=32, shared=2048, bias=True)
_SMALL = dict(dim=256, experts=8, top_k=2, hidden=512, dtype="fp32", score="softmax")
_BALANCED = dict(dim=1024, experts=64, top_k=6, hidden=512, dtype="bf16", score="sigmoid", quantile=True, aux=True,
                 padded_tokens=True)

_DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def listed():
    return [
        # generation, one sequence: a token runs through 8 experts; host time and launches count
        dict(name="decode-1", kind="forward", tokens=1, **_WIDE),
        # generation, a batch of sequences: most experts are touched, by two rows each
        dict(name="decode-33", kind="forward", tokens=33, **_WIDE),
        # generation on one expert-parallel rank of the large model, with its shared expert
        dict(name="decode-share-128", kind="forward", tokens=128, **_SHARE),
        # a chunk of a prompt, of no particular length
        dict(name="prefill-1000", kind="forward", tokens=1000, **_WIDE),
        # a full prompt batch
        dict(name="prefill-8192", kind="forward", tokens=8192, **_WIDE),
        # a training step of the block: the headline
        dict(name="train-8192", kind="train", tokens=8192, **_WIDE),
        # the same with the load of a router that is not balanced yet, segments padded to 128 rows
        dict(name="train-skewed-16384", kind="train", tokens=16384, pad=128, skew=True, **_WIDE),
        # a training step of one expert-parallel rank of the large model
        dict(name="train-share-4096", kind="train", tokens=4096, **_SHARE),
        # experiments and tests on a small model in fp32
        dict(name="train-fp32-512", kind="train", tokens=512, **_SMALL),
        # a small bf16 model whose widths are not multiples of the matrix-core kernels' 64 columns
        dict(name="train-narrow-1531", kind="train", tokens=1531, dim=320, experts=16, top_k=4, hidden=232,
             dtype="bf16", score="softmax"),
        # a step with the quantile-balanced router, the balance loss and padded tokens in the batch
        dict(name="train-balanced-3000", kind="train", tokens=3000, **_BALANCED),
        # the norm in front of the block, forward and backward
        dict(name="norm-8192", kind="norm", rows=8192, dim=2048, dtype="bf16"),
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    family = rng.choice(["forward", "forward", "train", "train", "share-forward", "share-train", "fp32", "narrow",
                         "balanced", "norm"])
    if family in ("forward", "train"):
        # blocks around the headline's: its widths and narrower ones, fewer experts, fewer per token
        case = dict(dim=64 * rng.randint(8, 32), experts=rng.choice([16, 32, 60, 64, 128]), top_k=rng.randint(2, 8),
                    hidden=64 * rng.randint(6, 16), dtype="bf16", score=rng.choice(["softmax", "sigmoid"]))
        if rng.random() < 0.5:
            case = dict(_WIDE)
        if family == "forward":
            return dict(kind="forward", tokens=_log_int(rng, 1, 8192), **case)
        tokens = _log_int(rng, 200, 12000)
        if rng.random() < 0.3:
            case.update(pad=rng.choice([16, 128]), skew=True)
        return dict(kind="train", tokens=tokens, **case)
    if family == "share-forward":
        return dict(kind="forward", tokens=_log_int(rng, 4, 2048), **_SHARE)
    if family == "share-train":
        return dict(kind="train", tokens=_log_int(rng, 250, 4096), **_SHARE)
    if family == "fp32":
        return dict(kind="train", tokens=_log_int(rng, 64, 4096), dim=4 * rng.randint(16, 160),
                    experts=rng.choice([4, 8, 16]), top_k=rng.randint(2, 4), hidden=4 * rng.randint(24, 256),
                    dtype="fp32", score="softmax")
    if family == "narrow":
        return dict(kind="train", tokens=_log_int(rng, 64, 4096), dim=8 * rng.randint(8, 60),
                    experts=rng.choice([4, 8, 16, 32]), top_k=rng.randint(2, 4),
                    hidden=8 * rng.randint(8, 46) + rng.choice([0, 4]), dtype="bf16", score="softmax")
    if family == "balanced":
        return dict(kind="train", tokens=_log_int(rng, 256, 8192), **_BALANCED)
    return dict(kind="norm", rows=_log_int(rng, 1, 32768), dim=_log_int(rng, 128, 8192) // 4 * 4,
                dtype=rng.choice(["bf16", "bf16", "fp32"]))


# ---- inputs ------------------------------------------------------------------------------------


def _block(case, normal, tokens):
    D, E, K, F = case["dim"], case["experts"], case["top_k"], case["hidden"]
    dtype, local = _DTYPES[case["dtype"]], case.get("local")
    aux = moe.MicrobatchWiseLoadBalanceLoss(coeff=1e-3) if case.get("aux") else None
    if case.get("quantile"):
        router = moe.QuantileBalancedTopKRouter(E, D, K, route_norm=True, aux_loss=aux)
    else:
        router = moe.TokenChoiceTopKRouter(
            E, D, K, score_func=case["score"], route_norm=True, route_scale=case.get("scale", 1.0),
            num_expert_groups=case.get("groups"), num_limited_groups=case.get("limited"), aux_loss=aux)
    if case.get("pad"):
        dispatcher = moe.PaddedTokenDispatcher(E, K, pad_multiple=case["pad"])
    elif local:
        dispatcher = moe.LocalShareTokenDispatcher(E, K, local_start=0, num_local_experts=local)
    else:
        dispatcher = moe.LocalTokenDispatcher(E, K)
    shared = moe.DenseSwiGLU(D, case["shared"]) if case.get("shared") else None
    block = moe.MoE(E, moe.RoutedExperts(moe.GroupedExperts(D, F, local or E), dispatcher), router,
                    load_balance_coeff=1e-3 if case.get("bias") else None, shared_experts=shared)
    block = block.to(dtype)
    block.router.gate.float()  # the router stays fp32 under bf16 experts
    with torch.no_grad():
        for p in block.parameters():
            normal(p).mul_(0.02)
        if block.expert_bias_E is not None:
            normal(block.expert_bias_E).mul_(0.05)
        if case.get("skew"):
            logits = tokens[:4096].float() @ block.router.gate.weight.T
            bias, _ = workloads.zipf_logit_bias(logits, K)
            block.router.gate.bias = torch.nn.Parameter(bias, requires_grad=False)
    if aux is not None:
        moe.MicrobatchWiseLoadBalanceLoss.set_step_denominator(
            torch.tensor(float(tokens.shape[0] * K), device=tokens.device), model_parts=[block])
    return block.train(case["kind"] == "train")


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(t):
        return t.normal_(generator=gen)

    dtype = _DTYPES[case["dtype"]]
    with torch.device("cuda"):
        if case["kind"] == "norm":
            x = normal(torch.empty(case["rows"], case["dim"], dtype=dtype)).requires_grad_()
            weight = normal(torch.empty(case["dim"])).mul(0.1).add(1.0).to(dtype).requires_grad_()
            return dict(kind="norm", x=x, weight=weight, gout=normal(torch.empty_like(x)))
        x = normal(torch.empty(case["tokens"], case["dim"], dtype=dtype))
        block = _block(case, normal, x)
        state = dict(kind=case["kind"], block=block, x=x, mask=None)
        if case.get("padded_tokens"):
            state["mask"] = torch.rand(case["tokens"], generator=gen) < 0.05
        if case["kind"] == "train":
            x.requires_grad_()
            state["gout"] = normal(torch.empty_like(x))
            state["params"] = [p for p in block.parameters() if p.requires_grad]
    return state


# ---- one pass ----------------------------------------------------------------------------------


def run(state):
    x = state["x"]
    if state["kind"] == "forward":
        with torch.no_grad():
            return state["block"](x)
    x.grad = None
    if state["kind"] == "norm":
        weight = state["weight"]
        weight.grad = None
        y = kernel_registry.rms_norm(x, weight, 1e-6)
        y.backward(state["gout"])
        return {"y": y.detach(), "dx": x.grad, "dweight": weight.grad}
    block, params = state["block"], state["params"]
    for p in params:
        p.grad = None
    out = block(x, padding_mask=state["mask"])
    out.backward(state["gout"])
    result = {"out": out.detach(), "dx": x.grad, "grads": [p.grad for p in params],
              "tokens_per_expert": block.tokens_per_expert_E}
    balancer = getattr(block.router, "quantile_balancer", None)
    if balancer is not None:
        result["required_bias_histogram"] = balancer.required_bias_histogram_EB
    return result


# ---- what a pass cannot do without ---------------------------------------------------------------


def work(case):
    size = 4 if case["dtype"] == "fp32" else 2
    D = case["dim"]
    if case["kind"] == "norm":
        # x read, y written; x and the gradient read, dx written
        n = case["rows"] * D
        return {"bytes": size * (5 * n + 3 * D), "flops": 12 * n}
    T, E, K, F = case["tokens"], case["experts"], case["top_k"], case["hidden"]
    local, shared = case.get("local") or E, case.get("shared") or 0
    rows = T * K * local / E  # expected on the experts held here
    touched = local * (1.0 - (1.0 - K / E) ** T)  # experts with at least one row
    flops = 2.0 * T * D * E + 6.0 * rows * D * F + 6.0 * T * D * shared
    moved = size * (2 * T * D + 3 * D * (touched * F + shared)) + 4 * E * D
    if case["kind"] == "train":
        flops *= 3
        # the output gradient in, the token gradient and every weight gradient out
        moved += size * (2 * T * D + 3 * D * (local * F + shared)) + 4 * E * D
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    # 32-bit sums in another order; bf16 results and bf16 intermediate roundings.  Counts are whole and
    # stay the same; a histogram entry moves to the next bin where a score is within a rounding of the edge.
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1e-2, "differ": 0.002} if case.get("quantile") else {"rel": 1e-2}
