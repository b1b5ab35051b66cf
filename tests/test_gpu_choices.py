"""The forward of a handful of tokens without a plan, against the grouped kernels it stands in for (a forward hook on the
router makes the block go by its stages), bit for bit, and against the oracle."""

from __future__ import annotations

import pytest
import torch

from oracle import moe_ref as R
from tests.helpers import build_block, make_params, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,D,E,K,F,kw", [
    (1, 2048, 128, 8, 768, {}),                       # quarters of the contraction of three steps
    (2, 384, 256, 16, 448, dict(groups=(8, 4), shared=384)),  # seven steps: quarters of one and two; more choices than waves take at once
    (3, 448, 60, 6, 384, dict(bias=True)),            # six steps, experts that are not a power of two
    (4, 512, 5, 5, 1024, {}),                         # every expert chosen by every token
    (4, 1024, 64, 1, 640, dict(gate_bias=True)),
    (5, 512, 16, 2, 384, {}),                         # one more token: the grouped kernels
    (2, 384, 32, 4, 384, dict(dispatcher="share", local=(8, 24))),  # some experts elsewhere: likewise
    (2, 384, 32, 4, 384, dict(dispatcher="padded", pad_multiple=16)),
])
def test_a_handful_of_tokens(T, D, E, K, F, kw):
    print(f"choices T={T} D={D} E={E} K={K} F={F} {kw}", flush=True)
    kw = dict(kw)
    groups, shared, bias, gate_bias = (kw.pop(k, None) for k in ("groups", "shared", "bias", "gate_bias"))
    spec = R.RouterSpec(E, K, score_func="sigmoid" if bias or groups else "softmax", route_norm=True,
                        num_expert_groups=groups and groups[0], num_limited_groups=groups and groups[1])
    El = kw["local"][1] - kw["local"][0] if "local" in kw else None
    p = make_params(E, D, F, torch.bfloat16, seed=T, std=0.05, shared_F=shared, El=El)
    if bias:
        p.expert_bias_E = torch.linspace(-0.1, 0.1, E)
    x = torch.randn(T, D, generator=torch.Generator().manual_seed(T)).bfloat16()

    def run(in_stages, train):
        block = build_block(p, spec, D, F, torch.bfloat16, DEV, load_balance_coeff=1e-3 if bias else None, **kw)
        if gate_bias:
            block.router.gate.bias = torch.nn.Parameter(torch.linspace(-1, 1, E, device=DEV))
        block.overlap_shared_experts = not in_stages
        if in_stages:
            block.router.register_forward_hook(lambda *a: None)
        with torch.no_grad():
            outs = [block.train(train)(x.to(DEV)) for _ in range(2)]
        return [*outs, block.tokens_per_expert_E]

    for train in (False, True):
        got = run(False, train)
        for a, b in zip(run(True, train), got):
            assert torch.equal(a, b), f"differs by {float((a.float() - b.float()).abs().max())}"
    if not gate_bias and "local" not in kw:
        ref, _ = R.moe_forward(x, p, spec)
        assert rel_l2(got[0], ref) < 2e-2  # the block's bf16 bar


def test_a_handful_of_tokens_in_a_captured_graph():
    print("choices captured", flush=True)
    D, E, K, F = 512, 32, 4, 384
    p = make_params(E, D, F, torch.bfloat16, seed=3, std=0.05)
    block = build_block(p, R.RouterSpec(E, K, score_func="softmax", route_norm=True), D, F, torch.bfloat16, DEV).eval()
    x = torch.randn(2, D, device=DEV).bfloat16()
    with torch.no_grad():
        block(x)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            block(x)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = block(x)
        for seed in range(3):
            x.copy_(torch.randn(2, D, generator=torch.Generator().manual_seed(seed)).bfloat16())
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, block(x))
            torch.cuda.synchronize()
