"""Experts of any width inside the one block operator, which reads the tokens' and the output gradient's rows where they lie:
against the stage operators, which copy them into row order, bit for bit."""

from __future__ import annotations

import pytest
import torch

from oracle import moe_ref as R
from tests.helpers import build_block, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype,T,D,E,K,F,kw", [
    (torch.bfloat16, 700, 68, 5, 2, 100, dict(dispatcher="padded", pad_multiple=16)),  # rows of whole and half 16-byte pieces
    (torch.bfloat16, 5000, 480, 32, 4, 400, {}),   # 128-row and 128-column tiles
    (torch.bfloat16, 333, 200, 40, 3, 332, {}),    # more experts than the joined gate backward takes
    (torch.bfloat16, 1, 64, 4, 4, 64, {}),
    (torch.float32, 700, 260, 8, 2, 516, dict(gate_bias=True)),   # 64-row tiles
    (torch.float32, 30, 64, 16, 3, 96, dict(dispatcher="share", local=(4, 12))),  # 32-row tiles, slots without a row
    (torch.float32, 4096, 64, 4, 2, 128, {}),      # contractions over many rows: indexes requested ahead
    (torch.float32, 65, 1100, 3, 1, 36, dict(shared=64)),
])
def test_rows_read_in_place_equal_copied_rows(dtype, T, D, E, K, F, kw):
    print(f"gathered experts {dtype} T={T} D={D} E={E} K={K} F={F} {kw}", flush=True)
    kw = dict(kw)
    gate_bias, shared = kw.pop("gate_bias", False), kw.pop("shared", None)
    El = kw["local"][1] - kw["local"][0] if "local" in kw else None
    spec = R.RouterSpec(E, K, score_func="softmax", route_norm=True)
    p = make_params(E, D, F, dtype, seed=T, std=0.05, shared_F=shared, El=El)
    g = torch.Generator().manual_seed(T + 1)
    x = torch.randn(T, D, generator=g).to(dtype).to(DEV)
    gout = torch.randn(T, D, generator=g).to(dtype).to(DEV)

    def run(in_stages, frozen=()):
        block = build_block(p, spec, D, F, dtype, DEV, **kw)
        if gate_bias:
            block.router.gate.bias = torch.nn.Parameter(torch.linspace(-1, 1, E, device=DEV))
        block.overlap_shared_experts = False
        if in_stages:
            block.router.register_forward_hook(lambda *a: None)
        for n, q in block.named_parameters():
            q.requires_grad_(not any(f in n for f in frozen if f != "x"))
        assert (block._forward_as_one(x) is None) == in_stages
        xin = x.clone().requires_grad_("x" not in frozen)
        out = block.train()(xin)
        out.backward(gout)
        return [out.detach(), xin.grad] + [q.grad for q in block.parameters()]

    whole = run(False)
    for i, (a, b) in enumerate(zip(run(True), whole)):
        assert torch.equal(a, b), f"tensor {i} differs by {float((a.float() - b.float()).abs().max())}"
    # a gradient that is not asked for leaves the others alone
    for frozen in (("x",), ("router.gate",), ("w1_", "w2_", "w3_"), ("x", "router.gate")):
        for i, (a, b) in enumerate(zip(run(False, frozen), whole)):
            assert a is None or torch.equal(a, b), f"{frozen}: tensor {i}"
