"""Forward row tiles, narrow and wide, as ever and turned: which of them a call reaches, their bits, and their rows against fp32 products.

Few rows run on the 16-, 64- and 128-row passes; room for more rows, of which a plan has the ones it has, takes the same rows to the row tiles."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from tests.test_gpu_narrow_tiles import row_errors, wide

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

EDGES = (0, 1, 15, 16, 17, 48, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 300, 511, 512, 513, 769)
MIXED = (60, 0, 100, 257, 3, 1, 15, 300, 17, 200, 64, 33)
PASS, NARROW, TURNED = 0x1FF, {"gate": 0x200, "y": 0x400}, {"gate": 0x800, "y": 0x1000}


def roomy(plan, rows):
    """The plan with room for `rows` rows an expert."""
    R = rows * plan.num_local_experts
    return dataclasses.replace(plan, row_capacity=R, token_of_row=torch.cat([plan.token_of_row, plan.token_of_row.new_zeros(R - plan.row_capacity)]))


def kernels(plan, D, Fd, gather):
    from torchllmtuner_amd import _lib

    return _lib.load().mi355_grouped_fwd_kernels(1, plan.num_local_experts, D, Fd, plan.row_capacity, plan.row_capacity,
                                                 plan.num_tokens if gather else 0, plan.tile_capacity)


# widths that end inside a narrow tile, inside a wide one and at one; rows of 4 KiB, and of 8, on either side of the 200 rows an expert up to which sums are
# turned, with whole output tiles and a last one that starts early; plans whose products are all on wide tiles.  room: rows an expert (0: the plan's own)
@pytest.mark.parametrize("counts,D,Fd,align,room,narrow,turned", [
    (MIXED[:5], 448, 576, 1, 1000, "gate y", ""), ((300, 9, 1, 17), 640, 384, 16, 2000, "gate y", ""), ((250, 251, 240), 1024, 512, 1, 2000, "gate y", ""),
    ((16,) * 70, 384, 448, 1, 200, "gate y", ""), ((12,) * 100, 2048, 448, 1, 201, "", ""), ((12,) * 100, 448, 2048, 1, 201, "", ""),
    (EDGES, 384, 384, 1, 1000, "gate y", ""), (EDGES, 640, 448, 128, 1000, "gate y", ""),
    (MIXED, 2048, 448, 1, 200, "gate y", "gate"), (MIXED, 2048, 512, 16, 200, "gate y", "gate"), (MIXED, 2048, 448, 1, 201, "gate y", ""),
    (MIXED, 448, 2048, 1, 200, "y", "y"), (MIXED[1:7], 4096, 384, 1, 200, "gate y", "gate"), ((70, 0, 0, 5, 2, 9), 640, 2048, 1, 200, "gate y", "y"),
    ((12,) * 100, 2048, 448, 1, 200, "", "gate"), ((12,) * 100, 448, 2048, 1, 200, "", "y"),
    ((200,) * 16, 2048, 448, 1, 0, "gate y", "gate"), ((200,) * 15 + (201,), 2048, 448, 1, 0, "gate y", "")])
def test_forward_row_tiles(counts, D, Fd, align, room, narrow, turned):
    from torchllmtuner_amd import ops

    print(f"forward row tiles {counts[:5]} D={D} F={Fd} align={align} room={room}", flush=True)
    g = torch.Generator().manual_seed(D + Fd)
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=g)][:, None].to(DEV)
    x = torch.randn(R, D, generator=g).bfloat16().to(DEV)
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(ids, El, align=align)
    plan = roomy(plan, room) if room else plan
    is_turned = {"gate": "gate" in turned, "y": "y" in turned}
    for q, is_narrow in ((plan, {k: k in narrow for k in NARROW}), (wide(plan), dict.fromkeys(NARROW, False))):
        for gather in (True, False):
            got = kernels(q, D, Fd, gather)
            assert got & PASS == 256
            assert {k: bool(got & b) for k, b in NARROW.items()} == is_narrow
            assert {k: bool(got & b) for k, b in TURNED.items()} == dict(is_turned, gate=is_turned["gate"] and gather)
    row = plan.row_of_slot.flatten().long()  # (one expert a token)
    rows = ops.permute_rows_fwd(x, plan)
    names = ("y", "gate", "up", "h")
    forms = {}
    for name, q in (("narrow", plan), ("wide", wide(plan))):
        forms[name] = [t[row] for t in (*ops.grouped_swiglu_fwd(x, w1, w3, w2, q, gather=True), ops.grouped_linear(rows, w1, q))]
        forms[name + ", in place"] = [t[row] for t in (*ops.grouped_swiglu_fwd(rows, w1, w3, w2, q), ops.grouped_linear(rows, w1, q))]
    # what a turned sum is in has bits of its own
    bits = set(names) - ({"gate", "up", "h", "y"} if is_turned["gate"] else {"y"} if is_turned["y"] else set())
    first = forms["narrow"]
    for form, other in forms.items():
        for name, a, b in zip(names, first, other):
            if name in bits:
                assert torch.equal(a, b), (form, name)
        gate, up, h = other[1:4]
        e = ids[:, 0]
        for i in range(El):
            t = (e == i).nonzero()[:, 0]
            if len(t) == 0:
                continue
            # one bf16 rounding of an fp32 sum
            for got, want in ((gate[t], x[t].float() @ w1[i].float().T), (up[t], x[t].float() @ w3[i].float().T),
                              (other[0][t], h[t].float() @ w2[i].float().T), (other[4][t], x[t].float() @ w1[i].float().T)):
                assert row_errors(got, want) < 2.0 ** -8, form
        # from the rounded gate and up: silu's rounding and the product's
        want = torch.nn.functional.silu(gate.float()) * up.float()
        assert row_errors(h, want) < 2.0 ** -7, form
