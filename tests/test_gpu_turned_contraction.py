"""Products whose contraction starts at a K step of the tile's own (weight rows a multiple of 4 KiB apart, few rows per
expert), against fp32 products of the same inputs, on the 64-row passes (turned row tiles: test_gpu_forward_tiles.py)."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from torchllmtuner_amd import ops as o

    return o


# one pass an expert and several; whole output tiles and a last one with columns left over (448 = 7 x 64, 3.5 x 128);
# row counts on both sides of the 200 rows per expert up to which the products are turned
@pytest.mark.parametrize("counts,D,Fd", [
    ((60, 0, 100, 257, 3), 2048, 512), ((60, 0, 100, 257, 3), 2048, 448), ((300, 9, 1, 17), 4096, 384),
    ((200, 200), 2048, 448), ((201, 200), 2048, 448), ((40, 30), 448, 2048), ((70, 0, 0), 640, 2048),
])
def test_turned_products(ops, counts, D, Fd):
    print(f"turned products {counts} D={D} F={Fd}", flush=True)
    g = torch.Generator().manual_seed(5)
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=g)][:, None]
    x = torch.randn(R, D, generator=g).bfloat16()
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16() for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(ids.to(DEV), El)
    y, gate, up, h = ops.grouped_swiglu_fwd(x.to(DEV), w1.to(DEV), w3.to(DEV), w2.to(DEV), plan, gather=True)
    tok, xf = plan.token_of_row.cpu().long(), x.float()
    e_of = ids[tok, 0]
    want_g = torch.stack([w1[e].float() @ xf[t] for e, t in zip(e_of, tok)])
    want_u = torch.stack([w3[e].float() @ xf[t] for e, t in zip(e_of, tok)])
    # one bf16 rounding of an fp32 sum: 2^-9 of each value, rms below 2e-3
    assert rel_l2(gate, want_g) < 3e-3 and rel_l2(up, want_u) < 3e-3
    want_y = torch.stack([w2[e].float() @ r for e, r in zip(e_of, h.cpu().float())])
    assert rel_l2(y, want_y) < 3e-3
    # h: three roundings of its own (silu, product, the operands' own)
    assert rel_l2(h, F.silu(want_g) * want_u) < 1e-2
