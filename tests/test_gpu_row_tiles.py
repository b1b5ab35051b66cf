"""The wide row tiles' ring of operand stages and dealt 16-row blocks, row by row against fp32 products: row counts on either
side of a block, of a round of the four wave rows and of a tile; contractions of six K steps (the fewest) and of odd numbers of
them; more tiles than workgroups, so that one tile's operands arrive while another's results leave."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_narrow_tiles import row_errors, wide

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

EDGES = (0, 1, 15, 16, 17, 48, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 300, 511, 512, 513, 769)


@pytest.mark.parametrize("counts,D,Fd", [(EDGES, 384, 384), (EDGES, 448, 576), (EDGES, 640, 448), (EDGES[::-1], 832, 384),
                                         ((513, 1, 255) * 24, 448, 448), ((1,), 384, 448), ((4099,), 448, 384)])
def test_rows(counts, D, Fd):
    from torchllmtuner_amd import ops

    print(f"row tiles {len(counts)} experts {sum(counts)} rows D={D} F={Fd}", flush=True)
    g = torch.Generator().manual_seed(D + Fd)
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=g)][:, None]
    x, dout = (torch.randn(R, D, generator=g).bfloat16().to(DEV) for _ in "xd")
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = wide(ops.permute_plan(ids.to(DEV), El))
    weights = torch.rand(R, 1, generator=g).to(DEV)
    y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan, gather=True)
    dx, _, _, _, dweights = ops.grouped_swiglu_combine_bwd(dout, x, weights, w1, w3, w2, gate, up, plan)
    tok = plan.token_of_row.long()
    rows = ops.permute_rows_fwd(x, plan)
    linear = ops.grouped_linear(rows, w1, plan)
    dlinear = ops.grouped_linear_bwd(linear, rows, w1, plan)[0]
    gather = ops.grouped_swiglu_fwd(rows, w1, w3, w2, plan)
    assert all(torch.equal(a, b) for a, b in zip((y, gate, up, h), gather))
    slot, start = plan.row_of_slot.flatten().long(), 0
    drows = torch.empty(R, D, device=DEV)
    drows[slot] = dx.float()  # (one expert a token)
    dots = torch.empty(R, device=DEV)
    dots[slot] = dweights.flatten()
    for e, n in enumerate(counts):
        if n == 0:
            continue
        r = slice(start, start + n)
        start += n
        xe, de, s = x[tok[r]].float(), dout[tok[r]].float(), weights[tok[r]]
        # one bf16 rounding of an fp32 sum
        for got, want in ((gate[r], xe @ w1[e].float().T), (up[r], xe @ w3[e].float().T), (linear[r], xe @ w1[e].float().T),
                          (y[r], h[r].float() @ w2[e].float().T), (dlinear[r], linear[r].float() @ w1[e].float())):
            assert row_errors(got, want) < 2.0 ** -8
        gf, uf = gate[r].float(), up[r].float()
        sig = torch.sigmoid(gf)
        dh = de @ w2[e].float()
        size = (dh.abs() * h[r].float().abs()).sum(1)
        # dh is rounded to bf16 before it meets h
        assert bool(((dots[r] - (dh * h[r].float()).sum(1)).abs() <= (2.0 ** -8 + Fd * 2.0 ** -24) * size).all())
        dh = dh * s
        dg, du = dh * uf * sig * (1 + gf * (1 - sig)), dh * gf * sig
        # dh, its products with up and with the activation's derivative and the row itself: four roundings of at most 2^-9 each
        assert row_errors(drows[r], dg @ w1[e].float() + du @ w3[e].float()) < 2.0 ** -7
