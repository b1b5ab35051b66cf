"""Products of few experts on 128-column tiles against fp32 products, and the folded backward's pieces of the score gradient."""

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


# widths that end inside a narrow tile, inside a wide one and at one; 576: five narrow tiles where wide ones leave six pieces a row.
# Then many experts: all products on wide tiles (with 70, gate/up on narrow ones for a second round that is mostly empty), also with rows
# of 4 KiB; and row tiles that are mostly full, of which only the small products are narrow
@pytest.mark.parametrize("counts,D,Fd", [((60, 0, 100, 257, 3), 448, 576), ((300, 9, 1, 17), 640, 384), ((40, 30), 2048, 448),
                                         ((16,) * 70, 384, 448), ((12,) * 100, 2048, 448), ((12,) * 100, 448, 2048),
                                         ((250, 251, 240), 1024, 512)])
def test_products(ops, counts, D, Fd):
    print(f"narrow tiles {counts[:5]} D={D} F={Fd}", flush=True)
    g = torch.Generator().manual_seed(7)
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=g)][:, None]
    x, dout = (torch.randn(R, D, generator=g).bfloat16().to(DEV) for _ in "xd")
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(ids.to(DEV), El)
    weights = torch.rand(R, 1, generator=g).to(DEV)
    y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan, gather=True)
    got = ops.grouped_swiglu_combine_bwd(dout, x, weights, w1, w3, w2, gate, up, plan)
    tok = plan.token_of_row.long()
    rows = [torch.arange(R, device=DEV)[ids.to(DEV)[tok, 0] == e] for e in range(El)]

    def by_expert(fn, like):
        out = torch.empty(like.shape, device=DEV)
        for e, r in enumerate(rows):
            out[r] = fn(e, r)
        return out

    xf, df, w1f, w3f, w2f, hf = (t.float() for t in (x[tok], dout[tok], w1, w3, w2, h))
    # one bf16 rounding of an fp32 sum: 2^-9 of each value, rms below 2e-3
    assert rel_l2(gate, by_expert(lambda e, r: xf[r] @ w1f[e].T, gate)) < 3e-3
    assert rel_l2(up, by_expert(lambda e, r: xf[r] @ w3f[e].T, up)) < 3e-3
    assert rel_l2(y, by_expert(lambda e, r: hf[r] @ w2f[e].T, y)) < 3e-3
    dx, dw1, dw3, dw2, dweights = got
    slot = plan.row_of_slot.flatten().long()  # (one expert a token: its row)
    scale = weights[tok]
    dh = by_expert(lambda e, r: df[r] @ w2f[e], h)
    gf, uf = gate.float(), up.float()
    sig = torch.sigmoid(gf)
    assert rel_l2(dweights.flatten(), (dh * hf).sum(1)[slot]) < 1e-2
    dh = dh * scale
    dg, du = dh * uf * sig * (1 + gf * (1 - sig)), dh * F.silu(gf)
    # several roundings in a row: dh, its products, their operands
    assert rel_l2(dx, by_expert(lambda e, r: dg[r] @ w1f[e] + du[r] @ w3f[e], dx)[slot]) < 1e-2
    for grad, a, b in ((dw1, dg, xf), (dw3, du, xf), (dw2, df, hf * scale)):
        assert rel_l2(grad, torch.stack([a[r].T @ b[r] for r in rows])) < 1e-2
