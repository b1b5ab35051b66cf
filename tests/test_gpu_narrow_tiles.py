"""Backward products of few experts on 128-column tiles against fp32 products and the same on 256-column ones, and the folded backward's pieces of the score
gradient.  Their forward, of as few rows, runs on 64-row passes (its row tiles: test_gpu_forward_tiles.py)."""

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


def wide(plan):
    """The same plan with room for so many row tiles that no row-tiled product of it runs on narrow ones."""
    import dataclasses

    room = 4096 + plan.num_local_experts
    grow = lambda t: torch.cat([t, t.new_zeros(room - t.numel())])
    return dataclasses.replace(plan, tile_expert=grow(plan.tile_expert), tile_row0=grow(plan.tile_row0), tile_capacity=room)


def row_errors(got, want):
    """Of each row: one wrong row does not vanish among the others."""
    got, want = got.double(), want.double()
    live = want.norm(dim=-1) > 0
    assert torch.equal(got[~live], want[~live])
    return float(((got - want).norm(dim=-1)[live] / want.norm(dim=-1)[live]).max())


# K choices a token and segments that are multiples of `align` rows; the shapes of the test above, and one with 3 slots of 640 columns
@pytest.mark.parametrize("T,K,El,D,Fd,align,share", [
    (420, 1, 5, 448, 576, 1, 0.5), (330, 1, 4, 640, 384, 1, 0.8), (1120, 1, 70, 384, 448, 1, 0.0), (741, 1, 3, 1024, 512, 1, 0.0),
    (200, 3, 6, 512, 640, 16, 0.4), (90, 4, 9, 384, 832, 128, 0.3), (300, 2, 7, 448, 384, 1, 1.0),
    (70, 1, 2, 2048, 448, 1, 0.0), (150, 2, 5, 448, 2048, 16, 0.0),  # rows of 4 KiB: each tile's contraction starts somewhere else
])
def test_narrow_tiles_give_the_wide_ones_bits(ops, T, K, El, D, Fd, align, share):
    print(f"narrow and wide T={T} K={K} El={El} D={D} F={Fd} align={align}", flush=True)
    g = torch.Generator().manual_seed(T + D)
    ids = torch.stack([torch.randperm(El, generator=g)[:K] for _ in range(T)])
    heavy = torch.rand(T, generator=g) < share  # one expert has most of the load, one has no rows
    ids = torch.where((ids == El - 1).any(1, keepdim=True) & (share > 0), torch.arange(K)[None], ids)
    ids[:, 0] = torch.where(heavy & ~(ids[:, 1:] == 0).any(1), 0, ids[:, 0])
    x, dout = (torch.randn(T, D, generator=g).bfloat16().to(DEV) for _ in "xd")
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(ids.to(DEV), El, align=align)
    weights = torch.rand(T, K, generator=g).to(DEV)
    total, used = int(plan.total_rows), torch.zeros(plan.row_capacity, dtype=torch.bool, device=DEV)
    used[plan.row_of_slot.long().flatten()] = True
    out = {}
    for form, q in (("narrow", plan), ("wide", wide(plan))):
        y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, q, gather=True)
        # (the backward of both from the same activations: a turned contraction's own bits are not the subject there)
        if form == "narrow":
            kept = gate, up
        dx, dw1, dw3, dw2, dweights = ops.grouped_swiglu_combine_bwd(dout, x, weights, w1, w3, w2, *kept, q)
        rows = ops.permute_rows_fwd(x, q)
        dy = ops.permute_rows_fwd(dout, q)
        plain = ops.grouped_swiglu_bwd(dy, rows, w1, w3, w2, *kept, h if form == "narrow" else out["narrow"]["h"], q)
        linear = ops.grouped_linear(rows, w1, q)
        dlinear = ops.grouped_linear_bwd(linear if form == "narrow" else out["narrow"]["linear"], rows, w1, q)
        out[form] = dict(y=y, gate=gate, up=up, h=h, linear=linear, dx=dx, dw1=dw1, dw3=dw3, dw2=dw2, dweights=dweights,
                         drows=plain[0], dw1_p=plain[1], dw3_p=plain[2], dw2_p=plain[3], dlin=dlinear[0], dwlin=dlinear[1])
    turned = ("gate", "up", "h", "y", "linear") if D == 2048 else ("y",) if Fd == 2048 else ()
    by_row = {"y", "gate", "up", "h", "linear", "drows", "dlin"}
    for name, a in out["narrow"].items():
        b = out["wide"][name]
        if name in by_row:
            a, b = a[:total][used[:total]], b[:total][used[:total]]
        if name == "dweights":
            # fp32 sums of F products in two orders: a rounding of at most half an ulp of what is summed for each of them
            tok = torch.arange(T, device=DEV)[:, None].expand(T, K)
            e = ids.to(DEV)
            dh = torch.stack([dout[tok[:, k]].float()[:, None].bmm(w2.float()[e[:, k]])[:, 0] for k in range(K)], 1)
            hk = out["narrow"]["h"].float()[plan.row_of_slot.long().view(T, K)]
            size = (dh.abs() * hk.abs()).sum(-1)
            assert bool(((a - b).abs() <= 2 * Fd * 2.0 ** -24 * size).all())
            # against fp32: dh is rounded to bf16 before it meets h
            assert bool(((a - (dh * hk).sum(-1)).abs() <= (2.0 ** -8 + Fd * 2.0 ** -24) * size).all())
        elif name in turned:
            # two bf16 roundings (h: of three factors each) of fp32 sums in different orders
            assert row_errors(a, b) < (2.0 ** -6 if name in ("h", "y") else 2.0 ** -8), name
        else:
            assert torch.equal(a, b), f"{name} differs by {float((a.float() - b.float()).abs().max())}"
    # what both are: rows against fp32 products, one rounding each
    e_of = torch.bucketize(torch.arange(total), plan.seg_offsets[1:].cpu().long(), right=True).to(DEV)
    tok = plan.token_of_row[:total].long()  # (of a padding row: no token)
    real = used[:total]
    n = out["narrow"]
    for e in range(El):
        r = ((e_of == e) & real).nonzero()[:, 0]
        if len(r):
            assert row_errors(n["gate"][r], x[tok[r]].float() @ w1[e].float().T) < 2.0 ** -8
            assert row_errors(n["up"][r], x[tok[r]].float() @ w3[e].float().T) < 2.0 ** -8
            assert row_errors(n["y"][r], n["h"][r].float() @ w2[e].float().T) < 2.0 ** -8


@pytest.mark.parametrize("T,E,K,D,Fd,kw", [
    (200, 5, 2, 512, 640, dict(dispatcher="padded", pad_multiple=16)), (333, 8, 2, 448, 576, {}),
    (400, 12, 3, 640, 384, dict(dispatcher="share", local=(2, 7))), (700, 16, 4, 1024, 512, dict(dispatcher="padded", pad_multiple=128)),
])
def test_block_on_narrow_tiles_row_by_row(T, E, K, D, Fd, kw):
    """The whole block, every output and input gradient row and every expert's gradient against the oracle."""
    from oracle import moe_ref as R
    from tests.helpers import build_block, make_params, stable_tokens

    print(f"block on narrow tiles T={T} E={E} K={K} D={D} F={Fd} {kw}", flush=True)
    spec = R.RouterSpec(E, K, score_func="softmax", route_norm=True)
    El = kw["local"][1] - kw["local"][0] if "local" in kw else None
    p = make_params(E, D, Fd, torch.bfloat16, seed=T, std=0.05, El=El)
    g = torch.Generator().manual_seed(T)
    x, gout = (torch.randn(T, D, generator=g).bfloat16() for _ in "xg")
    block = build_block(p, spec, D, Fd, torch.bfloat16, DEV, **kw).train()
    xd = x.to(DEV).requires_grad_()
    assert block._forward_as_one(xd) is not None
    out = block(xd)
    out.backward(gout.to(DEV))
    # in fp32, from the same bf16 values
    pf = make_params(E, D, Fd, torch.bfloat16, seed=T, std=0.05, El=El)
    names = ("router_w_ED", "w1_EFD", "w3_EFD", "w2_EDF")
    for name in names:
        setattr(pf, name, getattr(pf, name).float().requires_grad_())
    xr = x.float().requires_grad_()
    ref, aux = R.moe_forward(xr, pf, spec, pad_multiple=kw.get("pad_multiple"), local_experts=kw.get("local"))
    ref.backward(gout.float())
    assert stable_tokens(aux["logits"].detach(), spec).all()
    # the block's bf16 bar, for each row: h has three roundings of 2^-9, its gradient as many more
    assert row_errors(out.detach().cpu(), ref.detach()) < 2e-2
    assert row_errors(xd.grad.cpu(), xr.grad) < 3e-2
    ie = block.routed_experts.inner_experts
    for name in names[1:]:
        got, want = getattr(ie, name).grad.cpu(), getattr(pf, name).grad
        assert row_errors(got.flatten(1), want.flatten(1)) < 2e-2, name
    assert rel_l2(block.router.gate.weight.grad, pf.router_w_ED.grad) < 2e-2
