"""The rings of operand stages of the wide row tiles, whose 16-row blocks are dealt to the waves, and of the weight gradients, row by
row and expert by expert against fp32 products: row counts on either side of a block, of a round of the four wave rows, of a tile and of one and two
K steps of a weight gradient; contractions of six K steps (the fewest) and of odd numbers of
them; more tiles than workgroups, so that one tile's operands arrive while another's results leave."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_narrow_tiles import row_errors, wide

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

EDGES = (0, 1, 15, 16, 17, 48, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257, 300, 511, 512, 513, 769)


# (the forward of the first and of the last two runs on passes of fewer rows: test_gpu_forward_tiles.py has the first's on row tiles)
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
    dx, dw1, dw3, dw2, dweights = ops.grouped_swiglu_combine_bwd(dout, x, weights, w1, w3, w2, gate, up, plan)
    tok = plan.token_of_row.long()
    rows = ops.permute_rows_fwd(x, plan)
    linear = ops.grouped_linear(rows, w1, plan)
    dlinear, dwlinear = ops.grouped_linear_bwd(linear, rows, w1, plan)
    gather = ops.grouped_swiglu_fwd(rows, w1, w3, w2, plan)
    assert all(torch.equal(a, b) for a, b in zip((y, gate, up, h), gather))
    slot, start = plan.row_of_slot.flatten().long(), 0
    drows = torch.empty(R, D, device=DEV)
    drows[slot] = dx.float()  # (one expert a token)
    dots = torch.empty(R, device=DEV)
    dots[slot] = dweights.flatten()
    for e, n in enumerate(counts):
        if n == 0:
            assert not any(t[e].any() for t in (dw1, dw3, dw2, dwlinear))
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
        # one rounding; and those of dh, hs or the operands above before it
        assert row_errors(dwlinear[e].flatten()[None], (linear[r].float().T @ xe).flatten()[None]) < 2.0 ** -8
        for got, want in ((dw1[e], dg.T @ xe), (dw3[e], du.T @ xe), (dw2[e], de.T @ (s * h[r].float()))):
            assert row_errors(got.flatten()[None], want.flatten()[None]) < 2.0 ** -7


@pytest.mark.parametrize("counts", [(63, 1, 70, 129, 5), (128, 200, 64, 0, 3, 65), (1,) * 20])
def test_rows_of_other_experts_stay_out_of_a_weight_gradient(counts):
    """The last K step of an expert's contraction reads past its rows: what lies there must not count, whatever it is."""
    from torchllmtuner_amd import ops

    print(f"weight gradients beside rows that are not finite {counts[:6]}", flush=True)
    g = torch.Generator().manual_seed(3)
    El, R, D, Fd = len(counts), sum(counts), 448, 384
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[:, None]
    plan = ops.permute_plan(ids.to(DEV), El)
    assert torch.equal(plan.token_of_row.cpu().long(), torch.arange(R))
    x, dy = torch.randn(R, D, generator=g).bfloat16(), torch.randn(R, Fd, generator=g).bfloat16()
    w = (torch.randn(El, Fd, D, generator=g) * 0.03).bfloat16().to(DEV)
    gate, up = (torch.randn(R, Fd, generator=g).bfloat16().to(DEV) for _ in "gu")
    w2 = (torch.randn(El, D, Fd, generator=g) * 0.03).bfloat16().to(DEV)
    weights = torch.rand(R, 1, generator=g).to(DEV)

    def grads(x, dy):
        x, dy = x.to(DEV), dy.to(DEV)
        dout = x.flip(1).contiguous()
        return [ops.grouped_linear_bwd(dy, x, w, plan)[1], *ops.grouped_swiglu_combine_bwd(dout, x, weights, w, w, w2, gate, up, plan)[1:4]]

    clean = grads(x, dy)
    start = 0
    for bad, n in enumerate(counts):
        if n:
            xb, dyb = x.clone(), dy.clone()
            xb[start:start + n], dyb[start:start + n] = float("nan"), float("inf")
            for a, b in zip(clean, grads(xb, dyb)):
                for e in range(El):
                    assert torch.equal(a[e], b[e]) if e != bad else not bool(b[e].isfinite().any())
        start += n


# token matrices of 4 GiB less 256 and less 128 bytes, the largest that 32-bit byte offsets reach (rows are whole 128-byte lines)
@pytest.mark.parametrize("T,D", [(5592405, 384), (1082401, 1984)])
def test_rows_past_a_segment_of_the_largest_gathered_matrix(T, D):
    """No token's row stands in for the rows past an expert's last one, not even the matrix's first, which is not finite here."""
    from torchllmtuner_amd import _lib, ops

    assert T * D * 2 in (2 ** 32 - 256, 2 ** 32 - 128)
    print(f"gathered matrix {T} x {D}", flush=True)
    lib, Fd, counts = _lib.load(), 384, (1, 63, 64, 65, 130)
    g = torch.Generator(device=DEV).manual_seed(D)
    El, R = len(counts), sum(counts)
    plan = ops.permute_plan(torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[:, None].to(DEV), El)
    tok = torch.randint(1, T, (R,), generator=g, device=DEV, dtype=torch.int32)
    tok[:1], tok[-1:] = T - 1, T - 1
    normal = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    x = torch.zeros(T, D, dtype=torch.bfloat16, device=DEV)  # the tokens, and the output gradient of dW2
    x[tok.long()] = normal(R, D)
    x[0] = float("nan")
    dgate, dup, hs = (normal(R, Fd) for _ in "gus")
    dw1, dw3, dw2 = (torch.empty(El, *s, dtype=torch.bfloat16, device=DEV) for s in ((Fd, D), (Fd, D), (D, Fd)))
    w, gate, dots = normal(El, Fd, D), normal(R, Fd), torch.empty(R, 4, device=DEV)
    scale = torch.ones(R, device=DEV)
    at = lambda t: t.data_ptr()
    for stage in (16, 32, 64):  # dW2, dW1, dW3
        assert lib.mi355_grouped_swiglu_combine_bwd(
            at(x), at(x), at(tok), T, at(scale), at(w), at(w), at(w), at(gate), at(gate), 1, at(plan.seg_offsets), at(plan.seg_counts),
            at(plan.tile_expert), at(plan.tile_row0), at(plan.num_tiles), plan.tile_capacity, at(dgate), at(dup), at(hs), at(dots), None,
            at(dw1), at(dw3), at(dw2), El, D, Fd, R, stage, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    start = 0
    for e, n in enumerate(counts):
        r = slice(start, start + n)
        start += n
        xe = x[tok[r].long()].float()
        for got, want in ((dw1[e], dgate[r].float().T @ xe), (dw3[e], dup[r].float().T @ xe), (dw2[e], xe.T @ hs[r].float())):
            # one bf16 rounding of an fp32 sum
            assert bool(got.isfinite().all()) and row_errors(got.flatten()[None], want.flatten()[None]) < 2.0 ** -8


# rows an expert on either side of the 16 a pass takes; contractions of six steps (one or two a wave) and seven; weights past the
# memory-side cache, read with the non-temporal hint, of experts with a few rows (El = 40) and with one row tile (the last)
@pytest.mark.parametrize("counts,D,Fd", [((16, 0, 17, 1, 33, 5, 15, 2), 384, 448), ((40, 3, 1, 0, 0, 9), 448, 384), ((1,), 384, 640), ((60,), 1024, 512),
                                         ((3, 1, 20, 0) * 10, 2048, 768), ((200, 9, 40, 256) * 10, 2048, 768)])
def test_few_rows_and_streamed_weights(counts, D, Fd):
    from torchllmtuner_amd import ops

    print(f"few rows {counts[:8]} D={D} F={Fd}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(D)
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=torch.Generator().manual_seed(1))][:, None]
    normal = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=DEV) * std).bfloat16()
    x, w1, w3, w2 = normal(R, D), normal(El, Fd, D, std=0.03), normal(El, Fd, D, std=0.03), normal(El, D, Fd, std=0.03)
    plan = ops.permute_plan(ids.to(DEV), El)
    y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan, gather=True)
    if R <= 8 * El or D % 2048:  # (beyond, rows of 4 KiB are summed in turned order where they are gathered)
        copied = ops.grouped_swiglu_fwd(ops.permute_rows_fwd(x, plan), w1, w3, w2, plan)
        assert all(torch.equal(a, b) for a, b in zip((y, gate, up, h), copied))
    tok, start = plan.token_of_row.long(), 0
    for e, n in enumerate(counts):
        r = slice(start, start + n)
        start += n
        if n:
            xe = x[tok[r]].float()
            for got, want in ((gate[r], xe @ w1[e].float().T), (up[r], xe @ w3[e].float().T), (y[r], h[r].float() @ w2[e].float().T)):
                assert row_errors(got, want) < 2.0 ** -8


# the shared expert's gate/up tiles, four to 256 tokens, on either side of seven eighths of the CUs, one and one and a half rounds of them
@pytest.mark.parametrize("tokens", [56 * 256, 57 * 256 - 3, 64 * 256, 65 * 256, 96 * 256, 96 * 256 + 1])
def test_shared_expert_beside_the_router(tokens):
    """Beside the router on fewer workgroups, or in place on all: the same bits, forward and in the shared expert's gradients."""
    from tests.helpers import build_block, make_params
    from oracle import moe_ref as R

    print(f"shared expert beside the router, {tokens} tokens", flush=True)
    D, E, Fd = 384, 8, 384
    block = build_block(make_params(E, D, Fd, torch.bfloat16, seed=1, std=0.05, shared_F=448), R.RouterSpec(E, 1), D, Fd, torch.bfloat16, DEV)
    x, gout = (torch.randn(tokens, D, generator=torch.Generator(device=DEV).manual_seed(i), device=DEV).bfloat16() for i in (1, 2))
    results = []
    for overlap in (True, False, True):
        block.overlap_shared_experts = overlap
        block.zero_grad()
        out = block(x)
        out.backward(gout)
        results.append([out.detach().clone(), *(p.grad.clone() for p in block.shared_experts.parameters())])
    for other in results[1:]:
        assert all(torch.equal(a, b) for a, b in zip(results[0], other))


def test_two_weight_gradients_in_one_launch_and_in_two():
    """Many experts of one K step each: two launches; the same segments with room for more rows: one."""
    from torchllmtuner_amd import ops

    print("weight gradients in one launch and in two", flush=True)
    El, D, Fd = 256, 448, 1088  # 2560 tiles
    gen = torch.Generator(device=DEV).manual_seed(5)
    normal = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device=DEV).normal_(generator=gen)
    counts = torch.arange(El, device=DEV) % 7
    ids = torch.repeat_interleave(torch.arange(El, device=DEV), counts)[:, None]
    x, dout, w1, w3, w2 = normal(ids.shape[0], D), normal(ids.shape[0], D), normal(El, Fd, D), normal(El, Fd, D), normal(El, D, Fd)
    plan, weights = ops.permute_plan(ids, El), torch.rand(ids.shape[0], 1, device=DEV, generator=gen)
    _, gate, up, _ = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan, gather=True)
    apart, together = (ops.grouped_swiglu_combine_bwd(dout, x, weights, w1, w3, w2, gate, up, q) for q in (plan, wide(plan)))
    for name, a, b in zip(("dx", "dw1", "dw3", "dw2", "dweights"), apart, together):
        assert torch.equal(a, b), name
    assert not torch.equal(apart[1], apart[2])
