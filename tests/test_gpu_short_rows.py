"""Forward products in passes of 64 and 128 rows against the row tiles, bit for bit, and against fp32 where a contraction is turned."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# rows at the edges of a 16-row block, a pass and a row tile, two row tiles in passes, none
ROOM = 700
COUNTS = (1, 15, 16, 17, 0, 63, 64, 65, 127, 128, 129, 200, 256, 257, 300, 5)


@pytest.fixture(scope="module")
def ops():
    from torchllmtuner_amd import ops as o

    return o


def forward(ops, x, token_of_row, w1, w3, w2, plan, expected, save):
    """(y, gate, up, h) by the kernels that `expected` rows choose."""
    from torchllmtuner_amd import _lib

    El, F, D = w1.shape
    R = ROOM * El  # (more than the plan's rows, so that enough may be expected for the row tiles)
    assert plan.row_capacity <= R
    if token_of_row is not None:
        token_of_row = torch.cat([token_of_row, token_of_row.new_zeros(R - token_of_row.numel())])
    else:
        x = torch.cat([x, x.new_zeros(R - x.shape[0], D)])
    mk = lambda n: torch.zeros(R, n, dtype=x.dtype, device=DEV)
    y, h = mk(D), mk(F)
    gate, up = (mk(F), mk(F)) if save else (None, None)
    p = lambda t: None if t is None else t.data_ptr()
    rc = _lib.load().mi355_grouped_swiglu_fwd_expecting(
        p(x), p(token_of_row), x.shape[0], p(w1), p(w3), p(w2), 1, p(plan.seg_offsets), p(plan.seg_counts), p(plan.tile_expert),
        p(plan.tile_row0), p(plan.num_tiles), plan.tile_capacity, p(gate), p(up), p(h), p(y), El, D, F, R, expected,
        torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "grouped_swiglu_fwd_expecting")
    return y, gate, up, h


# the last group of down columns half empty (384: no; 448, 576: yes), no whole number of 256-column tiles, rows of 4 KiB (turned); 128-row passes are
# for products of more columns
@pytest.mark.parametrize("D,Fd,align,save,expected", [
    (384, 384, 1, True, 9), (448, 576, 1, False, 9), (576, 448, 16, True, 9), (2048, 384, 1, True, 9), (384, 2048, 1, False, 20),
    (448, 4032, 1, True, 60), (384, 4160, 16, False, 60), (2048, 2112, 1, True, 60)])
def test_passes_give_the_row_tiles_results(ops, D, Fd, align, save, expected):
    print(f"short rows D={D} F={Fd} align={align}", flush=True)
    g = torch.Generator().manual_seed(D + Fd)
    El = len(COUNTS)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(COUNTS))
    ids = ids[torch.randperm(ids.numel(), generator=g)].to(DEV)
    x = torch.randn(ids.numel(), D, generator=g).bfloat16().to(DEV)
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(ids[:, None], El, align=align)
    row = plan.row_of_slot.flatten().long()  # (one expert a token)
    tok = plan.token_of_row
    tiles = forward(ops, x, tok, w1, w3, w2, plan, ROOM * El, save)
    passes = forward(ops, x, tok, w1, w3, w2, plan, expected * El, save)
    plain = forward(ops, x[tok.long().clamp(min=0)].contiguous(), None, w1, w3, w2, plan, expected * El, save)
    # a turned contraction adds the same products up in another order
    turned = ("gate", "up", "h", "y") if D == 2048 else ("y",) if Fd == 2048 else ()
    for name, a, b, c in zip(("y", "gate", "up", "h"), passes, tiles, plain):
        if a is None:
            continue
        a, b, c = a[row], b[row], c[row]
        assert torch.equal(a, c), name  # rows read through the index and in place
        if name not in turned:
            assert torch.equal(a, b), name
        # a bf16 step (2^-8) of a few values, rms far below: no row is another's
        assert float(((a.double() - b.double()).norm(dim=1) / b.double().norm(dim=1)).max()) < 4e-3, name
    if save:
        want = torch.empty(ids.numel(), Fd, device=DEV)
        for e in range(El):
            want[ids == e] = x[ids == e].float() @ w1[e].float().T
        # one rounding to bf16 of an fp32 sum
        assert float(((passes[1][row].float() - want).norm(dim=1) / want.norm(dim=1)).max()) < 4e-3


# one rank's share, padded segments and everything here: as one operator and by its stages
@pytest.mark.parametrize("tokens,local,align", [(64, 8, 1), (200, 8, 1), (90, 32, 1), (500, 32, 1), (60, 32, 16), (300, 8, 32)])
def test_block_and_its_stages_choose_the_same_kernels(ops, tokens, local, align):
    from torchllmtuner_amd import moe

    print(f"short rows in the block T={tokens} local={local} align={align}", flush=True)
    D, F, E, K = 512, 384, 32, 4
    gen = torch.Generator(device=DEV).manual_seed(tokens)
    with torch.device(DEV):
        if align > 1 and local == E:
            dispatcher = moe.PaddedTokenDispatcher(E, K, pad_multiple=align)
        elif local < E:
            dispatcher = moe.LocalShareTokenDispatcher(E, K, local_start=8, num_local_experts=local)
        else:
            dispatcher = moe.LocalTokenDispatcher(E, K)
        block = moe.MoE(E, moe.RoutedExperts(moe.GroupedExperts(D, F, local), dispatcher), moe.TokenChoiceTopKRouter(
            E, D, K, score_func="softmax", route_norm=True), load_balance_coeff=None).bfloat16()
        block.router.gate.float()
        with torch.no_grad():
            for p in block.parameters():
                p.normal_(generator=gen).mul_(0.05)
        x = torch.empty(tokens, D, dtype=torch.bfloat16).normal_(generator=gen)
    block.eval()
    with torch.no_grad():
        one = block(x)
        hook = block.router.register_forward_hook(lambda *a: None)  # (the stages)
        staged = block(x)
        hook.remove()
    assert torch.equal(one, staged)
