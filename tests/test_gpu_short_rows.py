"""Forward products in passes of 64 and 128 rows against the row tiles, bit for bit where no contraction is turned, and against fp32 products."""

from __future__ import annotations

import pytest
import torch

from tests.test_gpu_narrow_tiles import row_errors

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# rows at the edges of a 16-row block, a pass and a row tile, two row tiles in passes, none
COUNTS = (1, 15, 16, 17, 0, 63, 64, 65, 127, 128, 129, 200, 256, 257, 300, 5)


@pytest.fixture(scope="module")
def ops():
    from torchllmtuner_amd import ops as o

    return o


def kernels(plan, D, F, R, expected, tokens):
    from torchllmtuner_amd import _lib

    return _lib.load().mi355_grouped_fwd_kernels(1, plan.num_local_experts, D, F, R, expected, tokens, plan.tile_capacity)


def forward(ops, x, token_of_row, w1, w3, w2, plan, R, expected, save):
    """(y, gate, up, h) by the kernels that `expected` of R rows choose."""
    from torchllmtuner_amd import _lib

    El, F, D = w1.shape
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


# the last group of down columns half empty (384: no; 448, 576: yes), no whole number of 256-column tiles; rows of 4 KiB, turned with room for up to 200 rows
# an expert; 128-row passes, which are for products of more columns; weights past the memory-side cache, read with the hint by experts of one pass alone
@pytest.mark.parametrize("D,Fd,align,save,expected,room,passes,turned,streamed", [
    (384, 384, 1, True, 9, 1000, 64, "", False), (448, 576, 1, False, 9, 700, 64, "", False), (576, 448, 16, True, 9, 700, 64, "", False),
    (2048, 384, 1, True, 9, 700, 64, "", False), (2048, 384, 1, True, 9, 200, 64, "gate", False), (384, 2048, 1, False, 20, 201, 64, "", False),
    (384, 2048, 16, True, 20, 200, 64, "y", False), (448, 4032, 1, True, 60, 700, 128, "", False), (384, 4160, 16, False, 60, 700, 128, "", False),
    (2048, 1664, 1, True, 60, 700, 128, "", False), (2048, 1664, 1, True, 60, 200, 128, "gate", False),
    (2048, 1792, 1, True, 20, 700, 64, "", True), (2048, 1792, 16, False, 20, 200, 64, "gate", True)])
def test_passes_give_the_row_tiles_results(ops, D, Fd, align, save, expected, room, passes, turned, streamed):
    print(f"short rows D={D} F={Fd} align={align} room={room}", flush=True)
    g = torch.Generator().manual_seed(D + Fd)
    El = len(COUNTS)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(COUNTS))
    ids = ids[torch.randperm(ids.numel(), generator=g)].to(DEV)
    x = torch.randn(ids.numel(), D, generator=g).bfloat16().to(DEV)
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(ids[:, None], El, align=align)
    R, flags = room * El, {"": 0, "gate": 0x800, "y": 0x1000}[turned]
    for tokens in (ids.numel(), 0):
        assert kernels(plan, D, Fd, R, expected * El, tokens) == passes + flags
        assert kernels(plan, D, Fd, R, R, tokens) & 0x1FF == 256
    assert (El * D * Fd * 6 > 320 << 20) == streamed
    row = plan.row_of_slot.flatten().long()  # (one expert a token)
    tok = plan.token_of_row
    tiles = forward(ops, x, tok, w1, w3, w2, plan, R, R, save)
    got = forward(ops, x, tok, w1, w3, w2, plan, R, expected * El, save)
    plain = forward(ops, x[tok.long().clamp(min=0)].contiguous(), None, w1, w3, w2, plan, R, expected * El, save)
    # a turned contraction adds the same products up in another order
    exempt = {"gate": ("gate", "up", "h", "y"), "y": ("y",), "": ()}[turned]
    for name, a, b, c in zip(("y", "gate", "up", "h"), got, tiles, plain):
        if a is None:
            continue
        a, b, c = a[row], b[row], c[row]
        assert torch.equal(a, c), name  # rows read through the index and in place
        if name not in exempt:
            assert torch.equal(a, b), name
        # a bf16 step (2^-8) of a few values, rms far below: no row is another's
        assert float(((a.double() - b.double()).norm(dim=1) / b.double().norm(dim=1)).max()) < 4e-3, name
    # one bf16 rounding of an fp32 sum
    y, gate, up, h = (None if t is None else t[row] for t in got)
    for e, n in enumerate(COUNTS):
        t = (ids == e).nonzero()[:, 0]
        if n and save:
            assert row_errors(gate[t], x[t].float() @ w1[e].float().T) < 2.0 ** -8
            assert row_errors(up[t], x[t].float() @ w3[e].float().T) < 2.0 ** -8
        if n:
            assert row_errors(y[t], h[t].float() @ w2[e].float().T) < 2.0 ** -8
