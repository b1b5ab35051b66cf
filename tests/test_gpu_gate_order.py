"""The order in which a logit is summed: a token whose K-th and next expert are equal to the last bits takes the one that the order
makes larger, so a token's logits, and its experts, may not depend on how many tokens its call has."""

from __future__ import annotations

import pytest
import torch

from torchllmtuner_amd import _lib, workloads

BF16, F32 = 1, 0


@pytest.mark.parametrize("dtype", [BF16, F32])
def test_slices_of_a_projection(dtype):
    """A slice is 1024 of the contraction, whatever the tokens, as long as the launch has at most 1024 workgroups of 32 x 32."""
    splits = _lib.load().mi355_router_gate_fwd_splits
    for D in (8, 64, 1000, 1024, 1032, 2048, 2880, 4096, 7168, 16384):
        for E in (1, 5, 60, 128, 130, 256, 512):
            for T in (1, 2, 4, 5, 31, 33, 200, 512, 513, 700, 1000, 1023):
                tiles = -(-T // 32) * -(-E // 32)
                assert splits(dtype, F32, T, D, E) == max(1, min(-(-D // 1024), 8, 1024 // tiles)), (T, D, E)


def gate(lib, x, w, bias):
    T, D, E = *x.shape, w.shape[0]
    work = torch.empty(lib.mi355_router_gate_fwd_workspace_bytes(T, D, E) + 16, dtype=torch.uint8, device=x.device)
    out = torch.empty(T, E, device=x.device)
    rc = lib.mi355_router_gate_fwd(x.data_ptr(), BF16 if x.dtype == torch.bfloat16 else F32, w.data_ptr(), F32, bias.data_ptr(),
                                   out.data_ptr(), work.data_ptr(), T, D, E, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return out


# tiles of 8, 16 and 32 experts (64 and 128 parts of 32 are the lines), ends inside each; rows that are no multiple of 64
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,E,lengths", [(2048, 128, (1, 4, 5, 33, 256, 257, 512, 513, 700)), (2040, 60, (1, 33, 500, 513, 900)),
                                         (1160, 5, (3, 800)), (1024, 64, (2, 999)), (7168, 256, (1, 9, 40, 130)),
                                         (520, 13, (7, 1000))])
def test_a_chunk_of_the_tokens_has_their_logits(dtype, D, E, lengths):
    lib, g = _lib.load(), torch.Generator().manual_seed(D + E)
    print(f"gate order {dtype} D={D} E={E}", flush=True)
    T = max(lengths)
    x, w = torch.randn(T, D, generator=g).to(dtype).cuda(), (torch.randn(E, D, generator=g) * 0.02).cuda()
    bias = torch.randn(E, generator=g).cuda()
    whole = gate(lib, x, w, bias)
    ref = x.double() @ w.double().T + bias.double()
    # a sum of D products, rounded to 24 bits as it grows
    assert float((whole - ref).norm() / ref.norm()) < D ** 0.5 * 2.0 ** -24
    for n in lengths:
        for first in (0, T - n):
            assert torch.equal(gate(lib, x[first:first + n], w, bias), whole[first:first + n]), (n, first)


@pytest.mark.gpu
def test_experts_of_a_skewed_router_are_a_chunks_too():
    """workloads.zipf_logit_bias bisects to a load share, which leaves a token on a tie."""
    from torchllmtuner_amd import ops

    lib = _lib.load()
    for seed in range(20):
        print(f"gate order, skewed, seed {seed}", flush=True)
        g = torch.Generator().manual_seed(seed)
        x, w = torch.randn(700, 2048, generator=g).bfloat16().cuda(), (torch.randn(128, 2048, generator=g) * 0.02).cuda()
        bias, _ = workloads.zipf_logit_bias(x.float() @ w.T, 8)
        bias = bias.float().contiguous()
        whole = ops.router_select_fwd(gate(lib, x, w, bias), None, 8, "softmax", True, 1.0)[1]
        for n in (33, 500, 513):
            assert torch.equal(ops.router_select_fwd(gate(lib, x[:n], w, bias), None, 8, "softmax", True, 1.0)[1], whole[:n]), n


# where the launches' widths change (33 and 65 tokens, 513 of more than 32 experts), by slices of a whole batch of requests, one more and one less
@pytest.mark.gpu
@pytest.mark.parametrize("T,E,K,lo,hi,splits", [
    (20, 256, 8, 0, 32, 7), (32, 256, 8, 224, 256, 8), (33, 256, 8, 0, 32, 4), (64, 256, 16, 0, 256, 5), (65, 256, 8, 0, 32, 7), (66, 33, 16, 1, 33, 8),
    (300, 128, 8, 0, 128, 6), (512, 64, 6, 0, 64, 1), (513, 64, 6, 0, 8, 2), (512, 200, 3, 0, 200, 8)])
def test_slices_in_order_and_plan_at_the_widths_of_its_launches(T, E, K, lo, hi, splits):
    """Logits are the slices' sums in their order, and ids, weights and the plan are those of the selection and the plan as two calls, with every row
    that has no slot empty."""
    from torchllmtuner_amd import ops

    print(f"route plan T={T} E={E} K={K} [{lo},{hi}) splits={splits}", flush=True)
    g = torch.Generator().manual_seed(T + E)
    partial = torch.randn(splits, T, E, generator=g).cuda()
    logits = partial[0].clone()
    for z in range(1, splits):
        logits += partial[z]
    w, ids, _ = ops.router_select_fwd(logits, None, K, "softmax", True, 1.0, 0, 0)
    plan = ops.permute_plan(ids, E, lo, hi, 1)
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device="cuda")
    cap, R_ = plan.tile_capacity, plan.row_capacity
    got_logits, got_w, got_ids = torch.empty(T, E, device="cuda"), torch.empty(T, K, device="cuda"), torch.empty(T, K, dtype=torch.int64, device="cuda")
    counts, offsets, seg_counts, ros, sor, tor = (i32(n) for n in (E, hi - lo + 1, 2 * (hi - lo), T * K, R_, R_))
    scale, te, tr, nt = torch.full((R_,), float("nan"), device="cuda"), i32(cap), i32(cap), i32(1)
    lib = _lib.load()
    work = torch.empty(max(1, lib.mi355_route_plan_workspace_bytes(T, K, E)), dtype=torch.uint8, device="cuda")
    _lib.check(lib.mi355_route_plan(
        partial.data_ptr(), splits, None, got_logits.data_ptr(), None, T, E, K, 1, 1, 1.0, 0, 0, got_w.data_ptr(), got_ids.data_ptr(), lo, hi, 1,
        ops.TILE_M, counts.data_ptr(), offsets.data_ptr(), seg_counts.data_ptr(), ros.data_ptr(), sor.data_ptr(), tor.data_ptr(), scale.data_ptr(), R_,
        te.data_ptr(), tr.data_ptr(), nt.data_ptr(), cap, work.data_ptr(), torch.cuda.current_stream().cuda_stream), "route_plan")
    n = int(nt)
    for name, a, b in (("logits", got_logits, logits), ("ids", got_ids, ids), ("weights", got_w, w), ("counts", counts, plan.counts_E),
                       ("offsets", offsets, plan.seg_offsets), ("row_of_slot", ros, plan.row_of_slot), ("slot_of_row", sor, plan.slot_of_row),
                       ("token_of_row", tor, plan.token_of_row), ("row_scale", scale, ops.combine_row_scale(w, plan)),
                       ("num_tiles", nt, plan.num_tiles), ("tile_expert", te[:n], plan.tile_expert[:n])):
        assert torch.equal(a, b), name


@pytest.mark.gpu
@pytest.mark.parametrize("D,E,lengths", [(1024, 64, (2, 999, 1024, 1500, 3072)), (128, 64, (33, 1023, 1025, 24576)), (2048, 64, (700, 1023, 1536))])
def test_a_chunk_has_its_logits_up_to_the_line_of_the_wide_kernel(D, E, lengths):
    """1024 tokens and more of few experts: the same slices as below."""
    assert max(lengths) * E * D <= 192 << 20
    test_a_chunk_of_the_tokens_has_their_logits(torch.bfloat16, D, E, lengths)
