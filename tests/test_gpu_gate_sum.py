"""The router gate's backward with the sum over a token's rows in front, in one launch, against the row sum and the gate's
backward as calls of their own: the same bits, at the edges of the 128-token and 128-column tiles."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T,D,E,K", [(1, 128, 64, 1), (127, 192, 64, 3), (128, 384, 128, 8), (129, 448, 192, 9), (700, 1024, 256, 16),
                                     (1, 64, 4, 1), (9, 260, 16, 4), (700, 448, 32, 9)])  # the last three: up to 32 experts, tiles of 8 tokens
@pytest.mark.parametrize("extra", [(), ("addend",), ("addend", "no dw")])
def test_gate_backward_with_the_row_sum(T, D, E, K, extra):
    from torchllmtuner_amd import _lib

    print(f"gate sum T={T} D={D} E={E} K={K} {extra}", flush=True)
    lib, g = _lib.load(), torch.Generator().manual_seed(T)
    R = T * K + 5
    x, drows, add = (torch.randn(n, D, generator=g).bfloat16().to(DEV) for n in (T, R, T))
    dl, w = torch.randn(T, E, generator=g).to(DEV) * 0.01, torch.randn(E, D, generator=g).to(DEV) * 0.02
    rows = torch.randperm(R, generator=g)[: T * K].int()
    rows[torch.rand(T * K, generator=g) < 0.2] = -1  # slots without a row
    rows = rows.to(DEV)
    addend = add.data_ptr() if "addend" in extra else None
    work = torch.empty(lib.mi355_router_gate_bwd_workspace_bytes(T, D, E), dtype=torch.uint8, device=DEV)
    s = torch.cuda.current_stream().cuda_stream

    def run(joined):
        dx, mid, dw = torch.empty_like(x), torch.empty_like(x), torch.zeros_like(w)
        dwp = None if "no dw" in extra else dw.data_ptr()
        if joined:
            assert lib.mi355_router_gate_sum_bwd_covers(1, 0, D, E, K) == 1
            rc = lib.mi355_router_gate_sum_bwd(dl.data_ptr(), x.data_ptr(), 1, w.data_ptr(), None, drows.data_ptr(),
                                               rows.data_ptr(), R, K, addend, dx.data_ptr(), dwp, work.data_ptr(), T, D, E, s)
        else:
            rc = lib.mi355_permute_rows_add_bwd(drows.data_ptr(), 1, rows.data_ptr(), addend, mid.data_ptr(), T, D, K, s)
            assert rc == 0
            rc = lib.mi355_router_gate_add_bwd(dl.data_ptr(), x.data_ptr(), 1, w.data_ptr(), 0, None, mid.data_ptr(),
                                               dx.data_ptr(), dwp, work.data_ptr(), T, D, E, s)
        assert rc == 0
        torch.cuda.synchronize()
        return dx, dw

    for a, b in zip(run(True), run(False)):
        assert torch.equal(a, b)
    assert lib.mi355_router_gate_sum_bwd_covers(1, 0, D, E, 17) == 0 and lib.mi355_router_gate_sum_bwd_covers(1, 0, D, 60, K) == 0
    assert lib.mi355_router_gate_sum_bwd_covers(0, 0, D, E, K) == 0


# more than 32 experts of no matrix tile: the fewest and the most, one part of 32 tokens and 256 columns and a little more, rows that are not whole
# 16-byte pieces apart, on either side of 6 Mi elements, where strided products go on; 64 experts in fp32
@pytest.mark.parametrize("T,D,E,dtype", [(1, 4, 36, "bf16"), (33, 260, 60, "bf16"), (300, 512, 60, "fp32"), (257, 516, 44, "bf16"), (6144, 1024, 60, "bf16"),
                                         (6145, 1024, 60, "bf16"), (700, 448, 64, "fp32"), (64, 256, 62, "bf16")])
@pytest.mark.parametrize("addend", [False, True])
def test_gate_backward_between_the_tiles(T, D, E, dtype, addend):
    from torchllmtuner_amd import _lib

    print(f"gate backward T={T} D={D} E={E} {dtype} addend={addend}", flush=True)
    lib, g = _lib.load(), torch.Generator(device=DEV).manual_seed(T + E)
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    x, add = (torch.randn(T, D, generator=g, device=DEV).to(dt) for _ in "xa")
    dl, w = torch.randn(T, E, generator=g, device=DEV) * 0.01, torch.randn(E, D, generator=g, device=DEV) * 0.02
    dl[T // 2, E - 1] = float("inf")  # reaches one row of dx and one of dW, and nothing else
    work = torch.empty(max(16, lib.mi355_router_gate_bwd_workspace_bytes(T, D, E)), dtype=torch.uint8, device=DEV)
    dx, dw = torch.empty_like(x), torch.empty_like(w)
    assert lib.mi355_router_gate_add_bwd(dl.data_ptr(), x.data_ptr(), int(dtype == "bf16"), w.data_ptr(), 0, None,
                                         add.data_ptr() if addend else None, dx.data_ptr(), dw.data_ptr(), work.data_ptr(), T, D, E,
                                         torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    want_x, want_w = dl.double() @ w.double(), dl.double().T @ x.double()
    # fp32 products and sums (n + 1 roundings of at most 2^-24 of the terms' sizes), then, of bf16 tokens, one rounding, and another behind the addend
    size_x, size_w = (dl.abs().double() @ w.abs().double()), dl.abs().double().T @ x.abs().double()
    unit = 2.0 ** -8 if dtype == "bf16" else 2.0 ** -24
    bound = (E + 1) * 2.0 ** -24 * size_x + unit * want_x.abs() * (1 + unit)
    if addend:
        want_x = want_x + add.double()
        bound = bound * (1 + unit) + unit * want_x.abs()
    for got, want, limit in ((dx, want_x, bound), (dw, want_w, (T + 1) * 2.0 ** -24 * size_w)):
        finite = want.isfinite()
        assert torch.equal(got.isfinite(), finite)
        assert bool(((got.double() - want).abs() <= limit)[finite].all())


@pytest.mark.parametrize("T,D,E", [(1, 128, 64), (33, 1024, 64), (700, 1088, 64), (1024, 512, 128), (2048, 1024, 64), (300, 192, 192), (513, 2048, 64)])
def test_pieces_that_a_forward_keeps_are_the_backwards_own(T, D, E):
    """mi355_router_gate_fwd_keeping leaves the weight pieces that the backward would form itself: the same gradients, bit for bit, and the same logits."""
    from torchllmtuner_amd import _lib

    print(f"kept pieces T={T} D={D} E={E}", flush=True)
    lib, bf16, f32 = _lib.load(), 1, 0
    g = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(T, D, generator=g, device="cuda").bfloat16()
    w, dlogits = torch.randn(E, D, generator=g, device="cuda") * 0.02, torch.randn(T, E, generator=g, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    splits, kept = lib.mi355_router_gate_fwd_splits(bf16, f32, T, D, E), lib.mi355_router_gate_fwd_kept_bytes(bf16, f32, T, D, E)
    assert kept == 4 * E * D and lib.mi355_router_gate_fwd_pieces_bytes(bf16, f32, T, D, E) == 0
    pieces = torch.full((kept + 64,), 0xAB, dtype=torch.uint8, device="cuda")
    logits = [torch.empty(splits, T, E, device="cuda") for _ in range(2)]
    _lib.check(lib.mi355_router_gate_fwd_partial(x.data_ptr(), bf16, w.data_ptr(), None, logits[0].data_ptr(), None, T, D, E, stream), "partial")
    _lib.check(lib.mi355_router_gate_fwd_keeping(x.data_ptr(), bf16, w.data_ptr(), None, logits[1].data_ptr(), pieces.data_ptr(), T, D, E, stream), "keeping")
    assert torch.equal(*logits) and bool((pieces[kept:] == 0xAB).all())
    hi = w.bfloat16()
    want = torch.stack([hi, (w - hi.float()).bfloat16()])
    assert torch.equal(pieces[:kept].view(torch.bfloat16).view(2, E, D), want)
    work = torch.empty(lib.mi355_router_gate_bwd_workspace_bytes(T, D, E), dtype=torch.uint8, device="cuda")
    got = []
    for p in (None, pieces.data_ptr()):
        dx, dw = torch.empty_like(x), torch.empty_like(w)
        _lib.check(lib.mi355_router_gate_add_bwd(dlogits.data_ptr(), x.data_ptr(), bf16, w.data_ptr(), f32, p, None, dx.data_ptr(), dw.data_ptr(),
                                                 work.data_ptr(), T, D, E, stream), "bwd")
        got.append((dx, dw))
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
