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
