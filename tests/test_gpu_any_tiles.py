"""Experts of any width whose tiles are dealt to the XCDs in runs, found from the segments' counts: every product, expert by expert, against fp64."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# one row; passes that end with a tile and one row past it, empty experts first, between and last; fewer tiles than XCDs; more experts than
# a wave has lanes, one past that, and more than two waves have; one expert with most of the rows
COUNTS = {
    "one": (1,),
    "ends": (0, 32, 33, 64, 0, 65, 128, 129, 256, 257, 0),
    "few": (3, 0, 5),
    "64": tuple((i * 7) % 41 for i in range(64)),
    "65": (0,) * 64 + (70,),
    "130": tuple(0 if i % 3 else 40 + i for i in range(130)),
    "most": (1400, 20, 31, 2, 50, 0, 17, 8, 64),
    # bf16 input and weight gradients on small tiles in one launch: large ones would cover a quarter more; a product just small enough and one past it
    "covers": (2100, 0, 1900, 2300, 1701),
    "small": (3000, 3100, 3050, 2900),
    "large": (4000, 3000, 3600, 3401),
}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("name,D,Fd", [("one", 64, 36), ("ends", 132, 200), ("few", 512, 260), ("64", 72, 100), ("65", 64, 64), ("130", 68, 132),
                                       ("most", 324, 232), ("covers", 400, 300), ("small", 480, 428), ("large", 480, 432)])
def test_every_tile_once(dtype, name, D, Fd):
    from torchllmtuner_amd import ops

    counts = COUNTS[name]
    print(f"any tiles {dtype} {name} D={D} F={Fd}", flush=True)
    g = torch.Generator().manual_seed(5)
    El, R = len(counts), sum(counts)
    x, dy = (torch.randn(R, D, generator=g).to(dtype).to(DEV) for _ in "xy")
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).to(dtype).to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    plan = ops.permute_plan(torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[:, None].to(DEV), El)
    y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan)
    dx, dw1, dw3, dw2 = ops.grouped_swiglu_bwd(dy, x, w1, w3, w2, gate, up, h, plan)
    # one rounding to bf16 of a result (at most half an ulp, 2^-9), or of fp32 a sum of n products, a walk of n roundings of half an ulp
    def bound(n):
        return 2.0 ** -9 if dtype == torch.bfloat16 else n ** 0.5 * 2.0 ** -24

    at = 0
    for e, c in enumerate(counts):
        r = slice(at, at + c)
        at += c
        if c == 0:
            assert not dw1[e].any() and not dw3[e].any() and not dw2[e].any()
            continue
        xd, dyd, gd, ud, hd = (t[r].double() for t in (x, dy, gate, up, h))
        a1, a3, a2 = w1[e].double(), w3[e].double(), w2[e].double()
        sig = torch.sigmoid(gd)
        dh = dyd @ a2
        dg, du = dh * ud * sig * (1 + gd * (1 - sig)), dh * F.silu(gd)
        # what the backward forms on the way is rounded too: dh, dh * up, silu, dgate, dup, and h of the forward silu and h
        chain = 4 * bound(D)
        for what, got, want, tol in (
                ("gate", gate[r], xd @ a1.T, bound(D)), ("up", up[r], xd @ a3.T, bound(D)), ("h", h[r], F.silu(gd) * ud, 2 * bound(D)),
                ("y", y[r], hd @ a2.T, bound(Fd)), ("dx", dx[r], dg @ a1 + du @ a3, chain + bound(2 * Fd)),
                ("dw1", dw1[e], dg.T @ xd, chain + bound(c)), ("dw3", dw3[e], du.T @ xd, chain + bound(c)), ("dw2", dw2[e], dyd.T @ hd, bound(c))):
            # (a 32-bit value's own rounding, where few products are added)
            assert rel_l2(got, want) < tol + 2.0 ** -23, f"{what} of expert {e}"
