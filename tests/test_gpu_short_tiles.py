"""Row products on tiles of up to 128 rows (weights past the memory-side cache, most experts of no more rows) against the 256-row tiles, bit for bit, a tile a workgroup and
several, and lists that leave tiles out, which stay with the 256-row tiles."""

from __future__ import annotations

import dataclasses

import pytest
import torch

from tests.test_gpu_forward_tiles import PASS, kernels, roomy
from tests.test_gpu_listed_tiles import FREE, run
from tests.test_gpu_narrow_tiles import row_errors

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

# the edges of a 16-row block, of the four wave rows, of a tile; none; and one expert of two tiles among them, which the rule has room for
FEW = (1, 15, 16, 17, 0, 63, 64, 65, 127, 128, 129, 112, 113, 5, 100, 2)
MANY = (130, 160, 200, 256, 129, 144, 145, 176, 177, 131, 140, 150, 170, 190, 201, 255)  # two tiles each: 256-row ones for all



def short(plan, D, Fd, tokens):
    """Work items on short tiles of gate/up, down and dRows, 0 for each that walks its list's tiles."""
    import ctypes

    from torchllmtuner_amd import _lib

    El = plan.num_local_experts
    counts = (ctypes.c_int32 * El)(*plan.seg_counts[:El].tolist())
    return [_lib.load().mi355_grouped_short_tiles(stage, El, D, Fd, plan.row_capacity, tokens, plan.tile_capacity, counts,
                                                  int(plan.num_tiles)) for stage in (1, 2, 8)]


def listing(plan, keep):
    """The plan with the tiles of the experts in `keep` alone."""
    some = [(e, r) for e, r in zip(plan.tile_expert.tolist()[:int(plan.num_tiles)], plan.tile_row0.tolist()) if e in keep]
    pad = lambda v: torch.tensor(list(v) + [0] * (plan.tile_capacity - len(some)), dtype=torch.int32, device=DEV)
    return dataclasses.replace(plan, tile_expert=pad(e for e, _ in some), tile_row0=pad(r for _, r in some),
                               num_tiles=torch.tensor([len(some)], dtype=torch.int32, device=DEV))


# 21, 14 and 32 K steps, last tiles that start early; rows of 4 KiB: gate/up and down turned, and dRows on 256-row tiles
@pytest.mark.parametrize("D,Fd,align,turned", [(1344, 1344, 1, 0), (2048, 896, 16, 0x800), (1344, 2048, 1, 0x1000)])
def test_short_tiles(D, Fd, align, turned):
    from torchllmtuner_amd import _lib, ops

    print(f"short tiles D={D} F={Fd}", flush=True)
    g = torch.Generator().manual_seed(D)
    El = len(FEW) + len(MANY)
    assert El * D * Fd * 6 > 320 << 20
    n, total = sum(FEW), sum(FEW) + sum(MANY)
    x, dy = (torch.randn(total, D, generator=g).bfloat16().to(DEV) for _ in "xd")
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(FEW + MANY))
    ids = torch.cat([ids[:n][torch.randperm(n, generator=g)], ids[n:]]).to(DEV)
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).bfloat16().to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    room = 200
    gate, up = (torch.randn(room * El, Fd, generator=g).bfloat16().to(DEV) for _ in "gu")

    def products(ids, keep=None):
        T = ids.numel()
        plan = roomy(ops.permute_plan(ids[:, None], El, align=align), room)
        assert kernels(plan, D, Fd, True) == 256 + turned
        rows = torch.zeros(plan.row_capacity, D, dtype=dy.dtype, device=DEV)
        rows[plan.row_of_slot.flatten().long()] = dy[:T]
        plan = plan if keep is None else listing(plan, keep)
        assert [bool(v) for v in short(plan, D, Fd, T)] == ([T == n, T == n, T == n and D % 2048 != 0] if keep is None else [False] * 3)
        out = run((ops, _lib), plan, x[:T], plan.token_of_row, T, w1, w3, w2, rows, gate, up, plan.row_capacity)
        return out, plan.row_of_slot.flatten().long()[:n], plan

    few, row, plan = products(ids[:n])
    many, _, _ = products(ids)
    for name, t in many.items():
        assert torch.equal(t[row], few[name][row]), name
    # one bf16 rounding of an fp32 sum
    own = ids[:n].cpu()
    for e, count in enumerate(FEW):
        r, t = row[own == e], (own == e).nonzero()[:, 0]
        if count:
            assert row_errors(few["gate"][r], x[t].float() @ w1[e].float().T) < 2.0 ** -8
            assert row_errors(few["y"][r], few["h"][r].float() @ w2[e].float().T) < 2.0 ** -8
            assert row_errors(few["drows"][r], few["dgate"][r].float() @ w1[e].float() + few["dup"][r].float() @ w3[e].float()) < 2.0 ** -8
    # every other expert left out
    some, row, plan = products(ids[:n], keep=range(0, El, 2))
    listed = (ids[:n] % 2 == 0)
    for name, t in some.items():
        assert torch.equal(t[row[listed]], few[name][row[listed]]), name
        assert bool((t[row[~listed]] == FREE).all()), name


# Several tiles a workgroup, of every height, those of the next arriving while the results of the last leave; three and six tiles of an expert among
# them.  21, 11 and 32 K steps; last tiles that start early and output of whole tiles; gate/up and down turned, dRows on 256-row tiles at rows of 4 KiB, gate/up
# where short tiles would be a round of workgroups more.
@pytest.mark.parametrize("D,Fd,align,products", [(1344, 704, 1, (1, 1, 1)), (2048, 768, 1, (1, 1, 0)), (2048, 704, 16, (1, 1, 0)), (1344, 2048, 1, (0, 1, 1))])
def test_several_short_tiles_a_workgroup(D, Fd, align, products):
    from torchllmtuner_amd import _lib, ops

    print(f"several short tiles D={D} F={Fd} align={align}", flush=True)
    g = torch.Generator().manual_seed(D + Fd)
    counts = list(FEW * 9)
    counts[0], counts[16] = 300, 700
    counts = [counts[i] for i in torch.randperm(len(counts), generator=g)]
    El, R = len(counts), sum(counts)
    dev = torch.Generator(device=DEV).manual_seed(D)
    normal = lambda *s, std=1.0: (torch.randn(*s, generator=dev, device=DEV, dtype=torch.float32) * std).bfloat16()
    x = normal(R, D)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=g)]
    w1, w3, w2 = normal(El, Fd, D, std=0.03), normal(El, Fd, D, std=0.03), normal(El, D, Fd, std=0.03)
    plan = ops.permute_plan(ids[:, None].to(DEV), El, align=align)
    cap = plan.row_capacity
    gate, up, dy = normal(cap, Fd), normal(cap, Fd), normal(cap, D)
    halves = [listing(plan, set(range(first, El, 2))) for first in (0, 1)]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    assert kernels(plan, D, Fd, True) & PASS == 256
    assert [(v > 0) + (v > 2 * cus) for v in short(plan, D, Fd, R)] == [2 * p for p in products]
    assert [short(q, D, Fd, R) for q in halves] == [[0, 0, 0]] * 2
    whole, even, odd = (run((ops, _lib), q, x, plan.token_of_row, R, w1, w3, w2, dy, gate, up, cap) for q in (plan, *halves))
    expert = torch.searchsorted(plan.seg_offsets[:El].contiguous(), torch.arange(cap, device=DEV, dtype=torch.int32), right=True) - 1
    is_even = (expert % 2 == 0)[:, None]
    row = plan.row_of_slot.flatten().long()
    for name, t in whole.items():
        assert torch.equal(t, torch.where(is_even, even[name], odd[name])), name
        assert not bool((even[name] != FREE).any(1)[~is_even[:, 0]].any()) and not bool((odd[name] != FREE).any(1)[is_even[:, 0]].any()), name
    # one bf16 rounding of an fp32 sum
    own = ids.to(DEV)
    for e in range(El):
        r, t = row[own == e], (own == e).nonzero()[:, 0]
        if len(t):
            assert row_errors(whole["gate"][r], x[t].float() @ w1[e].float().T) < 2.0 ** -8
            assert row_errors(whole["y"][r], whole["h"][r].float() @ w2[e].float().T) < 2.0 ** -8
            assert row_errors(whole["drows"][r], whole["dgate"][r].float() @ w1[e].float() + whole["dup"][r].float() @ w3[e].float()) < 2.0 ** -8
