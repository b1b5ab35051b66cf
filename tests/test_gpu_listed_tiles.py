"""A tile list that leaves tiles out: the listed rows are computed, with the bits of the whole list, and the others' results are not touched."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32
FREE = 3.0  # what results hold before

# the edges of passes of 32 to 128 rows, of a tile and of two and three tiles of even heights, no rows, and enough experts for a second look at the counts
COUNTS = (1, 31, 33, 64, 65, 0, 128, 129, 256, 257, 300, 513, 5)


@pytest.fixture(scope="module")
def api():
    from torchllmtuner_amd import _lib, ops

    return ops, _lib


def run(api, q, x, tok, T, w1, w3, w2, dy, gate, up, expected):
    """Every product that walks the list, by name, from the same operands."""
    ops, _lib = api
    lib = _lib.load()
    El, F, D = w1.shape
    R, dt = q.row_capacity, 0 if x.dtype == F32 else 1
    p = lambda t: None if t is None else t.data_ptr()
    plan = (p(q.seg_offsets), p(q.seg_counts), p(q.tile_expert), p(q.tile_row0), p(q.num_tiles), q.tile_capacity)
    s = torch.cuda.current_stream().cuda_stream
    new = lambda n: torch.full((R, n), FREE, dtype=x.dtype, device=DEV)
    out = dict(gate=new(F), up=new(F), h=new(F), y=new(D), dgate=new(F), dup=new(F), drows=new(D), linear=new(F), dlin=new(D))
    o = {k: p(t) for k, t in out.items()}
    rows = x if tok is None else x[tok.long().clamp(0)].contiguous()
    _lib.check(lib.mi355_grouped_swiglu_fwd_expecting(p(x), p(tok), T, p(w1), p(w3), p(w2), dt, *plan, o["gate"], o["up"], o["h"], o["y"], El, D, F, R,
                                                      expected, s), "forward")
    # (the backward from whole activations; the weight gradients are over segments, whatever is listed)
    h = (torch.nn.functional.silu(gate.float()) * up.float()).to(x.dtype)
    _lib.check(lib.mi355_grouped_swiglu_bwd(p(dy), p(rows), None, R, p(w1), p(w3), p(w2), p(gate), p(up), p(h), dt, *plan, o["dgate"], o["dup"],
                                            o["drows"], None, None, None, El, D, F, R, s), "backward")
    _lib.check(lib.mi355_grouped_linear_fwd(p(rows), p(w1), dt, *plan, o["linear"], El, D, F, R, s), "linear")
    _lib.check(lib.mi355_grouped_linear_bwd(p(gate), p(rows), p(w1), dt, *plan, o["dlin"], None, El, D, F, R, s), "linear backward")
    torch.cuda.synchronize()
    return out


# any width (32-, 64- and 128-row tiles); passes of 16, 64 and 128 rows; row tiles.  rows: what the forward is told of, an expert (0: what there is)
@pytest.mark.parametrize("dtype,D,F,times,rows,passes", [
    (F32, 64, 36, 1, 0, 0), (F32, 320, 132, 2, 0, 0), (F32, 516, 520, 6, 0, 0), (BF, 72, 100, 1, 0, 0), (BF, 360, 328, 6, 0, 0),
    (BF, 384, 384, 1, 4, 16), (BF, 384, 448, 2, 20, 64), (BF, 448, 4032, 1, 60, 128), (BF, 512, 384, 6, 0, 256)])
def test_rows_of_listed_tiles_alone(api, dtype, D, F, times, rows, passes):
    import dataclasses

    ops, _lib = api
    print(f"listed tiles {dtype} D={D} F={F} times={times} rows={rows}", flush=True)
    g = torch.Generator().manual_seed(D + F)
    counts = COUNTS * times
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[torch.randperm(R, generator=g)].to(DEV)
    normal = lambda *s, scale=1.0: (torch.randn(*s, generator=g) * scale).to(dtype).to(DEV)
    x, dy, gate, up = normal(R, D), normal(R, D), normal(R, F), normal(R, F)
    w1, w3, w2 = normal(El, F, D, scale=0.05), normal(El, F, D, scale=0.05), normal(El, D, F, scale=0.05)
    plan = ops.permute_plan(ids[:, None], El)
    gathered = passes > 0
    tok = plan.token_of_row if gathered else None
    expected = rows * El if rows else R
    if passes:
        assert _lib.load().mi355_grouped_fwd_kernels(1, El, D, F, R, expected, R, plan.tile_capacity) & 0x1FF == passes
    n = int(plan.num_tiles)
    expert, row0 = plan.tile_expert[:n].tolist(), plan.tile_row0[:n].tolist()
    first, count = plan.seg_offsets.tolist(), plan.seg_counts[:El].tolist()

    def covered(tiles):
        mask = torch.zeros(R, dtype=torch.bool)
        for i in tiles:
            e = expert[i]
            pieces = -(-count[e] // 256)
            height = 256 if pieces == 1 else (-(-count[e] // pieces) + 15) // 16 * 16
            mask[row0[i]:min(row0[i] + height, first[e] + count[e])] = True
        return mask.to(DEV)

    assert bool(covered(range(n)).all())
    args = (x, tok, R, w1, w3, w2, dy, gate, up, expected)
    whole = run(api, plan, *args)
    # of the matrix-core kernels whole experts, whose tiles follow each other
    groups = [[i for i in range(n) if expert[i] == e] for e in dict.fromkeys(expert)] if passes else [[i] for i in range(n)]
    for some in ([], groups[::2], groups[1::2], groups[-1:], groups[::-1]):
        keep = [i for group in some for i in group]
        pad = lambda v: torch.tensor(v + [0] * (plan.tile_capacity - len(v)), dtype=torch.int32, device=DEV)
        q = dataclasses.replace(plan, tile_expert=pad([expert[i] for i in keep]), tile_row0=pad([row0[i] for i in keep]),
                                num_tiles=torch.tensor([len(keep)], dtype=torch.int32, device=DEV))
        check(run(api, q, *args), whole, covered(keep))
    if not passes:
        short = dataclasses.replace(plan, tile_capacity=n // 2)  # the list's first half, by the room that the caller states
        check(run(api, short, *args), whole, covered(range(n // 2)))


def check(got, whole, rows):
    for name, t in got.items():
        assert torch.equal(t[rows], whole[name][rows]), name
        assert bool((t[~rows] == FREE).all()), name
