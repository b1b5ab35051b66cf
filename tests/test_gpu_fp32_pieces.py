"""fp32 expert products on tiles of 64 rows and more, whose operands are multiplied as three bf16 pieces each, against fp64."""

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


def problem(ops, counts, D, Fd):
    g = torch.Generator().manual_seed(11)
    El, R = len(counts), sum(counts)
    ids = torch.repeat_interleave(torch.arange(El), torch.tensor(counts))[:, None]
    x, dy = (torch.randn(R, D, generator=g).to(DEV) for _ in "xy")
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).to(DEV) for s in ((El, Fd, D), (El, Fd, D), (El, D, Fd)))
    rows = list(torch.arange(R).split(list(counts)))  # the plan keeps an expert's rows in token order
    return ops.permute_plan(ids.to(DEV), El), x, dy, w1, w3, w2, [r.to(DEV) for r in rows]


def per_expert(rows, fn, like):
    out = torch.empty(like.shape, dtype=torch.float64, device=DEV)
    for e, r in enumerate(rows):
        out[r] = fn(e, r)
    return out


# every product on 64-row tiles; some of them on 32-row ones; all on 128-row ones.  Segments that end inside a tile, widths
# that end inside one and inside a step of 32
@pytest.mark.parametrize("counts,D,Fd", [((520, 1000, 65), 772, 580), ((300, 70, 0, 401), 516, 900),
                                         ((3100, 2900, 3001), 900, 908)])
def test_products_against_fp64(ops, counts, D, Fd):
    print(f"fp32 pieces {counts} D={D} F={Fd}", flush=True)
    plan, x, dy, w1, w3, w2, rows = problem(ops, counts, D, Fd)
    y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan)
    dx, dw1, dw3, dw2 = ops.grouped_swiglu_bwd(dy, x, w1, w3, w2, gate, up, h, plan)
    # a sum of n products, rounded to 24 bits as it grows: a walk of at most n roundings of half an ulp each
    def bound(n):
        return n ** 0.5 * 2.0 ** -24

    d = [t.double() for t in (x, dy, w1, w3, w2, gate, up, h)]
    xd, dyd, w1d, w3d, w2d, gd, ud, hd = d
    assert rel_l2(gate, per_expert(rows, lambda e, r: xd[r] @ w1d[e].T, gate)) < bound(D)
    assert rel_l2(up, per_expert(rows, lambda e, r: xd[r] @ w3d[e].T, up)) < bound(D)
    assert rel_l2(y, per_expert(rows, lambda e, r: hd[r] @ w2d[e].T, y)) < bound(Fd)
    # (the element-wise ends: a few roundings each, below the sums' own)
    sig = torch.sigmoid(gd)
    dh = per_expert(rows, lambda e, r: dyd[r] @ w2d[e], h)
    dg, du = dh * ud * sig * (1 + gd * (1 - sig)), dh * F.silu(gd)
    want = per_expert(rows, lambda e, r: dg[r] @ w1d[e] + du[r] @ w3d[e], dx)
    assert rel_l2(dx, want) < bound(D) + bound(2 * Fd)
    for got, a, b, chain in ((dw1, dg, xd, bound(D)), (dw3, du, xd, bound(D)), (dw2, dyd, hd, 0.0)):
        want = torch.stack([a[r].T @ b[r] for r in rows])
        assert rel_l2(got, want) < chain + bound(max(counts))


def test_infinities_overflow_and_nan(ops):
    """A value beyond bf16's range and one that is none: what an fp32 product of the row gives, and nothing elsewhere."""
    plan, x, _, w1, w3, w2, rows = problem(ops, (520, 1000, 65), 772, 580)
    clean = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan)[1]
    x[3, 700], x[600, 1], x[601, 5] = float("inf"), float("nan"), 3.4e38  # (rounds to infinity in bf16)
    w1[1, 9, 5] = 0.0
    w1[1, 8, 5] = 0.5
    gate = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan)[1]
    torch.cuda.synchronize()
    assert torch.equal(gate[3], torch.sign(w1[0, :, 700]) * float("inf"))
    assert gate[600].isnan().all()
    assert gate[601].isfinite().all() and gate[601, 8].item() == pytest.approx(1.7e38, rel=1e-6)
    same = torch.ones(len(x), dtype=torch.bool, device=DEV)
    same[[3, 600, 601]] = False
    cols = torch.tensor([c for c in range(580) if c not in (8, 9)], device=DEV)
    # rows that share a tile with one of the three are formed in the other way: the same up to rounding
    assert rel_l2(gate[same][:, cols], clean[same][:, cols]) < 2 * 772 ** 0.5 * 2.0 ** -24


def reference(x, dy, w1, w3, w2, gate, up, h, rows):
    """fp64 products of what each launch is given; what it rounds in between (dgate, dup) is not."""
    x, dy, w1, w3, w2, gate, up, h = (t.double() for t in (x, dy, w1, w3, w2, gate, up, h))
    sig = torch.sigmoid(gate)
    dh = per_expert(rows, lambda e, r: dy[r] @ w2[e], h)
    dg, du = dh * up * (sig * (1 + gate * (1 - sig))), dh * (gate * sig)
    dw = lambda a, b: torch.stack([a[r].T @ b[r] for r in rows])
    return dict(gate=per_expert(rows, lambda e, r: x[r] @ w1[e].T, gate), up=per_expert(rows, lambda e, r: x[r] @ w3[e].T, up),
                y=per_expert(rows, lambda e, r: h[r] @ w2[e].T, x), dx=per_expert(rows, lambda e, r: dg[r] @ w1[e] + du[r] @ w3[e], x),
                dw1=dw(dg, x), dw3=dw(du, x), dw2=dw(dy, h))


# 64-row and 128-row tiles
@pytest.mark.parametrize("counts,D,Fd", [((520, 1000, 65), 772, 580), ((3100, 2900, 3001), 900, 908)])
def test_values_whose_pieces_end_below_bf16(ops, counts, D, Fd):
    """From 2^-110 down to fp32's own end a third piece would lose bits; rows and experts of such values are as exact as others."""
    print(f"fp32 pieces, small values {counts}", flush=True)
    plan, x, dy, w1, w3, w2, rows = problem(ops, counts, D, Fd)
    small = 2.0 ** -118
    x[3] *= small        # gate, up
    x[600] *= 2.0 ** -58  # h is about 2^-118: down
    dy[700] *= small     # dh, then the input gradient
    dy[rows[2]] *= small  # the weight gradients of an expert
    y, gate, up, h = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan)
    dx, dw1, dw3, dw2 = ops.grouped_swiglu_bwd(dy, x, w1, w3, w2, gate, up, h, plan)
    want = reference(x, dy, w1, w3, w2, gate, up, h, rows)

    def bound(n):  # as above
        return n ** 0.5 * 2.0 ** -24

    def err(got, ref):  # scaled: the norms of such values are below what rel_l2 divides by
        return rel_l2(got.double() / small, ref / small)

    assert err(gate[3], want["gate"][3]) < bound(D) and err(up[3], want["up"][3]) < bound(D)
    assert 0 < float(h[600].abs().max()) < 2.0 ** -110
    assert err(y[600], want["y"][600]) < bound(Fd)
    few = torch.cat([torch.tensor([700], device=DEV), rows[2]])
    assert err(dx[few], want["dx"][few]) < bound(D) + bound(2 * Fd)
    assert err(dw2[2], want["dw2"][2]) < bound(max(counts))
    for got, name in ((dw1, "dw1"), (dw3, "dw3")):
        assert err(got[2], want[name][2]) < bound(D) + bound(max(counts))


def test_products_that_only_their_first_pieces_overflow(ops):
    """(2 - 2^-13) 2^63 rounds up to 2^64 in bf16, and the square of that is no fp32 value, while its own is."""
    plan, x, _, w1, w3, w2, _ = problem(ops, (520, 1000, 65), 772, 580)
    big = (2 - 2.0 ** -13) * 2.0 ** 63
    x[10] = 0
    x[10, 5] = w1[0, 7, 5] = big
    gate = ops.grouped_swiglu_fwd(x, w1, w3, w2, plan)[1]
    assert gate[10, 7].item() == pytest.approx(big * big, rel=1e-6) and gate[10].isfinite().all()


def same(a, b):
    return bool(((a == b) | (a.isnan() & b.isnan())).all())


def alike(got, ref, tol):
    """Infinities of one sign and NaN in the same places, the rest within tol."""
    ref = ref.to(got.device)
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    assert torch.equal(got[got.isinf()] > 0, ref[ref.isinf()] > 0)
    finite = ref.isfinite()
    assert rel_l2(got[finite], ref[finite]) < tol


# 64-row tiles throughout, 128-row ones throughout (the weight gradients' too)
@pytest.mark.parametrize("T,D,Fd,E", [(900, 772, 580, 3), (4500, 900, 908, 3)])
def test_not_finite_and_small_values_in_every_product_copied_and_read_in_place(ops, T, D, Fd, E):
    from torchllmtuner_amd import _lib

    print(f"fp32 pieces, not finite T={T}", flush=True)
    lib, g = _lib.load(), torch.Generator().manual_seed(T)
    ids = torch.stack([torch.randperm(E, generator=g)[:2] for _ in range(T)])
    plan = ops.permute_plan(ids.to(DEV), E)
    x, dout = (torch.randn(T, D, generator=g).to(DEV) for _ in "xd")
    w1, w3, w2 = ((torch.randn(*s, generator=g) * 0.03).to(DEV) for s in ((E, Fd, D), (E, Fd, D), (E, D, Fd)))
    weights = torch.rand(T, 2, generator=g).to(DEV)
    x[3, 700], x[200, 1], x[201] = float("inf"), float("nan"), x[201] * 2.0 ** -118
    dout[5, 71], dout[320, 8], dout[321] = float("-inf"), float("nan"), dout[321] * 2.0 ** -118
    tok, R = plan.token_of_row.long(), plan.row_capacity
    scale = ops.combine_row_scale(weights, plan)
    rows_x, dy = x[tok], dout[tok] * scale[:, None]
    rows = [r for r in torch.arange(R, device=DEV).split(plan.seg_counts.tolist())]
    copied = ops.grouped_swiglu_fwd(rows_x, w1, w3, w2, plan)
    y, gate, up, h = copied
    p = lambda t: t.data_ptr()
    stream = torch.cuda.current_stream().cuda_stream
    plan_args = [p(t) for t in plan.segments()] + [plan.tile_capacity]
    assert lib.mi355_grouped_gather_covers(0, D, Fd, R, T) == 1
    gathered = [torch.empty_like(t) for t in copied]
    rc = lib.mi355_grouped_gather_fwd(p(x), p(plan.token_of_row), T, p(w1), p(w3), p(w2), 0, *plan_args, p(gathered[1]),
                                      p(gathered[2]), p(gathered[3]), p(gathered[0]), E, D, Fd, R, stream)
    assert rc == 0
    for name, a, b in zip(("y", "gate", "up", "h"), gathered, copied):
        assert same(a, b), name
    want = reference(rows_x, dy, w1, w3, w2, gate, up, h, rows)

    def bound(n):
        return n ** 0.5 * 2.0 ** -24

    alike(gate, want["gate"], bound(D))
    alike(up, want["up"], bound(D))
    alike(y, want["y"], bound(Fd))
    # backward on a clean forward (every gradient of an expert with a NaN activation would be NaN), then on this one
    for fx, clean in ((torch.where(x.isfinite(), x, 1.0), True), (x, False)):
        rows_f = fx[tok]
        _, gate, up, h = ops.grouped_swiglu_fwd(rows_f, w1, w3, w2, plan)
        grads = ops.grouped_swiglu_bwd(dy, rows_f, w1, w3, w2, gate, up, h, plan)
        dgate, dup = torch.empty_like(gate), torch.empty_like(gate)
        got = [torch.empty_like(t) for t in grads]
        rc = lib.mi355_grouped_gather_bwd(p(dout), p(fx), p(plan.token_of_row), T, p(scale), p(w1), p(w3), p(w2), p(gate), p(up),
                                          p(h), 0, *plan_args, p(dgate), p(dup), *(p(t) for t in got), None, None, 0, E, D,
                                          Fd, R, stream)
        assert rc == 0
        for name, a, b in zip(("dx", "dw1", "dw3", "dw2"), got, grads):
            assert same(a, b), name
        if not clean:
            continue
        want = reference(rows_f, dy, w1, w3, w2, gate, up, h, rows)
        alike(grads[0], want["dx"], bound(D) + bound(2 * Fd))
        alike(grads[3], want["dw2"], bound(max(len(r) for r in rows)))
        for i, name in ((1, "dw1"), (2, "dw3")):
            alike(grads[i], want[name], bound(D) + bound(max(len(r) for r in rows)))
