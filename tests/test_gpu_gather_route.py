"""The selection's backward and the experts' as one call against the two calls it stands for, bit for bit."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF, F32 = torch.bfloat16, torch.float32
FREE = 7.0  # what results hold before


# dH on tiles of 32, 64 and 128 rows (fp32) and of 64 and 128 (bf16), the selection beside it; then the selection in front: the products behind dH are launches of
# their own (fp32: 128 x 128 weight gradients from 400 rows an expert on; bf16: more than 2.4 Gi of rows D F, widths that large tiles cover without waste), no input
# gradient (drows), no weight gradients.  Tokens that are no multiple of four; one expert to 64, of which a share of them here; the gate's slices up to 32
@pytest.mark.parametrize("dtype,T,E,local,K,D,F,aux,want", [
    (F32, 7, 3, 3, 2, 64, 36, True, "x w gate"), (F32, 1001, 33, 33, 4, 128, 132, True, "x w"), (F32, 5001, 64, 64, 4, 256, 520, False, "x w"),
    (F32, 513, 8, 8, 2, 256, 512, False, "x w gate"), (F32, 33, 1, 1, 1, 20, 12, True, "x w gate"), (F32, 402, 32, 11, 3, 68, 100, True, "x w gate"),
    (BF, 1531, 16, 16, 4, 320, 232, True, "x w gate"), (BF, 3002, 64, 64, 2, 72, 100, True, "x w"), (BF, 4095, 32, 32, 4, 324, 436, False, "x w gate"),
    (BF, 255, 64, 20, 5, 40, 44, True, "x w"),
    (F32, 3301, 32, 32, 4, 260, 260, True, "x w gate"), (BF, 4202, 32, 32, 4, 472, 364, True, "x w gate"), (BF, 4202, 40, 40, 4, 472, 364, True, "x w"),
    (F32, 333, 5, 5, 2, 64, 64, True, "w gate"), (BF, 333, 5, 5, 2, 72, 68, True, "x gate"), (BF, 333, 5, 5, 2, 72, 68, True, "w")])
def test_one_call_gives_the_two_calls_bits(dtype, T, E, local, K, D, F, aux, want):
    from torchllmtuner_amd import _lib, ops

    print(f"gather route {dtype} T={T} E={E} local={local} K={K} D={D} F={F} {want}", flush=True)
    lib, want, dt = _lib.load(), want.split(), 0 if dtype == F32 else 1
    g = torch.Generator(device=DEV).manual_seed(T + E)
    normal = lambda *s, dtype=dtype: torch.randn(*s, generator=g, device=DEV).to(dtype)
    logits = normal(T, E, dtype=F32)
    ids = logits.topk(K, dim=1).indices
    plan = ops.permute_plan(ids, E, 0, local)
    R = plan.row_capacity
    x, dout, y = normal(T, D), normal(T, D), normal(R, D)
    gate, up, h = normal(R, F), normal(R, F), normal(R, F)
    w1, w3, w2 = normal(local, F, D), normal(local, F, D), normal(local, D, F)
    scale = torch.rand(R, generator=g, device=DEV)
    aux_f = torch.rand(E, generator=g, device=DEV) if aux else None
    aux_scale = torch.rand(1, generator=g, device=DEV) if aux else None
    padding = (torch.rand(T, generator=g, device=DEV) < 0.3).to(torch.uint8) if aux else None
    p = lambda t: None if t is None else t.data_ptr()
    seg = (p(plan.seg_offsets), p(plan.seg_counts), p(plan.tile_expert), p(plan.tile_row0), p(plan.num_tiles), plan.tile_capacity)
    stream = torch.cuda.current_stream().cuda_stream
    select = (ops.SCORE_FUNCS["sigmoid"], 1, 2.5)  # score function (sigmoid), normalised, scale

    def outputs():
        new = lambda *s, dtype=dtype: torch.full(s, FREE, dtype=dtype, device=DEV)
        out = dict(dgate=new(R, F), dup=new(R, F), drows=new(R, D) if "x" in want else None)
        for name, shape in (("dw1", (local, F, D)), ("dw3", (local, F, D)), ("dw2", (local, D, F))):
            out[name] = new(*shape) if "w" in want else None
        out["dlogits"] = new(T, E, dtype=F32)
        floats = lib.mi355_router_gate_bwd_workspace_bytes(T, D, E) // 4
        out["partial"] = new(floats, dtype=F32) if "gate" in want else None
        return out

    def experts(f, o, *route):
        return f(p(dout), p(x), p(plan.token_of_row), T, p(scale), p(w1), p(w3), p(w2), p(gate), p(up), p(h), dt, *seg, p(o["dgate"]), p(o["dup"]),
                 p(o["drows"]), p(o["dw1"]), p(o["dw3"]), p(o["dw2"]), *route, local, D, F, R, stream)

    two, one = outputs(), outputs()
    _lib.check(lib.mi355_router_select_rows_bwd(p(logits), p(ids), p(dout), p(y), dt, p(plan.row_of_slot), R, D, p(aux_f), p(aux_scale), p(padding),
                                                p(two["dlogits"]), T, E, K, *select, stream), "select_rows_bwd")
    joined = "gate" in want
    _lib.check(experts(lib.mi355_grouped_gather_bwd, two, p(two["dlogits"]) if joined else None, p(two["partial"]), E), "gather_bwd")
    _lib.check(experts(lib.mi355_grouped_gather_route_bwd, one, p(logits), p(ids), p(y), p(plan.row_of_slot), p(aux_f), p(aux_scale), p(padding),
                       p(one["dlogits"]), p(one["partial"]), E, K, *select), "gather_route_bwd")
    for name, a in two.items():
        if a is None:
            continue
        n = int(plan.total_rows) if a.shape[0] == R and a.dim() == 2 and name != "dlogits" else a.shape[0]
        assert torch.equal(a[:n], one[name][:n]), name
        assert not bool((a[:n] == FREE).all()), name
    # what they are: the selection's gradient against autograd in 64 bits (fp32 dot products of D terms, then sums over E)
    z = logits.double().requires_grad_()
    score = torch.sigmoid(z)
    chosen = score.gather(1, ids)
    rows = plan.row_of_slot.long().view(T, K)
    dw = torch.where(rows >= 0, (dout.double()[:, None] * y.double()[rows.clamp(min=0)]).sum(-1), 0.0)
    loss = (2.5 * chosen / (chosen.sum(1, keepdim=True) + 1e-20) * dw).sum()
    if aux:
        part = (score / score.sum(1, keepdim=True) * aux_f.double()).sum(1)
        loss = loss + aux_scale.double().squeeze() * part[padding == 0].sum()
    want_dlogits, = torch.autograd.grad(loss, z)
    error = (one["dlogits"].double() - want_dlogits).norm() / want_dlogits.norm().clamp(min=1e-30)
    assert K == 1 or float(error) < 1e-5
