"""The block as one operator (csrc/torch_block.cpp) and the kernels only it uses, at the edges of their
tiles: against the stage operators (a forward hook on the router makes the block visible in stages),
bit for bit, and the gate projection against fp64."""

import pytest
import torch

from oracle import moe_ref as R
from tests.helpers import build_block, make_params

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype,T,D,E,K,F,kw", [
    (torch.bfloat16, 1, 384, 128, 8, 384, {}),
    (torch.bfloat16, 63, 384, 256, 16, 448, dict(groups=(8, 4))),
    (torch.bfloat16, 64, 512, 60, 6, 384, dict(dispatcher="padded", pad_multiple=16)),
    (torch.bfloat16, 65, 512, 64, 5, 384, dict(bias=True)),
    (torch.bfloat16, 1023, 448, 128, 2, 384, dict(dispatcher="share", local=(32, 80))),
    (torch.bfloat16, 1025, 512, 128, 8, 384, dict(shared=448)),
    (torch.bfloat16, 16449, 384, 64, 2, 384, {}),  # two chunks of tokens per workgroup
    (torch.bfloat16, 200, 72, 17, 3, 100, dict(shared=60)),
    (torch.float32, 65, 100, 5, 2, 92, dict(dispatcher="padded", pad_multiple=8, shared=64)),
    (torch.float32, 1, 36, 1, 1, 40, {}),
    (torch.float32, 129, 33, 12, 4, 31, dict(gate_bias=True)),
])
def test_one_operator_equals_the_stages_bit_for_bit(dtype, T, D, E, K, F, kw):
    print(f"one operator {dtype} T={T} D={D} E={E} K={K} F={F} {kw}", flush=True)
    kw = dict(kw)
    groups, shared, bias, gate_bias = kw.pop("groups", None), kw.pop("shared", None), kw.pop("bias", False), kw.pop("gate_bias", False)
    spec = R.RouterSpec(E, K, score_func="sigmoid" if bias or groups else "softmax", route_norm=True,
                        num_expert_groups=groups and groups[0], num_limited_groups=groups and groups[1])
    El = kw["local"][1] - kw["local"][0] if "local" in kw else None
    p = make_params(E, D, F, dtype, seed=T, std=0.05, shared_F=shared, El=El)
    if bias:
        p.expert_bias_E = torch.linspace(-0.1, 0.1, E)
    g = torch.Generator().manual_seed(T + 1)
    x = torch.randn(T, D, generator=g).to(dtype).to(DEV)
    gout = torch.randn(T, D, generator=g).to(dtype).to(DEV)

    def run(in_stages):
        block = build_block(p, spec, D, F, dtype, DEV, load_balance_coeff=1e-3 if bias else None, **kw)
        if gate_bias:
            block.router.gate.bias = torch.nn.Parameter(torch.linspace(-1, 1, E, device=DEV))
        block.train()
        block.overlap_shared_experts = not in_stages  # (one stream: the stages' order of the three input gradients)
        if in_stages:
            block.router.register_forward_hook(lambda *a: None)
        whole = block._forward_as_one(x)
        assert (whole is None) == in_stages
        xin = x.clone().requires_grad_()
        out = block(xin)
        out.backward(gout)
        with torch.no_grad():
            plain = block.eval()(x)
        return [out.detach(), plain, xin.grad, block.tokens_per_expert_E] + [q.grad for q in block.parameters()]

    for i, (a, b) in enumerate(zip(run(True), run(False))):
        assert torch.equal(a, b), f"tensor {i} differs by {float((a.float() - b.float()).abs().max())}"


@pytest.mark.parametrize("quantile,masked,T,E,K,groups", [
    (True, True, 64, 64, 6, None), (True, False, 65, 24, 3, None), (False, True, 1000, 128, 8, (8, 4)), (False, True, 16500, 256, 2, None),
    (False, False, 3, 5, 2, None)])
def test_router_statistics_of_the_one_operator_match_the_stages(quantile, masked, T, E, K, groups):
    """Histogram, counts without padding, the balance loss's metric and gradient: one operator against the
    stages.  Counts and histogram are equal; the loss is the same sums in another order."""
    from torchllmtuner_amd import moe

    print(f"one operator statistics quantile={quantile} masked={masked} T={T} E={E} K={K}", flush=True)
    D, F = 384, 384
    p = make_params(E, D, F, torch.bfloat16, seed=T, std=0.05)
    g = torch.Generator().manual_seed(T + 1)
    x = torch.randn(T, D, generator=g).bfloat16().to(DEV)
    gout = torch.randn(T, D, generator=g).bfloat16().to(DEV)
    mask = (torch.rand(T, generator=g) < 0.2).to(DEV) if masked else None
    denom = torch.tensor(float(T * K), device=DEV)

    def run(in_stages):
        aux = moe.MicrobatchWiseLoadBalanceLoss(coeff=2.0)
        if quantile:
            router = moe.QuantileBalancedTopKRouter(E, D, K, num_bins=500, route_norm=True, aux_loss=aux)
        else:
            router = moe.TokenChoiceTopKRouter(E, D, K, score_func="softmax", aux_loss=aux,
                                               num_expert_groups=groups and groups[0], num_limited_groups=groups and groups[1])
        block = moe.MoE(E, moe.RoutedExperts(moe.GroupedExperts(D, F, E), moe.LocalTokenDispatcher(E, K)), router,
                        load_balance_coeff=None).to(torch.bfloat16)
        router.gate.float()
        aux.to(torch.bfloat16 if masked else torch.float32)
        with torch.no_grad():
            router.gate.weight.copy_(p.router_w_ED)
            ie = block.routed_experts.inner_experts
            ie.w1_EFD.copy_(p.w1_EFD); ie.w3_EFD.copy_(p.w3_EFD); ie.w2_EDF.copy_(p.w2_EDF)
            if quantile:
                block.expert_bias_E.copy_(torch.linspace(-0.05, 0.05, E))
        block = block.to(DEV).train()
        moe.AuxLoss.set_step_denominator(denom, model_parts=[block])
        if in_stages:
            router.register_forward_hook(lambda *a: None)
        assert (block._forward_as_one(x, mask) is None) == in_stages
        if not in_stages:  # (the call above kept statistics)
            aux.instance_acc.zero_()
            if quantile:
                router.quantile_balancer.required_bias_histogram_EB.zero_()
        xin = x.clone().requires_grad_()
        out = block(xin, padding_mask=mask)
        out.backward(gout)
        exact = [out.detach(), block.tokens_per_expert_E] + [q.grad for q in ie.parameters()]
        if quantile:
            exact.append(router.quantile_balancer.required_bias_histogram_EB)
        return exact, [aux.instance_acc, router.gate.weight.grad, xin.grad]

    (exact_a, close_a), (exact_b, close_b) = run(True), run(False)
    for i, (a, b) in enumerate(zip(exact_a, exact_b)):
        assert torch.equal(a, b), f"tensor {i}"
    for i, (a, b) in enumerate(zip(close_a, close_b)):
        err = float((a.double() - b.double()).norm() / a.double().norm())
        assert err < (2e-3 if i == 2 else 4e-3 if a.dtype == torch.bfloat16 else 2e-6), f"tensor {i}: {err}"


@pytest.mark.parametrize("E,K,T", [(5, 5, 3), (16, 4, 65), (60, 16, 64), (128, 8, 130), (256, 1, 33)])
@pytest.mark.parametrize("bias", [False, True])
def test_selection_among_equal_values_takes_the_lower_experts(E, K, T, bias):
    """Integer keys of the choice values (csrc/select_rows.h): whole-number logits with many ties, both zeros,
    -inf; with a bias (of zeros) the choice is by score, whose ties are the logits'."""
    from torchllmtuner_amd import ops

    print(f"selection ties E={E} K={K} T={T} bias={bias}", flush=True)
    g = torch.Generator().manual_seed(E)
    x = torch.randint(-2, 3, (T, E), generator=g).float()
    x[x == 0] *= torch.where(torch.rand(int((x == 0).sum()), generator=g) < 0.5, -1.0, 1.0)
    x[:, ::3] = torch.where(torch.rand(T, (E + 2) // 3, generator=g) < 0.2, float("-inf"), x[:, ::3])
    if bias:  # scores of -inf and of logits far below are equal zeros or not: keep the ties exact
        x = x.clamp(min=-2)
    w, ids, _ = ops.router_select_fwd(x.to(DEV), torch.zeros(E, device=DEV) if bias else None, K, "sigmoid", False, 1.0)
    want = torch.sort(x + 0.0, dim=1, descending=True, stable=True).indices[:, :K]
    assert torch.equal(ids.cpu(), want)
    assert torch.allclose(w.cpu(), torch.sigmoid(x).gather(1, want), rtol=1e-6, atol=0)


@pytest.mark.parametrize("dtype,T,D,E", [
    (torch.bfloat16, 1, 8, 1), (torch.bfloat16, 33, 2056, 33), (torch.bfloat16, 1000, 7168, 256), (torch.bfloat16, 32, 1024, 66),
    (torch.float32, 1, 4, 3), (torch.float32, 31, 1028, 32), (torch.float32, 2000, 640, 10), (torch.float32, 4, 3000, 5)])
def test_gate_projection_of_few_tokens_matches_fp64(dtype, T, D, E):
    from torchllmtuner_amd import ops

    print(f"gate {dtype} T={T} D={D} E={E}", flush=True)
    g = torch.Generator().manual_seed(D)
    x, w, b = torch.randn(T, D, generator=g).to(dtype), torch.randn(E, D, generator=g) * 0.05, torch.randn(E, generator=g)
    want = x.double() @ w.double().T + b.double()
    got = ops.router_gate_fwd(x.to(DEV), w.to(DEV), b.to(DEV)).cpu().double()
    # fp32 sums of D products: the error of a plain fp32 dot product bounds it
    scale = (x.double().abs() @ w.double().abs().T + b.double().abs()).max()
    assert float((got - want).abs().max()) < 4e-7 * float(scale)


@pytest.mark.parametrize("counts,D,F", [
    ([1], 384, 384), ([0, 3, 0, 16], 448, 576), ([17, 0, 1, 15, 7], 512, 1024), ([2] * 40, 2048, 384), ([64], 384, 832)])
def test_forward_experts_of_few_rows_match_fp32(counts, D, F):
    """A handful of rows per expert (csrc/grouped_few.hip): one row, exactly 16 and one more, experts
    without rows, contractions whose steps do not divide by the four waves."""
    from torchllmtuner_amd import ops

    print(f"few rows {counts} D={D} F={F}", flush=True)
    g = torch.Generator().manual_seed(D + F)
    R_, E = sum(counts), len(counts)
    x = torch.randn(R_, D, generator=g).bfloat16()
    w1, w3, w2 = (torch.randn(E, *s, generator=g).mul(0.05).bfloat16() for s in ((F, D), (F, D), (D, F)))
    plan = ops.segments_from_counts(torch.tensor(counts, dtype=torch.int32, device=DEV), R_)
    y, gate, up, h = ops.grouped_swiglu_fwd(x.to(DEV), w1.to(DEV), w3.to(DEV), w2.to(DEV), plan)
    seg = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))
    xf = x.float()
    want_g = torch.stack([w1[e].float() @ xf[r] for r, e in enumerate(seg)])
    want_u = torch.stack([w3[e].float() @ xf[r] for r, e in enumerate(seg)])
    want_h = (torch.nn.functional.silu(want_g.bfloat16().float()).bfloat16().float() * want_u.bfloat16().float())
    want_y = torch.stack([w2[e].float() @ h[r].float().cpu() for r, e in enumerate(seg)])
    for name, got, want in (("gate", gate, want_g), ("up", up, want_u), ("h", h, want_h), ("y", y, want_y)):
        err = float((got.float().cpu() - want).norm() / want.norm())
        assert err < 4e-3, f"{name}: rel-L2 {err}"


@pytest.mark.parametrize("dtype,counts,D,F", [
    (torch.float32, [33, 31, 0, 32, 1], 160, 1028), (torch.float32, [5], 36, 28), (torch.float32, [2100], 60, 68),
    (torch.float32, [1, 0, 65], 4, 8), (torch.float32, [130, 3], 68, 36), (torch.float32, [200, 57, 300], 132, 260),
    (torch.bfloat16, [1, 0, 65], 4, 8), (torch.bfloat16, [130, 3], 68, 36), (torch.bfloat16, [0, 257], 124, 380),
    (torch.float32, [700] * 12, 640, 516), (torch.bfloat16, [700] * 12, 652, 644)])
def test_experts_of_any_width_match_fp64(dtype, counts, D, F):
    """csrc/grouped_any.hip, forward and backward: contractions and columns that end inside a tile, empty
    experts, segments that end inside a row tile; the last two sizes take the large tiles."""
    from torchllmtuner_amd import ops

    print(f"any width {dtype} {counts[:4]} D={D} F={F}", flush=True)
    g = torch.Generator().manual_seed(D + F)
    R_, E = sum(counts), len(counts)
    mk = lambda *s, std=0.05: torch.randn(*s, generator=g).mul(std).to(dtype)
    x, dy = mk(R_, D, std=1.0), mk(R_, D, std=1.0)
    w1, w3, w2 = mk(E, F, D), mk(E, F, D), mk(E, D, F)
    dev = [t.to(DEV) for t in (x, w1, w3, w2)]
    plan = ops.segments_from_counts(torch.tensor(counts, dtype=torch.int32, device=DEV), R_)
    y, gate, up, h = ops.grouped_swiglu_fwd(*dev, plan)
    dx, dw1, dw3, dw2 = ops.grouped_swiglu_bwd(dy.to(DEV), *dev, gate, up, h, plan)
    only_dx = ops.grouped_swiglu_bwd(dy.to(DEV), *dev, gate, up, h, plan, need_dw=False)[0]
    assert torch.equal(only_dx, dx)
    ref = [t.double().requires_grad_() for t in (x, w1, w3, w2)]
    out, r0 = [], 0
    for e, c in enumerate(counts):
        xe = ref[0][r0:r0 + c]
        out.append((torch.nn.functional.silu(xe @ ref[1][e].T) * (xe @ ref[2][e].T)) @ ref[3][e].T)
        r0 += c
    want = torch.cat(out)
    want.backward(dy.double())
    tol = 2e-6 if dtype == torch.float32 else 1e-2
    for name, got, exp in (("y", y.detach(), want.detach()), ("dx", dx, ref[0].grad), ("dw1", dw1, ref[1].grad), ("dw3", dw3, ref[2].grad),
                           ("dw2", dw2, ref[3].grad)):
        err = float((got.double().cpu() - exp).norm() / exp.norm())
        assert err < tol, f"{name}: rel-L2 {err}"


@pytest.mark.parametrize("dtype,T,D,E", [(torch.bfloat16, 1, 8, 2), (torch.bfloat16, 1531, 324, 17), (torch.float32, 33, 260, 32),
                                         (torch.float32, 4097, 256, 8)])
def test_gate_gradients_of_few_experts_match_fp64(dtype, T, D, E):
    from torchllmtuner_amd import ops

    print(f"gate backward {dtype} T={T} D={D} E={E}", flush=True)
    g = torch.Generator().manual_seed(T)
    x, w, dl = torch.randn(T, D, generator=g).to(dtype), torch.randn(E, D, generator=g), torch.randn(T, E, generator=g)
    dx, dw = ops.router_gate_bwd(dl.to(DEV), x.to(DEV), w.to(DEV))
    for name, got, exp, tol in (("dx", dx, dl.double() @ w.double(), 1e-6 if dtype == torch.float32 else 4e-3),
                                ("dw", dw, dl.double().T @ x.double(), 1e-6)):
        err = float((got.double().cpu() - exp).norm() / exp.norm())
        assert err < tol, f"{name}: rel-L2 {err}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,K,addend", [(2056, 8, True), (8, 1, False), (516, 11, True), (70, 3, True)])
def test_combine_of_few_tokens_equals_that_of_many(dtype, D, K, addend):
    """The combine deals a row's columns over workgroups: the tokens of a 4096-token call, bit for bit, whatever the
    number of tokens, with absent slots, more than eight slots, rows that end inside a 1 KiB piece and rows that
    are not whole 16-byte vectors; and fp64 sums."""
    from torchllmtuner_amd import _lib

    print(f"combine {dtype} D={D} K={K}", flush=True)
    lib, T, code = _lib.load(), 4096, 0 if dtype == torch.float32 else 1
    g = torch.Generator().manual_seed(D)
    y = torch.randn(500, D, generator=g).to(dtype).to(DEV)
    add = torch.randn(T, D, generator=g).to(dtype).to(DEV) if addend else None
    w = torch.rand(T, K, generator=g).to(DEV)
    rows = torch.randint(-1, 500, (T, K), generator=g, dtype=torch.int32).to(DEV)

    def run(n):
        out = torch.full((n, D), float("nan"), dtype=dtype, device=DEV)
        rc = lib.mi355_combine_add_fwd(y.data_ptr(), code, w.data_ptr(), rows.data_ptr(), add.data_ptr() if addend else None,
                                       out.data_ptr(), n, D, K, 0, torch.cuda.current_stream().cuda_stream)
        _lib.check(rc, "combine_fwd")
        return out

    many = run(T)
    for n in (1, 5, 4095):
        assert torch.equal(run(n), many[:n])
    terms = torch.where((rows >= 0)[..., None], y.double()[rows.clamp(min=0).long()] * w.double()[..., None], 0.0)
    want = terms.sum(1) + (add.double() if addend else 0.0)
    # one rounding of the sum and one of the addition; fp32 sums of K terms
    tol = (2 ** -8 * 2 if dtype == torch.bfloat16 else 2 ** -24 * (K + 2))
    scale = terms.abs().sum(1) + (add.double().abs() if addend else 0.0)
    assert bool(((many.double() - want).abs() <= tol * scale + 1e-30).all())


@pytest.mark.parametrize("dtype,rows,D", [
    (torch.bfloat16, 1, 8), (torch.bfloat16, 5, 520), (torch.bfloat16, 513, 2048), (torch.bfloat16, 1, 2056),
    (torch.bfloat16, 1030, 4096), (torch.bfloat16, 7, 4104), (torch.bfloat16, 515, 8192), (torch.bfloat16, 3, 8200),
    (torch.bfloat16, 2, 16392), (torch.bfloat16, 9, 2051), (torch.float32, 1, 4), (torch.float32, 514, 1024),
    (torch.float32, 3, 1028), (torch.float32, 600, 2052), (torch.float32, 1030, 5000), (torch.float32, 2, 8192),
    (torch.float32, 5, 8196)])
def test_rms_norm_rows_in_registers_match_fp64(dtype, rows, D):
    """csrc/rmsnorm.hip at the ends of its row widths: one wave to a row, four, rows in memory."""
    from torchllmtuner_amd import ops

    print(f"rms {dtype} {rows} x {D}", flush=True)
    g = torch.Generator().manual_seed(D)
    x, dy = torch.randn(rows, D, generator=g).to(dtype), torch.randn(rows, D, generator=g).to(dtype)
    w = (1 + 0.1 * torch.randn(D, generator=g)).to(dtype)
    y, rstd = ops.rms_norm_fwd(x.to(DEV), w.to(DEV), 1e-6)
    dx, dw = ops.rms_norm_bwd(dy.to(DEV), x.to(DEV), w.to(DEV), rstd)
    ref = [t.double().requires_grad_() for t in (x, w)]
    want = ref[0] * torch.rsqrt(ref[0].square().mean(-1, keepdim=True) + 1e-6) * ref[1]
    want.backward(dy.double())
    # one rounding to bf16 (half an ulp: 2^-9) per result; fp32 sums of D or of rows terms, relative to their norms
    tol = 2 ** -8 if dtype == torch.bfloat16 else 2e-6
    for name, got, exp in (("y", y, want.detach()), ("dx", dx, ref[0].grad), ("dw", dw, ref[1].grad)):
        err = float((got.double().cpu() - exp).norm() / exp.norm())
        assert err < tol, f"{name}: rel-L2 {err}"
    only_dw = ops.rms_norm_bwd(dy.to(DEV), x.to(DEV), w.to(DEV), rstd, need_dx=False)[1]
    assert torch.equal(only_dw, dw)


@pytest.mark.parametrize("T,E,K,local,align,groups", [
    (1, 1, 1, None, 1, None), (32, 60, 16, None, 1, None), (33, 128, 8, (32, 96), 1, None), (64, 256, 16, None, 128, (8, 4)),
    (65, 17, 3, None, 1, None), (1000, 256, 8, (0, 32), 16, (8, 4)), (7000, 132, 4, None, 1, None),
    (7001, 132, 4, None, 1, None), (8192, 128, 8, None, 1, None), (8193, 128, 8, (5, 6), 1, None),
    (16449, 64, 2, None, 16, None)])
def test_route_plan_equals_selection_and_plan(T, E, K, local, align, groups):
    """The C entry without statistics: ids, weights and every array of the plan, against the selection and the plan
    as two calls; around the sizes at which its launches change."""
    from torchllmtuner_amd import _lib, ops

    print(f"route plan T={T} E={E} K={K} local={local} align={align} groups={groups}", flush=True)
    lo, hi = local or (0, E)
    El, splits = hi - lo, 3
    g = torch.Generator().manual_seed(T)
    partial = torch.randn(splits, T, E, generator=g).to(DEV)
    bias, expert_b = torch.randn(E, generator=g).to(DEV), (0.1 * torch.randn(E, generator=g)).to(DEV)
    logits = partial[0] + partial[1] + partial[2] + bias
    G, L = groups or (0, 0)
    w, ids, _ = ops.router_select_fwd(logits, expert_b, K, "sigmoid", True, 2.5, G, L)
    plan = ops.permute_plan(ids, E, lo, hi, align)
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=DEV)
    f32 = lambda *n: torch.full(n, float("nan"), device=DEV)
    R_, cap = plan.row_capacity, plan.tile_capacity
    got_logits, got_w, got_ids = f32(T, E), f32(T, K), torch.empty(T, K, dtype=torch.int64, device=DEV)
    counts, offsets, seg_counts, ros, sor, tor = i32(E), i32(El + 1), i32(2 * El), i32(T * K), i32(R_), i32(R_)
    scale, te, tr, nt = f32(R_), i32(cap), i32(cap), i32(1)
    lib = _lib.load()
    work = torch.empty(max(1, lib.mi355_route_plan_workspace_bytes(T, K, E)), dtype=torch.uint8, device=DEV)
    rc = lib.mi355_route_plan(
        partial.data_ptr(), splits, bias.data_ptr(), got_logits.data_ptr(), expert_b.data_ptr(), T, E, K, 0, 1, 2.5, G, L,
        got_w.data_ptr(), got_ids.data_ptr(), lo, hi, align, ops.TILE_M, counts.data_ptr(), offsets.data_ptr(),
        seg_counts.data_ptr(), ros.data_ptr(), sor.data_ptr(), tor.data_ptr(), scale.data_ptr(), R_, te.data_ptr(),
        tr.data_ptr(), nt.data_ptr(), cap, work.data_ptr(), torch.cuda.current_stream().cuda_stream)
    _lib.check(rc, "route_plan")
    n = int(nt)
    for name, a, b in (("logits", got_logits, logits), ("ids", got_ids, ids), ("weights", got_w, w), ("counts", counts, plan.counts_E),
                       ("offsets", offsets, plan.seg_offsets), ("seg_counts", seg_counts[:El], plan.seg_counts),
                       ("order", seg_counts[El:], plan.expert_order), ("row_of_slot", ros, plan.row_of_slot),
                       ("slot_of_row", sor, plan.slot_of_row), ("token_of_row", tor, plan.token_of_row),
                       ("row_scale", scale, ops.combine_row_scale(w, plan)), ("num_tiles", nt, plan.num_tiles),
                       ("tile_expert", te[:n], plan.tile_expert[:n]), ("tile_row0", tr[:n], plan.tile_row0[:n])):
        assert torch.equal(a, b), name


# the statistics' sums take 8 * (512 // E) workgroups of 32 tokens at a time, or 8 * (1024 // E) of 64 above 8192 tokens (7000 past 128 experts): whole rounds of
# them and one workgroup more, the fewest workgroups, experts that do not divide the lanes, workgroups of several chunks of tokens
@pytest.mark.parametrize("T,E,K", [(512, 256, 2), (513, 256, 2), (2048, 60, 4), (2049, 60, 4), (65, 1, 1), (8192, 128, 8), (8193, 128, 8), (7001, 256, 3), (16449, 5, 2),
                                   (20000, 100, 16)])
@pytest.mark.parametrize("counts,loss", [(True, True), (True, False), (False, True)])
def test_statistics_of_many_workgroups(T, E, K, counts, loss):
    """Valid counts, and the balance loss of them and of the tokens' score shares in fp64."""
    from torchllmtuner_amd import _lib, ops

    print(f"route plan statistics T={T} E={E} K={K} counts={counts} loss={loss}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(T + E)
    logits = torch.randn(T, E, generator=g, device=DEV)
    padding = torch.rand(T, generator=g, device=DEV) < 0.2
    denominator = torch.tensor([float(T)], device=DEV)
    i32 = lambda n: torch.full((n,), -7, dtype=torch.int32, device=DEV)
    cap = T * K // ops.TILE_M + E + 1
    w, ids = torch.empty(T, K, device=DEV), torch.empty(T, K, dtype=torch.int64, device=DEV)
    total, offsets, seg_counts, ros, sor, tor, te, tr, nt, valid = (i32(n) for n in (E, E + 1, 2 * E, T * K, T * K, T * K, cap, cap, 1, E))
    f, scale, acc = (torch.full((n,), v, device=DEV) for n, v in ((E, float("nan")), (1, float("nan")), (1, 0.5)))
    lib = _lib.load()
    work, stats = (torch.empty(max(1, n), dtype=torch.uint8, device=DEV)
                   for n in (lib.mi355_route_plan_workspace_bytes(T, K, E), lib.mi355_route_stats_workspace_bytes(T, E)))
    at = lambda t, wanted=True: t.data_ptr() if wanted else None
    _lib.check(lib.mi355_route_plan_stats(
        at(logits), 1, None, None, None, T, E, K, 1, 0, 1.0, 0, 0, at(w), at(ids), 0, E, 1, ops.TILE_M, at(total), at(offsets),
        at(seg_counts), at(ros), at(sor), at(tor), None, T * K, at(te), at(tr), at(nt), cap, at(work), at(padding), at(valid, counts), None, None,
        at(f, loss), at(scale, loss), at(acc, loss), 0, at(denominator), 2.0, at(stats), torch.cuda.current_stream().cuda_stream),
        "route_plan_stats")
    assert torch.equal(total.long(), torch.bincount(ids.flatten(), minlength=E))
    want = torch.bincount(ids[~padding].flatten(), minlength=E)
    assert torch.equal(valid.long(), want) if counts else bool((valid == -7).all())
    if not loss:
        assert bool(f.isnan().all()) and float(acc) == 0.5
        return
    scores = logits.double().softmax(1)
    p = (scores / scores.sum(1, keepdim=True))[~padding].sum(0)
    want_f = want.double() * (E / want.sum().clamp(min=1e-12))
    want_loss = float((want_f * p).sum()) / T
    assert abs(float(scale) * T / 2.0 - 1.0) <= 2.0 ** -23
    # (one rounding; of f two.  Of the loss: each share an exponential, sums of up to 256 terms by fours and their quotients, 2^-20; then sums of at most T / 4096 + 2
    # tokens of a wave, 16 waves, 256 workgroups and 8 steps of a tree over the experts, products, and the sum with what was there)
    assert float((f.double() - want_f).abs().max()) <= 2.0 ** -22 * float(want_f.max())
    bound = (2.0 ** -20 + (T / 4096 + 2 + 16 + 256 + 8 + 4) * 2.0 ** -24) * want_loss + 2.0 ** -24 * (0.5 + want_loss)
    assert abs(float(acc) - 0.5 - want_loss) <= bound


def test_default_overlap_adds_the_input_gradients_in_another_order_than_the_stages():
    """With a shared expert beside the routed path, as by default, the engine adds the stages' three bf16 input
    gradients as (routed + gate) + shared; the operator as (routed + shared) + gate, whatever the overlap.  All
    else is the same bits; the two sums differ by their roundings."""
    dtype, T, D, E, K, F = torch.bfloat16, 1025, 512, 64, 4, 384
    spec = R.RouterSpec(E, K, score_func="softmax", route_norm=True)
    p = make_params(E, D, F, dtype, seed=3, std=0.05, shared_F=448)
    g = torch.Generator().manual_seed(4)
    x, gout = (torch.randn(T, D, generator=g).to(dtype).to(DEV) for _ in range(2))

    def run(in_stages, overlap=True, shared=True, gate=True):
        block = build_block(p, spec, D, F, dtype, DEV).train()
        assert block.overlap_shared_experts
        block.overlap_shared_experts = overlap
        if not shared:
            block.shared_experts = None
        if in_stages:
            block.router.register_forward_hook(lambda m, a, out: None if gate else (out[0].detach(), *out[1:]))
        xin = x.clone().requires_grad_()
        out = block(xin)
        out.backward(gout)
        return [xin.grad, out.detach(), block.tokens_per_expert_E] + [q.grad for q in block.parameters() if q.grad is not None]

    one, stages = run(False), run(True)
    for overlap in (True, False):
        for a, b in zip(one, run(False, overlap), strict=True):
            assert torch.equal(a, b)
    for i, (a, b) in enumerate(zip(one[1:], stages[1:], strict=True)):
        assert torch.equal(a, b), f"tensor {i}"
    assert torch.equal(one[0], run(True, overlap=False)[0])  # (one stream: the operator's order)
    # routed, gate and shared by themselves bound the two roundings of either sum (unit roundoff 2^-8)
    block = build_block(p, spec, D, F, dtype, DEV)
    xin = x.clone().requires_grad_()
    block.shared_experts(xin).backward(gout)
    shared, routed, routed_gate = (t.double() for t in (xin.grad, run(True, shared=False, gate=False)[0], run(True, shared=False)[0]))
    total = routed_gate + shared
    bound = 2.0 ** -8 * (routed_gate.abs() + (routed + shared).abs() + 2 * total.abs()) * (1 + 2.0 ** -5) + 1e-30
    diff = (one[0].double() - stages[0].double()).abs()
    assert bool((diff <= bound).all()), float((diff / bound).max())


@pytest.mark.parametrize("dtype,T,D,F", [(torch.bfloat16, 700, 512, 384), (torch.bfloat16, 3, 512, 384), (torch.float32, 300, 64, 100)])
@pytest.mark.parametrize("padded", [False, True])
def test_running_counts_are_added_once_whichever_launch_adds_them(dtype, T, D, F, padded):
    """In the combine's launch, or, where a checkpoint may replay the forward and stop before its end, behind it; without gradients too, and for
    buffers that the operator does not take."""
    from torch.utils.checkpoint import checkpoint

    from torchllmtuner_amd.moe.layer import in_checkpoint_recompute

    E, K = 20, 3
    print(f"running counts {dtype} T={T} padded={padded}", flush=True)
    p = make_params(E, D, F, dtype, seed=T, std=0.05)
    g = torch.Generator().manual_seed(T)
    x = torch.randn(T, D, generator=g).to(dtype).to(DEV)
    mask = (torch.rand(T, generator=g) < 0.3).to(DEV) if padded else None
    block = build_block(p, R.RouterSpec(E, K, score_func="softmax", route_norm=True), D, F, dtype, DEV).train()
    with torch.no_grad():
        ids = block._forward_as_one(x, mask)
        want = ids[1].double()
    assert want.sum() == K * (T if mask is None else int((~mask).sum())) and not block.tokens_per_expert_E.any()

    def counted(run, times=1):
        block.tokens_per_expert_E.fill_(5.0)
        run()
        assert torch.equal(block.tokens_per_expert_E.double(), 5.0 + times * want)

    call = lambda: block(x.clone().requires_grad_(), padding_mask=mask)
    assert block._totals(x) is block.tokens_per_expert_E
    counted(call)
    counted(lambda: (call(), call()), 2)
    counted(lambda: torch.no_grad()(call)())
    counted(lambda: checkpoint(call, use_reentrant=False).sum().backward())
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert block._totals(x) is None
        counted(call)
    handle = block.router.register_forward_hook(lambda *a: None)  # the stages
    counted(call)
    handle.remove()
    token = in_checkpoint_recompute.set(True)
    counted(call, 0)
    in_checkpoint_recompute.reset(token)
    block.eval()
    counted(call, 0)
    block.train()
    for other in (torch.zeros(E, dtype=torch.float64, device=DEV), torch.zeros(E, 2, device=DEV)[:, 0]):
        block.tokens_per_expert_E = other
        assert block._totals(x) is None
        counted(call)


@pytest.mark.parametrize("T", [0, 1, 5])
def test_the_combine_adds_counts_with_and_without_tokens(T):
    from torchllmtuner_amd import _lib

    E, K, D = 300, 2, 16
    p = lambda t: t.data_ptr() if t is not None else None
    counts = torch.arange(E, dtype=torch.int32, device=DEV)
    totals = torch.full((E,), 2.0, device=DEV)
    y, out = torch.ones(T * K, D, device=DEV), torch.zeros(T, D, device=DEV)
    weights, rows = torch.full((T, K), 0.5, device=DEV), torch.arange(T * K, dtype=torch.int32, device=DEV)
    some = lambda t: p(t) if T else None
    _lib.check(_lib.load().mi355_combine_count_fwd(some(y), 0, some(weights), some(rows), None, some(out), T, D, K, 0, p(counts), p(totals), E,
                                                   torch.cuda.current_stream().cuda_stream), "combine_count_fwd")
    assert torch.equal(totals, counts + 2.0) and torch.equal(out, torch.ones_like(out))
