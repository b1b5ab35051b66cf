// The whole MoE block as one operator: router, plan, routed experts, combine and (when there is one)
// the dense shared expert, with one autograd node whose backward is written out below.
//
// The stage operators of torch_ext.cpp compute the same things one at a time, for callers that
// look between the stages (hooks, other dispatchers, other routers, tracing); MoE.forward comes here
// when nothing hangs on the stages.  What the single operator saves:
//   * host time: a forward pass is one trip through the dispatcher and about ten C calls instead of four
//     operators, a plan object and its views (83 -> 35 us at one token), a training step has one autograd
//     node instead of three to five;
//   * launches: the router's partial logits are summed by the selection, selection and plan are one or two
//     launches instead of four, the score gradient's pieces are summed by the selection's backward, and
//     the additions of (T, D) tensors -- shared expert's output, the two or three input gradients -- ride
//     in kernels that hold the other operand anyway.
// Every kernel and every rounding is the stage operators' own: both ways give the same bits.
//
// Memory.  Integers and fp32 of the plan and the router share one allocation (`meta`, kept for the
// backward); everything else comes from PyTorch's allocator on the current stream.  Work on the
// library's side streams is forked from the current stream and joined before the operator returns, so
// buffers need no record_stream.
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/library.h>

#include <cstring>
#include <tuple>
#include <vector>

#include "torch_common.h"

namespace {

using namespace mi355_torch;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Config {
  int64_t K, score_func, route_norm, num_groups, num_limited, lo, hi, align, round_terms, overlap;
  double route_scale;

  std::vector<int64_t> pack() const {
    std::vector<int64_t> v{K, score_func, route_norm, num_groups, num_limited, lo, hi, align, round_terms, overlap, 0};
    std::memcpy(&v[10], &route_scale, sizeof(double));
    return v;
  }
  static Config unpack(const std::vector<int64_t>& v) {
    Config c{v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8], v[9], 0.0};
    std::memcpy(&c.route_scale, &v[10], sizeof(double));
    return c;
  }
};

// The block's tensors; undefined where the block has none.
struct Block {
  Tensor x, gate_w, gate_b, expert_b, w1, w3, w2, sg, su, sd;
  Config c;
  int64_t T, D, E, F, El, N, R, Fs, tile_m, tile_cap, shared_cap;
  int dt, gate_dt;
  bool folded;         // the folded kernels (token gather, combine's backward inside the experts') serve the routed part
  bool shared_folded;  // the bf16 MFMA kernels serve the shared expert

  void sizes() {
    T = x.size(0); D = x.size(1); E = gate_w.size(0); F = w1.size(1); El = c.hi - c.lo;
    N = T * c.K;
    R = N + (c.align > 1 ? El * (c.align - 1) : 0);
    tile_m = mi355_grouped_tile_m(MI355_BF16);
    tile_cap = N / tile_m + El + 1;
    dt = dtype_code(x);
    gate_dt = dtype_code(gate_w);
    folded = mi355_grouped_combine_bwd_slots(dt, D, F) > 0 && T * D * 2 < (int64_t{1} << 32);
    Fs = sg.defined() ? sg.size(0) : 0;
    shared_cap = Fs > 0 ? (T + tile_m - 1) / tile_m : 0;
    shared_folded = Fs > 0 && mi355_grouped_combine_bwd_slots(dt, D, Fs) > 0;
  }
};

// The plan's and the router's arrays inside `meta`.
struct Meta {
  int64_t* ids;
  float *weights, *logits, *row_scale;
  int32_t *counts, *seg_offsets, *seg_counts, *tile_expert, *tile_row0, *num_tiles, *row_of_slot, *slot_of_row,
      *token_of_row;
  int32_t *s_offsets, *s_counts, *s_expert, *s_row0, *s_num;
  int64_t bytes;

  Meta(const Block& b, void* base, int32_t* counts_E) : counts(counts_E) {
    char* p = static_cast<char*>(base);
    int64_t at = 0;
    auto take = [&](auto*& out, int64_t n) {
      using T = std::remove_reference_t<decltype(*out)>;
      out = reinterpret_cast<T*>(p + at);
      at += (n * static_cast<int64_t>(sizeof(T)) + 255) / 256 * 256;
    };
    take(ids, b.N);
    take(weights, b.N);
    take(logits, b.T * b.E);
    take(row_scale, b.R);
    take(row_of_slot, b.N);
    take(slot_of_row, b.R);
    take(token_of_row, b.R);
    take(seg_offsets, b.El + 1);
    take(seg_counts, 2 * b.El);
    take(tile_expert, b.tile_cap);
    take(tile_row0, b.tile_cap);
    take(num_tiles, 1);
    take(s_offsets, 2);
    take(s_counts, 2);
    take(s_expert, b.shared_cap);
    take(s_row0, b.shared_cap);
    take(s_num, 1);
    bytes = at;
  }
};

// Forks `side` behind everything `main` holds so far, and back.
struct Fork {
  SideStream* side;
  hipStream_t main;
  bool open = false;
  Fork(SideStream* s, hipStream_t m) : side(s), main(m) {}
  void start() { follow(main); }
  // the side stream waits for everything on `from`, which is behind `main` itself
  void follow(hipStream_t from) {
    TORCH_CHECK(side->chain(side->fork, from, side->stream), "moe_block: cannot fork to the side stream: ",
                hipGetErrorString(hipGetLastError()));
    open = true;
  }
  void join() {
    if (!open) return;
    open = false;
    TORCH_CHECK(side->chain(side->join, side->stream, main), "moe_block: cannot join the side stream: ",
                hipGetErrorString(hipGetLastError()));
  }
  // an error between the two must not leave the side stream's work unordered with the buffers' next use
  ~Fork() {
    if (open) (void)side->chain(side->join, side->stream, main);
  }
};

struct Kept {  // what the backward reads besides the inputs
  Tensor meta, pieces, rows, gate, up, h, y, s_gate, s_up, s_h;
};

void shared_forward(const Block& b, const Meta& m, Kept& kept, const Tensor& y, bool save, void* stream) {
  check(mi355_segments_dense(b.T, b.tile_m, m.s_offsets, m.s_counts, m.s_expert, m.s_row0, m.s_num, b.shared_cap, stream),
        "segments_dense");
  // (gate and up are the generic kernels' own intermediates)
  const bool gu = save || !b.shared_folded;
  check(mi355_grouped_swiglu_fwd(ptr(b.x), nullptr, b.T, ptr(b.sg), ptr(b.su), ptr(b.sd), b.dt, m.s_offsets, m.s_counts,
                                 m.s_expert, m.s_row0, m.s_num, b.shared_cap, gu ? ptr(kept.s_gate) : nullptr,
                                 gu ? ptr(kept.s_up) : nullptr, ptr(kept.s_h), ptr(y), 1, b.D, b.Fs, b.T, stream),
        "shared expert");
}

std::tuple<Tensor, Tensor> block_forward(const Block& b, bool save, Kept& kept) {
  Launch L(b.x);
  const Config& c = b.c;
  const auto opts = b.x.options();
  const hipStream_t main = static_cast<hipStream_t>(L.stream);
  Tensor counts = at::empty({b.E}, opts.dtype(at::kInt));
  const int64_t meta_bytes = Meta(b, nullptr, nullptr).bytes;
  kept.meta = bytes(meta_bytes, b.x);
  const Meta m(b, kept.meta.data_ptr(), counts.data_ptr<int32_t>());
  Tensor gate_b, expert_b;
  if (b.gate_b.defined()) gate_b = cf(b.gate_b);
  if (b.expert_b.defined()) expert_b = cf(b.expert_b);

  // shared expert: beside the router and the routed experts when it may, else right before the sum
  SideStream* aux = b.Fs > 0 && c.overlap ? side_stream(b.x.device().index(), main, 1) : nullptr;
  Fork shared(aux, main);
  Tensor y_shared;
  if (b.Fs > 0) {
    const bool gu = save || !b.shared_folded;
    y_shared = at::empty({b.T, b.D}, opts);
    kept.s_h = at::empty({b.T, b.Fs}, opts);
    if (gu) {
      kept.s_gate = at::empty({b.T, b.Fs}, opts);
      kept.s_up = at::empty({b.T, b.Fs}, opts);
    }
    if (aux) {
      shared.start();
      shared_forward(b, m, kept, y_shared, save, aux->stream);
    }
  }

  // router: partial logits, then selection and plan
  const int splits = mi355_router_gate_fwd_splits(b.dt, b.gate_dt, b.T, b.D, b.E);
  const int64_t piece_bytes = splits > 0 ? mi355_router_gate_fwd_pieces_bytes(b.dt, b.gate_dt, b.T, b.D, b.E) : 0;
  const int64_t partial_bytes = splits > 1 ? splits * b.T * b.E * 4
                                : splits == 0 ? mi355_router_gate_fwd_workspace_bytes(b.T, b.D, b.E) : 0;
  const int64_t plan_bytes = mi355_route_plan_workspace_bytes(b.T, c.K, b.E);
  const int64_t plan_at = (partial_bytes + 255) / 256 * 256;
  Tensor scratch;
  if (partial_bytes + plan_bytes > 0) scratch = bytes(plan_at + plan_bytes, b.x);
  char* work = scratch.defined() ? static_cast<char*>(scratch.data_ptr()) : nullptr;
  if (piece_bytes > 0) kept.pieces = bytes(piece_bytes, b.x);
  float* partial = splits > 1 ? reinterpret_cast<float*>(work) : m.logits;
  if (splits > 0)
    check(mi355_router_gate_fwd_partial(ptr(b.x), b.dt, fptr(b.gate_w), fptr(gate_b), partial, ptr(kept.pieces), b.T,
                                        b.D, b.E, L.stream),
          "router_gate_fwd");
  else
    check(mi355_router_gate_fwd(ptr(b.x), b.dt, ptr(b.gate_w), b.gate_dt, fptr(gate_b), m.logits,
                                partial_bytes > 0 ? work : nullptr, b.T, b.D, b.E, L.stream),
          "router_gate_fwd");
  check(mi355_route_plan(partial, splits > 1 ? splits : 1, fptr(gate_b), save && splits > 1 ? m.logits : nullptr,
                         fptr(expert_b), b.T, b.E, c.K, (int)c.score_func, (int)c.route_norm, (float)c.route_scale,
                         (int)c.num_groups, (int)c.num_limited, m.weights, m.ids, c.lo, c.hi, c.align, b.tile_m,
                         m.counts, m.seg_offsets, m.seg_counts, m.row_of_slot, m.slot_of_row, m.token_of_row,
                         save && b.folded ? m.row_scale : nullptr, b.R, m.tile_expert, m.tile_row0, m.num_tiles,
                         b.tile_cap, plan_bytes > 0 ? work + plan_at : nullptr, L.stream),
        "route_plan");

  // routed experts
  Tensor y = at::empty({b.R, b.D}, opts), h = at::empty({b.R, b.F}, opts);
  if (b.folded) {
    if (save) {
      kept.gate = at::empty({b.R, b.F}, opts);
      kept.up = at::empty({b.R, b.F}, opts);
    }
    check(mi355_grouped_swiglu_fwd(ptr(b.x), m.token_of_row, b.T, ptr(b.w1), ptr(b.w3), ptr(b.w2), b.dt, m.seg_offsets,
                                   m.seg_counts, m.tile_expert, m.tile_row0, m.num_tiles, b.tile_cap, ptr(kept.gate),
                                   ptr(kept.up), ptr(h), ptr(y), b.El, b.D, b.F, b.R, L.stream),
          "grouped_swiglu_fwd");
  } else {
    kept.rows = at::empty({b.R, b.D}, opts);
    kept.gate = at::empty({b.R, b.F}, opts);
    kept.up = at::empty({b.R, b.F}, opts);
    check(mi355_permute_rows_fwd(ptr(b.x), b.dt, m.row_of_slot, c.align > 1 ? m.slot_of_row : nullptr,
                                 m.seg_offsets + b.El, ptr(kept.rows), b.T, b.D, c.K, b.R, L.stream),
          "permute_rows_fwd");
    check(mi355_grouped_swiglu_fwd(ptr(kept.rows), nullptr, b.R, ptr(b.w1), ptr(b.w3), ptr(b.w2), b.dt, m.seg_offsets,
                                   m.seg_counts, m.tile_expert, m.tile_row0, m.num_tiles, b.tile_cap, ptr(kept.gate),
                                   ptr(kept.up), ptr(h), ptr(y), b.El, b.D, b.F, b.R, L.stream),
          "grouped_swiglu_fwd");
    kept.h = h;
    kept.y = y;
  }
  if (b.Fs > 0 && !aux) shared_forward(b, m, kept, y_shared, save, L.stream);
  shared.join();
  Tensor out = at::empty({b.T, b.D}, opts);
  check(mi355_combine_add_fwd(ptr(y), b.dt, m.weights, m.row_of_slot, ptr(y_shared), ptr(out), b.T, b.D, c.K,
                              (int)c.round_terms, L.stream),
        "combine_fwd");
  return {out, counts};
}

struct Needs {
  bool x, gate_w, gate_b, experts, shared;
};
struct Grads {
  Tensor x, gate_w, gate_b, w1, w3, w2, sg, su, sd;
};

Grads block_backward(const Block& b, const Kept& k, const Tensor& dout_, const Needs& need) {
  Launch L(b.x);
  const Config& c = b.c;
  const auto opts = b.x.options();
  const auto f32 = opts.dtype(at::kFloat);
  const hipStream_t main = static_cast<hipStream_t>(L.stream);
  const Tensor dout = (dout_.scalar_type() == b.x.scalar_type() ? dout_ : dout_.to(b.x.scalar_type())).contiguous();
  const Meta m(b, k.meta.data_ptr(), nullptr);
  const int device = b.x.device().index();
  Grads g;
  const bool gate = need.gate_w || need.gate_b, routed = need.x || gate || need.experts;

  // ---- shared expert: dH and dX beside the routed part where they may be, its weight gradients in front
  // of the routed ones on the stream those use
  Tensor dx_shared, s_dgate, s_dup;
  const bool run_shared = b.Fs > 0 && (need.x || need.shared);
  SideStream* aux = run_shared && c.overlap && routed ? side_stream(device, main, 1) : nullptr;
  SideStream* side = routed && need.x && ((b.folded && need.experts) || (b.shared_folded && aux && need.shared))
                         ? side_stream(device, main, 0) : nullptr;
  Fork shared(aux, main), weights(side, main);
  if (run_shared) {
    s_dgate = at::empty({b.T, b.Fs}, opts);
    s_dup = at::empty({b.T, b.Fs}, opts);
    if (need.x) dx_shared = at::empty({b.T, b.D}, opts);
    if (need.shared) {
      g.sg = at::empty_like(b.sg);
      g.su = at::empty_like(b.su);
      g.sd = at::empty_like(b.sd);
    }
    if (aux) shared.start();
    void* stream = aux ? static_cast<void*>(aux->stream) : L.stream;
    if (b.shared_folded) {
      auto stage = [&](int s, void* on) {
        check(mi355_grouped_swiglu_stage(s, ptr(dout), ptr(b.x), nullptr, b.T, ptr(b.sg), ptr(b.su), ptr(b.sd),
                                         ptr(k.s_gate), ptr(k.s_up), ptr(k.s_h), nullptr, m.s_offsets, m.s_counts,
                                         m.s_expert, m.s_row0, m.s_num, b.shared_cap, ptr(s_dgate), ptr(s_dup),
                                         ptr(dx_shared), ptr(g.sg), ptr(g.su), ptr(g.sd), 1, b.D, b.Fs, b.T, on),
              "shared expert backward");
      };
      stage(MI355_STAGE_DH, stream);
      void* weight_stream = stream;
      if (aux && side && need.shared) {
        weights.follow(aux->stream);
        weight_stream = side->stream;
      }
      if (need.x) stage(MI355_STAGE_DX, stream);
      if (need.shared)
        for (int s : {MI355_STAGE_DW2, MI355_STAGE_DW1, MI355_STAGE_DW3}) stage(s, weight_stream);
    } else {
      check(mi355_grouped_swiglu_bwd(ptr(dout), ptr(b.x), nullptr, b.T, ptr(b.sg), ptr(b.su), ptr(b.sd), ptr(k.s_gate),
                                     ptr(k.s_up), ptr(k.s_h), b.dt, m.s_offsets, m.s_counts, m.s_expert, m.s_row0,
                                     m.s_num, b.shared_cap, ptr(s_dgate), ptr(s_dup), ptr(dx_shared), ptr(g.sg),
                                     ptr(g.su), ptr(g.sd), 1, b.D, b.Fs, b.T, stream),
            "shared expert backward");
    }
  }
  if (!routed) return g;

  // ---- routed experts: dx_routed is the sum over a token's rows plus the shared expert's part
  Tensor dx_routed, dlogits;
  if (need.x) dx_routed = at::empty({b.T, b.D}, opts);
  if (need.experts) {
    g.w1 = at::empty_like(b.w1);
    g.w3 = at::empty_like(b.w3);
    g.w2 = at::empty_like(b.w2);
  }
  if (need.x || gate) dlogits = at::empty({b.T, b.E}, f32);
  auto row_sum = [&](const Tensor& drows) {
    if (!need.x) return;
    shared.join();
    check(mi355_permute_rows_add_bwd(ptr(drows), b.dt, m.row_of_slot, ptr(dx_shared), ptr(dx_routed), b.T, b.D, c.K,
                                     L.stream),
          "permute_rows_bwd");
  };
  Tensor dgate = at::empty_like(k.gate), dup = at::empty_like(k.up);
  Tensor drows, hs, partial, dy, dweights;
  if (need.x) drows = at::empty({b.R, b.D}, opts);
  if (b.folded) {
    const int64_t slots = mi355_grouped_combine_bwd_slots(b.dt, b.D, b.F);
    hs = at::empty_like(k.gate);
    partial = at::empty({b.R, slots}, f32);
    auto run = [&](int stages, void* stream) {
      check(mi355_grouped_swiglu_combine_bwd(
                ptr(dout), ptr(b.x), m.token_of_row, b.T, m.row_scale, ptr(b.w1), ptr(b.w3), ptr(b.w2), ptr(k.gate),
                ptr(k.up), b.dt, m.seg_offsets, m.seg_counts, m.tile_expert, m.tile_row0, m.num_tiles, b.tile_cap,
                ptr(dgate), ptr(dup), ptr(hs), static_cast<float*>(ptr(partial)), ptr(drows), ptr(g.w1), ptr(g.w3),
                ptr(g.w2), b.El, b.D, b.F, b.R, stages, stream),
            "grouped_swiglu_combine_bwd");
    };
    constexpr int kWeights = MI355_STAGE_DW2 | MI355_STAGE_DW1 | MI355_STAGE_DW3;
    run(MI355_STAGE_DH, L.stream);
    // Everything after dH reads what dH wrote and nothing else of this call: the weight gradients go to the
    // side stream, the input gradient and everything behind it stay here.
    if (side && need.experts) {
      weights.start();
      run(kWeights, side->stream);
    }
    if (need.x) run(MI355_STAGE_DX, L.stream);
    row_sum(drows);
    if (dlogits.defined())
      check(mi355_router_select_dots_bwd(m.logits, m.ids, fptr(partial), slots, m.row_of_slot, b.R,
                                         dlogits.data_ptr<float>(), b.T, b.E, c.K, (int)c.score_func,
                                         (int)c.route_norm, (float)c.route_scale, L.stream),
            "router_select_bwd");
    if (need.experts && !side) run(kWeights, L.stream);
  } else {
    const int32_t* pad = c.align > 1 ? m.slot_of_row : nullptr;
    dy = at::empty({b.R, b.D}, opts);
    dweights = at::empty({b.T, c.K}, f32);
    check(mi355_combine_bwd(ptr(dout), ptr(k.y), b.dt, m.weights, m.row_of_slot, pad, m.seg_offsets + b.El, ptr(dy),
                            dweights.data_ptr<float>(), b.T, b.D, c.K, b.R, L.stream),
          "combine_bwd");
    if (need.x || need.experts)
      check(mi355_grouped_swiglu_bwd(ptr(dy), ptr(k.rows), nullptr, b.R, ptr(b.w1), ptr(b.w3), ptr(b.w2), ptr(k.gate),
                                     ptr(k.up), ptr(k.h), b.dt, m.seg_offsets, m.seg_counts, m.tile_expert, m.tile_row0,
                                     m.num_tiles, b.tile_cap, ptr(dgate), ptr(dup), ptr(drows), ptr(g.w1), ptr(g.w3),
                                     ptr(g.w2), b.El, b.D, b.F, b.R, L.stream),
            "grouped_swiglu_bwd");
    row_sum(drows);
    if (dlogits.defined())
      check(mi355_router_select_bwd(m.logits, m.ids, fptr(dweights), nullptr, dlogits.data_ptr<float>(), b.T, b.E, c.K,
                                    (int)c.score_func, (int)c.route_norm, (float)c.route_scale, MI355_SELECT_TOPK,
                                    L.stream),
            "router_select_bwd");
  }

  // ---- router gate; the input gradient is complete with its part
  if (need.x || need.gate_w) {
    if (need.x) g.x = at::empty({b.T, b.D}, opts);
    if (need.gate_w) g.gate_w = at::empty_like(b.gate_w);
    Tensor ws = bytes(mi355_router_gate_bwd_workspace_bytes(b.T, b.D, b.E), b.x);
    check(mi355_router_gate_add_bwd(fptr(dlogits), ptr(b.x), b.dt, ptr(b.gate_w), b.gate_dt, ptr(k.pieces),
                                    ptr(dx_routed), ptr(g.x), ptr(g.gate_w), ptr(ws), b.T, b.D, b.E, L.stream),
          "router_gate_bwd");
  }
  if (need.gate_b) g.gate_b = dlogits.sum(0).to(b.gate_b.scalar_type());
  weights.join();
  shared.join();
  return g;
}

Tensor some(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }

struct MoeBlock : public torch::autograd::Function<MoeBlock> {
  static variable_list forward(AutogradContext* ctx, const Tensor& x, const Tensor& gate_w, const OptTensor& gate_b,
                               const OptTensor& expert_b, const Tensor& w1, const Tensor& w3, const Tensor& w2,
                               const OptTensor& sg, const OptTensor& su, const OptTensor& sd, const Config& c) {
    at::AutoDispatchBelowADInplaceOrView below;
    Block b{x, gate_w, some(gate_b), some(expert_b), w1, w3, w2, some(sg), some(su), some(sd), c};
    b.sizes();
    Kept k;
    auto [out, counts] = block_forward(b, true, k);
    ctx->save_for_backward({x, gate_w, b.gate_b, w1, w3, w2, b.sg, b.su, b.sd, k.meta, k.pieces, k.rows, k.gate, k.up, k.h, k.y,
                            k.s_gate, k.s_up, k.s_h});
    auto packed = c.pack();
    packed.push_back(b.expert_b.defined());
    ctx->saved_data["config"] = packed;
    ctx->set_materialize_grads(false);
    ctx->mark_non_differentiable({counts});
    return {out, counts};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(11);
    if (!grads[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto packed = ctx->saved_data["config"].toIntVector();
    Block b{s[0], s[1], s[2], Tensor(), s[3], s[4], s[5], s[6], s[7], s[8], Config::unpack(packed)};
    b.sizes();
    const Kept k{s[9], s[10], s[11], s[12], s[13], s[14], s[15], s[16], s[17], s[18]};
    // needs_input_grad counts the tensors among the arguments: an absent one has no index
    const int gb = 2, w = gb + (b.gate_b.defined() ? 1 : 0) + (packed.back() ? 1 : 0), sh = w + 3;
    auto wants = [&](int i) { return ctx->needs_input_grad(i); };
    const bool shared = b.Fs > 0;
    const Needs need{wants(0), wants(1), b.gate_b.defined() && wants(gb), wants(w) || wants(w + 1) || wants(w + 2),
                     shared && (wants(sh) || wants(sh + 1) || wants(sh + 2))};
    Grads g = block_backward(b, k, grads[0], need);
    auto put = [&](int argument, int tensor, const Tensor& t) {
      if (t.defined() && wants(tensor)) out[argument] = t;
    };
    put(0, 0, g.x);
    put(1, 1, g.gate_w);
    if (need.gate_b) out[2] = g.gate_b;
    put(4, w, g.w1);
    put(5, w + 1, g.w3);
    put(6, w + 2, g.w2);
    if (shared) {
      put(7, sh, g.sg);
      put(8, sh + 1, g.su);
      put(9, sh + 2, g.sd);
    }
    return out;
  }
};

Tensor contiguous(const OptTensor& t) { return t.has_value() && t->defined() ? t->contiguous() : Tensor(); }

std::tuple<Tensor, Tensor> moe_block(const Tensor& x_, const Tensor& gate_w_, const OptTensor& gate_b_,
                                     const OptTensor& expert_b_, const Tensor& w1_, const Tensor& w3_,
                                     const Tensor& w2_, const OptTensor& sg_, const OptTensor& su_,
                                     const OptTensor& sd_, int64_t K, int64_t score_func, bool route_norm,
                                     double route_scale, int64_t num_groups, int64_t num_limited, int64_t lo,
                                     int64_t hi, int64_t align, bool round_terms, bool overlap_shared) {
  const Tensor x = x_.contiguous(), gate_w = gate_w_.contiguous(), w1 = w1_.contiguous(), w3 = w3_.contiguous(),
               w2 = w2_.contiguous();
  const Tensor gate_b = contiguous(gate_b_), expert_b = contiguous(expert_b_), sg = contiguous(sg_),
               su = contiguous(su_), sd = contiguous(sd_);
  TORCH_CHECK_VALUE(x.dim() == 2 && x.size(0) >= 1 && gate_w.dim() == 2 && gate_w.size(1) == x.size(1), "gate weight ",
                    gate_w.sizes(), " does not match input ", x.sizes());
  TORCH_CHECK_VALUE(w1.dim() == 3 && w1.size(2) == x.size(1) && w3.sizes() == w1.sizes() && w2.dim() == 3 &&
                        w2.size(0) == w1.size(0) && w2.size(1) == w1.size(2) && w2.size(2) == w1.size(1),
                    "expert weight shapes do not match (E,F,D)/(E,F,D)/(E,D,F)");
  TORCH_CHECK_VALUE(lo >= 0 && hi - lo == w1.size(0) && hi <= gate_w.size(0) && align >= 1,
                    "local expert range [", lo, ",", hi, ") does not match the weights");
  const auto type = x.scalar_type();
  TORCH_CHECK_TYPE((type == at::kFloat || type == at::kBFloat16) && w1.scalar_type() == type &&
                       w3.scalar_type() == type && w2.scalar_type() == type,
                   "expert weights and rows must share one dtype, float32 or bfloat16");
  TORCH_CHECK_VALUE((!gate_b.defined() || gate_b.numel() == gate_w.size(0)) &&
                        (!expert_b.defined() || expert_b.numel() == gate_w.size(0)),
                    "a bias does not match the number of experts");
  TORCH_CHECK_VALUE(sg.defined() == su.defined() && sg.defined() == sd.defined(), "shared expert: three weights or none");
  if (sg.defined()) {
    TORCH_CHECK_VALUE(sg.dim() == 2 && sg.size(1) == x.size(1) && su.sizes() == sg.sizes() && sd.dim() == 2 &&
                          sd.size(0) == x.size(1) && sd.size(1) == sg.size(0),
                      "shared expert weight shapes do not match (F,D)/(F,D)/(D,F)");
    TORCH_CHECK_TYPE(sg.scalar_type() == type && su.scalar_type() == type && sd.scalar_type() == type,
                     "shared expert weights and tokens must share one dtype");
  }
  for (const Tensor* t : {&gate_w, &gate_b, &expert_b, &w1, &w3, &w2, &sg, &su, &sd})
    TORCH_CHECK(!t->defined() || t->device() == x.device(), "moe_block: tensors on different devices: ", x.device(),
                " and ", t->device());
  const Config c{K, score_func, route_norm, num_groups, num_limited, lo, hi, align, round_terms, overlap_shared, route_scale};
  if (torch::autograd::compute_requires_grad(x, gate_w, gate_b, w1, w3, w2, sg, su, sd)) {
    auto r = MoeBlock::apply(x, gate_w, opt(gate_b), opt(expert_b), w1, w3, w2, opt(sg), opt(su), opt(sd), c);
    return {r[0], r[1]};
  }
  at::AutoDispatchBelowADInplaceOrView below;
  Block b{x, gate_w, gate_b, expert_b, w1, w3, w2, sg, su, sd, c};
  b.sizes();
  Kept k;
  return block_forward(b, false, k);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(mi355_moe, m) {
  m.def(
      "moe_block(Tensor x, Tensor gate_w, Tensor? gate_bias, Tensor? expert_bias, Tensor w1, Tensor w3, Tensor w2, "
      "Tensor? shared_gate, Tensor? shared_up, Tensor? shared_down, int top_k, int score_func, bool route_norm, "
      "float route_scale, int num_groups, int num_limited, int local_lo, int local_hi, int align, bool round_terms, "
      "bool overlap_shared) -> (Tensor, Tensor)");
}
TORCH_LIBRARY_IMPL(mi355_moe, CUDA, m) { m.impl("moe_block", moe_block); }
TORCH_LIBRARY_IMPL(mi355_moe, Autograd, m) { m.impl("moe_block", moe_block); }
