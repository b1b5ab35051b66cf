// The whole MoE block as one operator: router, plan, routed experts, combine and (when there is one)
// the dense shared expert, with one autograd node whose backward is written out below.
//
//   moe_block       what callers use.  Its Autograd kernel passes on to the two below when an input asks for
//                   a gradient, and to its own device kernel otherwise.
//   moe_block_fwd   the forward that also returns what the backward reads
//   moe_block_bwd   the backward
// All three are reached through the dispatcher, also from inside the autograd node: whatever stands in its
// way -- a tracing mode, fake tensors, a function transform -- sees an operator with its inputs and
// outputs and never this file's allocations.
//
// The stage operators of torch_ext.cpp compute the same things one at a time, for callers that
// look between the stages (hooks, other dispatchers, other routers, tracing, dispatch modes); MoE.forward
// comes here when nothing hangs on the stages.  What the single operator saves:
//   * host time: a forward pass is one trip through the dispatcher and about ten C calls instead of four
//     operators, a plan object and its views (83 -> 28 us at one token, launches included), a training step has one
//     autograd node instead of three to five;
//   * launches: the router's partial logits are summed by the selection, selection and plan are one or two
//     launches instead of four, the score gradient's pieces are summed by the selection's backward, and
//     the additions of (T, D) tensors -- shared expert's output, the two or three input gradients -- ride
//     in kernels that hold the other operand anyway.
// Every kernel and every rounding is the stage operators' own: both ways give the same bits, but for the order of
// two sums.  The load-balance loss adds its tokens up in another order, and with a shared expert the input
// gradient is (routed + shared) + gate here, while the autograd engine adds the stages' three as
// (routed + gate) + shared when the shared expert runs on its own stream, as it does by default: as many
// roundings, other bits.
//
// Memory.  From PyTorch's allocator on the current stream: the results one by one, what the backward
// reads in one allocation, a pass's scratch in another.  Work on the
// library's side streams is forked from the current stream and joined before the operator returns, so
// buffers need no record_stream.
#include <torch/csrc/autograd/autograd_not_implemented_fallback.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/library.h>

#include <string>
#include <tuple>
#include <utility>
#include <vector>

#include "torch_common.h"

namespace {

using namespace mi355_torch;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

struct Config {
  int64_t K, score_func, route_norm, num_groups, num_limited, lo, hi, align, round_terms, overlap;
  int64_t aux;  // the router injects a load-balance loss
  double route_scale;
};

// What a router that keeps statistics brings; undefined / zero where it keeps none.  Written in the forward.
struct Stats {
  Tensor histogram, aux_acc, aux_denominator;
  double aux_coeff = 0.0;
  Tensor totals;  // what the counts per expert are added to
};

// The block's tensors; undefined where the block has none.
struct Block {
  Tensor x, gate_w, gate_b, expert_b, w1, w3, w2, sg, su, sd;
  Tensor mask;  // (T) bool, true = padding
  Config c;
  int64_t T, D, E, F, El, N, R, Fs, tile_m, tile_cap, shared_cap;
  int dt, gate_dt;
  int splits;           // partial sums of the router's forward (0: the kernel without them)
  int64_t piece_bytes, kept_bytes;  // its weight pieces: what it needs, what it leaves for the backward
  bool gather;         // the kernels of any width serve the routed part and read the tokens' rows in place
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
    gather = !folded && mi355_grouped_gather_covers(dt, D, F, R, T);
    Fs = sg.defined() ? sg.size(0) : 0;
    shared_cap = Fs > 0 ? (T + tile_m - 1) / tile_m : 0;
    splits = mi355_router_gate_fwd_splits(dt, gate_dt, T, D, E);
    piece_bytes = splits > 0 ? mi355_router_gate_fwd_pieces_bytes(dt, gate_dt, T, D, E) : 0;
    kept_bytes = splits > 0 ? mi355_router_gate_fwd_kept_bytes(dt, gate_dt, T, D, E) : 0;
    shared_folded = Fs > 0 && mi355_grouped_combine_bwd_slots(dt, D, Fs) > 0;
  }
};

// Hands out 256-byte aligned pieces of one allocation.  With a null base it only measures.
struct Carver {
  char* base;
  int64_t at = 0;
  template <typename T>
  T* take(int64_t n) {
    T* p = reinterpret_cast<T*>(base + at);
    at += (n * static_cast<int64_t>(sizeof(T)) + 255) / 256 * 256;
    return base ? p : nullptr;
  }
  void* take(int64_t n, int64_t item) { return take<char>(n * item); }
};

// Runs `layout` twice, to measure and to hand out, around one allocation.
template <typename Layout>
Tensor carve(const Tensor& like, Layout layout) {
  Carver measure{nullptr};
  layout(measure);
  Tensor t = bytes(measure.at, like);
  Carver c{static_cast<char*>(t.data_ptr())};
  layout(c);
  return t;
}

// Elements of the tokens.  Not a sharp line: 28 steps of four routers, 0.5 to 12 Mi elements, together / apart 0.96-1.01.
constexpr int64_t kShortRowSum = 6 << 20;

// A folded backward so small that the host is what takes the time: a second stream's fork and join cost it more than the weight
// gradients gain beside the input gradient.  A training step, us, beside / behind it: 64 experts of 768 x 448 (384 tiles), two each, 100 to 1500 tokens 208 / 149,
// 204 / 155, 208 / 156, 198 / 157, 200 / 160, 204 / 168; 32 of 640 x 640 (288), four each, 300 to 1500 tokens 197 / 140, 199 / 145, 200 / 159, 203 / 166, 204 / 187;
// 48 of 1024 x 512 (384), four each, 208 / 177, 212 / 201, 211 / 192, 215 / 205, 214 / 218; 60 of it (480), three each, 212 / 191, 212 / 215, 214 / 203, 213 / 205, 224 / 224; 64 of it
// (512), six each, 300 to 1500 tokens 211 / 188, 213 / 193, 213 / 202, 219 / 222, 249 / 248; 24 of 1536 x 768 (432), four each, 209 / 174, 209 / 189, 210 / 202, 225 / 225, 269 /
// 282; 128 of 768 x 512 (768) 249 / 257, 254 / 259, 266 / 272.  32 of 1024 x 704 (384), four each, 300 to 2500 tokens 203 / 158,
// 203 / 164, 203 / 180, 208 / 188, 216 / 216, 288 / 292.  The second line lies where the products take as long as the host: 1500 tokens of the 48, 1000 of the 64
// or of the last, 700 of the 24.
bool short_backward(int64_t El, int64_t D, int64_t F, int64_t R) {
  return El * ((D + 255) / 256) * ((F + 255) / 256) <= 512 && R * D * F <= (int64_t{3} << 30);
}

// What the backward reads besides the inputs, in one allocation: the plan's and the router's arrays, the
// activations, the shared expert's plan and activations.
struct Kept {
  int64_t* ids;
  float *weights, *logits, *row_scale, *aux_f = nullptr, *aux_scale = nullptr;
  int32_t *seg_offsets, *seg_counts, *tile_expert, *tile_row0, *num_tiles, *row_of_slot, *slot_of_row, *token_of_row;
  int32_t *s_offsets, *s_counts, *s_expert, *s_row0, *s_num;
  void *pieces = nullptr, *rows = nullptr, *gate = nullptr, *up = nullptr, *h = nullptr, *y = nullptr;
  void *s_gate = nullptr, *s_up = nullptr, *s_h = nullptr;

  // save: someone will run the backward (else only what the forward itself needs is there)
  void layout(Carver& c, const Block& b, bool save) {
    const int64_t item = b.dt == MI355_F32 ? 4 : 2;
    ids = c.take<int64_t>(b.N);
    weights = c.take<float>(b.N);
    logits = c.take<float>(b.T * b.E);
    row_scale = c.take<float>(b.R);
    row_of_slot = c.take<int32_t>(b.N);
    slot_of_row = c.take<int32_t>(b.R);
    token_of_row = c.take<int32_t>(b.R);
    seg_offsets = c.take<int32_t>(b.El + 1);
    seg_counts = c.take<int32_t>(2 * b.El);
    tile_expert = c.take<int32_t>(b.tile_cap);
    tile_row0 = c.take<int32_t>(b.tile_cap);
    num_tiles = c.take<int32_t>(1);
    if (b.c.aux) {
      aux_f = c.take<float>(b.E);
      aux_scale = c.take<float>(1);
    }
    if (const int64_t n = save ? b.kept_bytes : b.piece_bytes) pieces = c.take(n, 1);
    if (save || !b.folded) {  // (gate and up are the other kernels' own intermediates)
      gate = c.take(b.R * b.F, item);
      up = c.take(b.R * b.F, item);
    }
    if (!b.folded) {
      if (!b.gather) rows = c.take(b.R * b.D, item);
      h = c.take(b.R * b.F, item);
      y = c.take(b.R * b.D, item);
    }
    if (b.Fs > 0) layout_shared(c, b, save);
  }
  void layout_shared(Carver& c, const Block& b, bool save) {
    const int64_t item = b.dt == MI355_F32 ? 4 : 2;
    s_offsets = c.take<int32_t>(2);
    s_counts = c.take<int32_t>(2);
    s_expert = c.take<int32_t>(b.shared_cap);
    s_row0 = c.take<int32_t>(b.shared_cap);
    s_num = c.take<int32_t>(1);
    s_h = c.take(b.T * b.Fs, item);
    if (save || !b.shared_folded) {
      s_gate = c.take(b.T * b.Fs, item);
      s_up = c.take(b.T * b.Fs, item);
    }
  }
};

// Forks `side` behind everything `main` holds so far, and back.
struct Fork {
  SideStream* side;
  hipStream_t main;
  bool open = false;
  Fork(SideStream* s, hipStream_t m) : side(s), main(m) {}
  // in front of the call's first launch; behind one
  void enter() { follow(main, side->entry); }
  void start() { follow(main, side->fork); }
  // the side stream waits for everything on `from`, another side stream with a launch of the call
  void follow(hipStream_t from) { follow(from, side->fork); }
  void follow(hipStream_t from, hipEvent_t event) {
    TORCH_CHECK(side->chain(event, from, side->stream), "moe_block: cannot fork to the side stream: ",
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

// beside: on a stream of its own, beside the router and the routed experts
void shared_forward(const Block& b, const Kept& k, void* y, void* stream, bool beside) {
  check(mi355_segments_dense(b.T, b.tile_m, k.s_offsets, k.s_counts, k.s_expert, k.s_row0, k.s_num, b.shared_cap, stream),
        "segments_dense");
  const auto forward = beside ? mi355_grouped_swiglu_fwd_beside : mi355_grouped_swiglu_fwd;
  check(forward(ptr(b.x), nullptr, b.T, ptr(b.sg), ptr(b.su), ptr(b.sd), b.dt, k.s_offsets, k.s_counts, k.s_expert, k.s_row0, k.s_num,
                b.shared_cap, k.s_gate, k.s_up, k.s_h, y, 1, b.D, b.Fs, b.T, stream),
        "shared expert");
}

// The forward of a handful of tokens that nobody differentiates and no statistics hang on, without a plan: (output, counts per
// expert).  Four tokens, all experts here: grouped_few.hip has both sides measured.
bool few_choices(const Block& b, const Stats& st) {
  return b.dt == MI355_BF16 && b.folded && b.splits > 0 && b.piece_bytes == 0 && b.c.align == 1 && !b.mask.defined() && !b.c.aux &&
         !st.histogram.defined() && b.T <= 4 && b.c.lo == 0 && b.c.hi == b.E && mi355_choice_covers(b.T, b.D, b.F, b.E, b.c.K, (int)b.c.num_groups);
}

std::tuple<Tensor, Tensor> choices_forward(const Block& b, const Tensor& totals) {
  Launch L(b.x);
  const Config& c = b.c;
  const auto opts = b.x.options();
  const hipStream_t main = static_cast<hipStream_t>(L.stream);
  Tensor counts = at::empty({b.E}, opts.dtype(at::kInt));
  Tensor out = at::empty({b.T, b.D}, opts);
  Kept k;  // (the shared expert's part)
  float *partial = nullptr, *weights = nullptr;
  int32_t* ids = nullptr;
  void *h = nullptr, *y_shared = nullptr;
  Tensor scratch = carve(b.x, [&](Carver& cv) {
    partial = cv.take<float>(b.splits * b.T * b.E);
    weights = cv.take<float>(b.N);
    ids = cv.take<int32_t>(b.N);
    h = cv.take(b.N * b.F, 2);
    if (b.Fs > 0) {
      y_shared = cv.take(b.T * b.D, 2);
      k.layout_shared(cv, b, false);
    }
  });
  Tensor gate_b, expert_b;
  if (b.gate_b.defined()) gate_b = cf(b.gate_b);
  if (b.expert_b.defined()) expert_b = cf(b.expert_b);
  SideStream* aux = b.Fs > 0 && c.overlap ? side_stream(b.x.device().index(), main, 1) : nullptr;
  Fork shared(aux, main);
  if (aux) {
    shared.enter();
    shared_forward(b, k, y_shared, aux->stream, true);
  }
  check(mi355_router_gate_fwd_partial(ptr(b.x), b.dt, fptr(b.gate_w), fptr(gate_b), partial, nullptr, b.T, b.D, b.E, L.stream),
        "router_gate_fwd");
  check(mi355_choice_gateup_fwd(partial, b.splits, fptr(gate_b), fptr(expert_b), b.T, b.E, c.K, (int)c.score_func,
                                (int)c.route_norm, (float)c.route_scale, (int)c.num_groups, (int)c.num_limited, c.lo, c.hi,
                                ptr(b.x), ptr(b.w1), ptr(b.w3), h, weights, ids, counts.data_ptr<int32_t>(), b.D, b.F, L.stream),
        "choice_gateup_fwd");
  if (b.Fs > 0 && !aux) shared_forward(b, k, y_shared, L.stream, false);
  shared.join();
  if (totals.defined()) totals.add_(counts);
  check(mi355_choice_down_fwd(h, ptr(b.w2), weights, ids, y_shared, ptr(out), b.T, c.K, b.El, b.D, b.F, (int)c.round_terms,
                              L.stream),
        "choice_down_fwd");
  return {out, counts};
}

// (output, counts per expert, what the backward reads)
std::tuple<Tensor, Tensor, Tensor> block_forward(const Block& b, const Stats& st, bool save) {
  Launch L(b.x);
  const Config& c = b.c;
  const auto opts = b.x.options();
  const int64_t item = b.dt == MI355_F32 ? 4 : 2;
  const hipStream_t main = static_cast<hipStream_t>(L.stream);
  Tensor counts = at::empty({b.E}, opts.dtype(at::kInt));
  Tensor out = at::empty({b.T, b.D}, opts);
  Kept k;
  Tensor kept = carve(b.x, [&](Carver& cv) { k.layout(cv, b, save); });
  // scratch of this call
  const int64_t partial_bytes = b.splits > 1 ? b.splits * b.T * b.E * 4
                                : b.splits == 0 ? mi355_router_gate_fwd_workspace_bytes(b.T, b.D, b.E) : 0;
  const int64_t plan_bytes = mi355_route_plan_workspace_bytes(b.T, c.K, b.E);
  const bool stats = b.mask.defined() || c.aux;
  float *scores = nullptr, *cutoff = nullptr;
  void* stats_work = nullptr;
  int32_t* all_counts = nullptr;  // the plan's counts where `counts` leaves the padding out
  void *gate_work = nullptr, *plan_work = nullptr, *y_shared = nullptr, *h = k.h, *y = k.y;
  Tensor scratch = carve(b.x, [&](Carver& cv) {
    if (partial_bytes > 0) gate_work = cv.take(partial_bytes, 1);
    if (plan_bytes > 0) plan_work = cv.take(plan_bytes, 1);
    if (stats) {
      stats_work = cv.take(mi355_route_stats_workspace_bytes(b.T, b.E), 1);
      all_counts = cv.take<int32_t>(b.E);
    }
    if (st.histogram.defined()) {
      scores = cv.take<float>(b.T * b.E);
      cutoff = cv.take<float>(b.T);
    }
    if (b.Fs > 0) y_shared = cv.take(b.T * b.D, item);
    if (b.folded) {
      h = cv.take(b.R * b.F, item);
      y = cv.take(b.R * b.D, item);
    }
  });
  Tensor gate_b, expert_b;
  if (b.gate_b.defined()) gate_b = cf(b.gate_b);
  if (b.expert_b.defined()) expert_b = cf(b.expert_b);

  // shared expert: beside the router and the routed experts when it may, else right before the sum
  SideStream* aux = b.Fs > 0 && c.overlap ? side_stream(b.x.device().index(), main, 1) : nullptr;
  Fork shared(aux, main);
  if (aux) {
    shared.enter();
    shared_forward(b, k, y_shared, aux->stream, true);
  }

  // router: partial logits, then selection and plan; few experts in one launch less
  float* partial = b.splits > 1 ? static_cast<float*>(gate_work) : k.logits;
  const bool one_launch = mi355_route_gate_plan_covers(b.dt, b.gate_dt, b.T, b.D, b.E, c.K, (int)c.num_groups);
  if (one_launch) {
    // (in front of the selection, below)
  } else if (b.splits > 0) {
    check((save ? mi355_router_gate_fwd_keeping : mi355_router_gate_fwd_partial)(ptr(b.x), b.dt, fptr(b.gate_w), fptr(gate_b), partial,
                                                                                 k.pieces, b.T, b.D, b.E, L.stream),
          "router_gate_fwd");
  } else {
    check(mi355_router_gate_fwd(ptr(b.x), b.dt, ptr(b.gate_w), b.gate_dt, fptr(gate_b), k.logits, gate_work, b.T, b.D,
                                b.E, L.stream),
          "router_gate_fwd");
  }
  const uint8_t* padding = static_cast<const uint8_t*>(ptr(b.mask));
  // what both forms take behind the logits
  auto plan = [&](auto f, auto... logits) {
    return f(logits..., fptr(expert_b), b.T, b.E, c.K, (int)c.score_func, (int)c.route_norm, (float)c.route_scale,
             (int)c.num_groups, (int)c.num_limited, k.weights, k.ids, c.lo, c.hi, c.align, b.tile_m,
             stats ? all_counts : counts.data_ptr<int32_t>(), k.seg_offsets, k.seg_counts, k.row_of_slot, k.slot_of_row,
             k.token_of_row, save && (b.folded || b.gather) ? k.row_scale : nullptr, b.R, k.tile_expert, k.tile_row0,
             k.num_tiles, b.tile_cap, plan_work, padding, stats ? counts.data_ptr<int32_t>() : nullptr, scores, cutoff, k.aux_f,
             k.aux_scale, ptr(st.aux_acc), st.aux_acc.defined() ? dtype_code(st.aux_acc) : MI355_F32,
             fptr(st.aux_denominator), (float)st.aux_coeff);
  };
  int64_t* histogram = st.histogram.defined() ? st.histogram.data_ptr<int64_t>() : nullptr;
  const int64_t bins = histogram ? st.histogram.size(1) : 1;
  auto with_gate = [&](auto... a) { return mi355_route_gate_plan_stats(a..., stats_work, L.stream); };
  auto of_logits = [&](auto... a) { return mi355_route_plan_observe(a..., stats_work, histogram, bins, L.stream); };
  check(one_launch ? plan(with_gate, ptr(b.x), b.dt, fptr(b.gate_w), b.D, fptr(gate_b),
                          save ? k.logits : nullptr)
                   : plan(of_logits, partial, b.splits > 1 ? b.splits : 1, fptr(gate_b),
                          save && b.splits > 1 ? k.logits : nullptr),
        "route_plan");
  if (histogram && one_launch)
    check(mi355_quantile_observe(scores, cutoff, fptr(expert_b), padding, histogram, b.T, b.E, bins, L.stream), "quantile_observe");

  // routed experts
  if (!b.folded && !b.gather)
    check(mi355_permute_rows_fwd(ptr(b.x), b.dt, k.row_of_slot, c.align > 1 ? k.slot_of_row : nullptr,
                                 k.seg_offsets + b.El, k.rows, b.T, b.D, c.K, b.R, L.stream),
          "permute_rows_fwd");
  if (b.gather)
    check(mi355_grouped_gather_fwd(ptr(b.x), k.token_of_row, b.T, ptr(b.w1), ptr(b.w3), ptr(b.w2), b.dt, k.seg_offsets,
                                   k.seg_counts, k.tile_expert, k.tile_row0, k.num_tiles, b.tile_cap, k.gate, k.up, h, y, b.El,
                                   b.D, b.F, b.R, L.stream),
          "grouped_gather_fwd");
  else
    check(mi355_grouped_swiglu_fwd_expecting(b.folded ? ptr(b.x) : k.rows, b.folded ? k.token_of_row : nullptr, b.folded ? b.T : b.R,
                                             ptr(b.w1), ptr(b.w3), ptr(b.w2), b.dt, k.seg_offsets, k.seg_counts, k.tile_expert,
                                             k.tile_row0, k.num_tiles, b.tile_cap, k.gate, k.up, h, y, b.El, b.D, b.F, b.R, b.N,
                                             L.stream),
          "grouped_swiglu_fwd");
  if (b.Fs > 0 && !aux) shared_forward(b, k, y_shared, L.stream, false);
  shared.join();
  check(mi355_combine_count_fwd(y, b.dt, k.weights, k.row_of_slot, y_shared, ptr(out), b.T, b.D, c.K, (int)c.round_terms,
                                iptr(counts), st.totals.defined() ? st.totals.data_ptr<float>() : nullptr, b.E, L.stream),
        "combine_fwd");
  return {out, counts, kept};
}

struct Needs {
  bool x, gate_w, gate_b, experts, shared;
};
struct Grads {
  Tensor x, gate_w, gate_b, w1, w3, w2, sg, su, sd;
};

Grads block_backward(const Block& b, const Tensor& kept, const Tensor& dout_, const Needs& need) {
  Launch L(b.x);
  const Config& c = b.c;
  const auto opts = b.x.options();
  const int64_t item = b.dt == MI355_F32 ? 4 : 2;
  const hipStream_t main = static_cast<hipStream_t>(L.stream);
  const Tensor dout = dense(dout_.scalar_type() == b.x.scalar_type() ? dout_ : dout_.to(b.x.scalar_type()));
  Kept k;
  Carver held{static_cast<char*>(kept.data_ptr())};
  k.layout(held, b, true);
  const int device = b.x.device().index();
  const bool gate = need.gate_w || need.gate_b, routed = need.x || gate || need.experts, logits = need.x || gate;
  const bool run_shared = b.Fs > 0 && (need.x || need.shared);

  Grads g;
  auto like = [](Tensor& out, const Tensor& t) { out = at::empty(t.sizes(), t.options()); };
  if (need.x) like(g.x, b.x);
  if (need.gate_w) like(g.gate_w, b.gate_w);
  if (need.experts) {
    like(g.w1, b.w1);
    like(g.w3, b.w3);
    like(g.w2, b.w2);
  }
  if (need.shared) {
    like(g.sg, b.sg);
    like(g.su, b.su);
    like(g.sd, b.sd);
  }
  const int64_t slots = b.folded ? mi355_grouped_combine_bwd_slots(b.dt, b.D, b.F) : 0;
  // the gate's weight gradient in slices beside the experts' dH, its input gradient together with the row sum
  const bool joined = b.gather && mi355_router_gate_rows_bwd_covers(b.dt, b.gate_dt, b.D, b.E);
  // ... or, behind the matrix-core kernels, both gradients and the row sum together, where they are short: beside the experts'
  // weight gradients, whose workgroups keep to their tiles and their CUs, a long launch holds back whichever of those its own CUs
  // were due to (router_gemm.hip has both sides).  Up to 32 experts that is where nothing runs beside (a step, us, apart / together: 1000
  // tokens of 16, 32 experts of 1024 x 512, four each, 159 / 154, 178 / 170; 2500 of 32 of 1536 x 768, four each, 438 / 447).
  const bool short_sum = b.E > 32 ? b.T * b.D <= kShortRowSum : short_backward(b.El, b.D, b.F, b.R);
  const bool summed = b.folded && need.x && short_sum && mi355_router_gate_sum_bwd_covers(b.dt, b.gate_dt, b.D, b.E, c.K);
  const bool joined_dw = joined && need.gate_w && (need.x || need.experts);
  const int64_t gate_bytes = need.x || need.gate_w ? mi355_router_gate_bwd_workspace_bytes(b.T, b.D, b.E) : 0;
  void *s_dgate = nullptr, *s_dup = nullptr, *dx_shared = nullptr, *dx_routed = nullptr, *dgate = nullptr, *dup = nullptr,
       *drows = nullptr, *hs = nullptr, *dy = nullptr, *gate_work = nullptr;
  float *dots = nullptr, *dlogits = nullptr;  // dots: pieces (R, slots), or whole (T, K)
  Tensor dlogits_t;
  if (need.gate_b) dlogits_t = at::empty({b.T, b.E}, opts.dtype(at::kFloat));
  Tensor scratch = carve(b.x, [&](Carver& cv) {
    if (run_shared) {
      s_dgate = cv.take(b.T * b.Fs, item);
      s_dup = cv.take(b.T * b.Fs, item);
      if (need.x) dx_shared = cv.take(b.T * b.D, item);
    }
    if (!routed) return;
    if (need.x) {
      if (!joined && !summed) dx_routed = cv.take(b.T * b.D, item);
      drows = cv.take(b.R * b.D, item);
    }
    dgate = cv.take(b.R * b.F, item);
    dup = cv.take(b.R * b.F, item);
    if (b.folded) {
      hs = cv.take(b.R * b.F, item);
      dots = cv.take<float>(b.R * slots);
    } else if (!b.gather) {
      dy = cv.take(b.R * b.D, item);
      dots = cv.take<float>(b.N);
    }
    if (logits) dlogits = need.gate_b ? dlogits_t.data_ptr<float>() : cv.take<float>(b.T * b.E);
    if (gate_bytes > 0) gate_work = cv.take(gate_bytes, 1);
  });

  // ---- shared expert: dH and dX beside the routed part where they may be, its weight gradients in front
  // of the routed ones on the stream those use
  SideStream* aux = run_shared && c.overlap && routed ? side_stream(device, main, 1) : nullptr;
  const bool beside = b.folded && need.experts && (aux || !short_backward(b.El, b.D, b.F, b.R));
  SideStream* side = routed && need.x && (beside || (b.shared_folded && aux && need.shared)) ? side_stream(device, main, 0) : nullptr;
  Fork shared(aux, main), weights(side, main);
  if (run_shared) {
    if (aux) shared.enter();
    void* stream = aux ? static_cast<void*>(aux->stream) : L.stream;
    if (b.shared_folded) {
      auto stage = [&](int s, void* on) {
        check(mi355_grouped_swiglu_stage(s, ptr(dout), ptr(b.x), nullptr, b.T, ptr(b.sg), ptr(b.su), ptr(b.sd), k.s_gate,
                                         k.s_up, k.s_h, nullptr, k.s_offsets, k.s_counts, k.s_expert, k.s_row0, k.s_num,
                                         b.shared_cap, s_dgate, s_dup, dx_shared, ptr(g.sg), ptr(g.su), ptr(g.sd), 1,
                                         b.D, b.Fs, b.T, on),
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
      check(mi355_grouped_swiglu_bwd(ptr(dout), ptr(b.x), nullptr, b.T, ptr(b.sg), ptr(b.su), ptr(b.sd), k.s_gate, k.s_up,
                                     k.s_h, b.dt, k.s_offsets, k.s_counts, k.s_expert, k.s_row0, k.s_num, b.shared_cap,
                                     s_dgate, s_dup, dx_shared, ptr(g.sg), ptr(g.su), ptr(g.sd), 1, b.D, b.Fs, b.T, stream),
            "shared expert backward");
    }
  }
  if (!routed) return g;

  // ---- routed experts: dx_routed is the sum over a token's rows plus the shared expert's part
  auto row_sum = [&]() {
    if (!need.x) return;
    shared.join();
    check(mi355_permute_rows_add_bwd(drows, b.dt, k.row_of_slot, dx_shared, dx_routed, b.T, b.D, c.K, L.stream),
          "permute_rows_bwd");
  };
  auto select = [&]() {
    check(mi355_router_select_dots_bwd(k.logits, k.ids, dots, slots, k.row_of_slot, b.R, k.aux_f, k.aux_scale,
                                       static_cast<const uint8_t*>(ptr(b.mask)), dlogits, b.T, b.E, c.K,
                                       (int)c.score_func, (int)c.route_norm, (float)c.route_scale, L.stream),
          "router_select_bwd");
  };
  if (b.folded) {
    auto run = [&](int stages, void* stream) {
      check(mi355_grouped_swiglu_combine_bwd(ptr(dout), ptr(b.x), k.token_of_row, b.T, k.row_scale, ptr(b.w1), ptr(b.w3),
                                             ptr(b.w2), k.gate, k.up, b.dt, k.seg_offsets, k.seg_counts, k.tile_expert,
                                             k.tile_row0, k.num_tiles, b.tile_cap, dgate, dup, hs, dots, drows, ptr(g.w1),
                                             ptr(g.w3), ptr(g.w2), b.El, b.D, b.F, b.R, stages, stream),
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
    if (!summed) row_sum();
    if (logits) select();
    if (need.experts && !side) run(kWeights, L.stream);
  } else if (b.gather) {
    const bool experts = need.x || need.experts;
    auto rows = [&](auto f, auto... route) {
      check(f(ptr(dout), ptr(b.x), k.token_of_row, b.T, k.row_scale, ptr(b.w1), ptr(b.w3), ptr(b.w2), k.gate, k.up, k.h, b.dt,
              k.seg_offsets, k.seg_counts, k.tile_expert, k.tile_row0, k.num_tiles, b.tile_cap, dgate, dup, drows, ptr(g.w1),
              ptr(g.w3), ptr(g.w2), route..., b.El, b.D, b.F, b.R, L.stream),
            "grouped_gather_bwd");
    };
    const uint8_t* padding = static_cast<const uint8_t*>(ptr(b.mask));
    float* gate_partial = joined_dw ? static_cast<float*>(gate_work) : nullptr;
    if (logits && experts && b.E <= 64) {
      rows(mi355_grouped_gather_route_bwd, k.logits, k.ids, k.y, k.row_of_slot, k.aux_f, k.aux_scale, padding, dlogits, gate_partial,
           b.E, c.K, (int)c.score_func, (int)c.route_norm, (float)c.route_scale);
    } else {
      if (logits)
        check(mi355_router_select_rows_bwd(k.logits, k.ids, ptr(dout), k.y, b.dt, k.row_of_slot, b.R, b.D, k.aux_f, k.aux_scale,
                                           padding, dlogits, b.T, b.E, c.K, (int)c.score_func, (int)c.route_norm,
                                           (float)c.route_scale, L.stream),
              "router_select_rows_bwd");
      if (experts) rows(mi355_grouped_gather_bwd, joined_dw ? dlogits : nullptr, gate_partial, b.E);
    }
    if (!joined) row_sum();
  } else {
    const int32_t* pad = c.align > 1 ? k.slot_of_row : nullptr;
    check(mi355_combine_bwd(ptr(dout), k.y, b.dt, k.weights, k.row_of_slot, pad, k.seg_offsets + b.El, dy, dots, b.T, b.D,
                            c.K, b.R, L.stream),
          "combine_bwd");
    if (need.x || need.experts)
      check(mi355_grouped_swiglu_bwd(dy, k.rows, nullptr, b.R, ptr(b.w1), ptr(b.w3), ptr(b.w2), k.gate, k.up, k.h, b.dt,
                                     k.seg_offsets, k.seg_counts, k.tile_expert, k.tile_row0, k.num_tiles, b.tile_cap,
                                     dgate, dup, drows, ptr(g.w1), ptr(g.w3), ptr(g.w2), b.El, b.D, b.F, b.R, L.stream),
            "grouped_swiglu_bwd");
    row_sum();
    if (logits) select();
  }

  // ---- router gate; the input gradient is complete with its part
  if (summed) {
    shared.join();
    check(mi355_router_gate_sum_bwd(dlogits, ptr(b.x), b.dt, fptr(b.gate_w), k.pieces, drows, k.row_of_slot, b.R, c.K, dx_shared,
                                    ptr(g.x), need.gate_w ? g.gate_w.data_ptr<float>() : nullptr, gate_work, b.T, b.D, b.E,
                                    L.stream),
          "router_gate_sum_bwd");
  } else if (joined && need.x) {
    shared.join();
    check(mi355_router_gate_rows_bwd(dlogits, b.dt, fptr(b.gate_w), drows, k.row_of_slot, b.R, c.K, dx_shared, ptr(g.x),
                                     static_cast<const float*>(gate_work), joined_dw ? g.gate_w.data_ptr<float>() : nullptr,
                                     b.T, b.D, b.E, L.stream),
          "router_gate_rows_bwd");
  } else if (joined_dw) {
    check(mi355_router_gate_rows_bwd(nullptr, b.dt, nullptr, nullptr, nullptr, b.R, c.K, nullptr, nullptr,
                                     static_cast<const float*>(gate_work), g.gate_w.data_ptr<float>(), b.T, b.D, b.E,
                                     L.stream),
          "router_gate_rows_bwd");
  } else if (need.x || need.gate_w) {
    check(mi355_router_gate_add_bwd(dlogits, ptr(b.x), b.dt, ptr(b.gate_w), b.gate_dt, k.pieces, dx_routed, ptr(g.x),
                                    ptr(g.gate_w), gate_work, b.T, b.D, b.E, L.stream),
          "router_gate_bwd");
  }
  if (need.gate_b) g.gate_b = dlogits_t.sum(0).to(b.gate_b.scalar_type());
  weights.join();
  shared.join();
  return g;
}

Tensor some(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : std::nullopt; }

// The arguments of moe_block and moe_block_fwd, once as parameters and once to pass on.
#define BLOCK_PARAMS                                                                                               \
  const Tensor &x, const Tensor &gate_w, const OptTensor &gate_b, const OptTensor &expert_b, const Tensor &w1,     \
      const Tensor &w3, const Tensor &w2, const OptTensor &sg, const OptTensor &su, const OptTensor &sd, int64_t K, \
      int64_t score_func, bool route_norm, double route_scale, int64_t num_groups, int64_t num_limited, int64_t lo, \
      int64_t hi, int64_t align, bool round_terms, bool overlap_shared, const OptTensor &mask,                     \
      const OptTensor &histogram, const OptTensor &aux_denominator, double aux_coeff, const OptTensor &aux_acc,    \
      const OptTensor &totals
#define BLOCK_ARGS                                                                                                 \
  x, gate_w, gate_b, expert_b, w1, w3, w2, sg, su, sd, K, score_func, route_norm, route_scale, num_groups,         \
      num_limited, lo, hi, align, round_terms, overlap_shared, mask, histogram, aux_denominator, aux_coeff, aux_acc, totals

using BlockSig = std::tuple<Tensor, Tensor>(BLOCK_PARAMS);
using BlockFwdSig = std::tuple<Tensor, Tensor, Tensor>(BLOCK_PARAMS);
using NineTensors = std::tuple<Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor>;
using BlockBwdSig = NineTensors(const Tensor&, const Tensor&, const Tensor&, const OptTensor&, const Tensor&,
                                const Tensor&, const Tensor&, const OptTensor&, const OptTensor&, const OptTensor&,
                                const Tensor&, const OptTensor&, int64_t, int64_t, bool, double, int64_t, int64_t,
                                int64_t, bool, bool, bool, bool, bool, bool, bool);

// The statistics are written through their pointers: what autograd compares before it uses a saved tensor is raised as an operator of torch's own
// does.  (By whichever kernel is in front: one more hop of 27 arguments shows in a forward of 70 us.)
void statistics_written(const OptTensor& histogram, const OptTensor& aux_acc, const OptTensor& totals) {
  for (const OptTensor* t : {&histogram, &aux_acc, &totals}) wrote(*t);
}

struct MoeBlock : public torch::autograd::Function<MoeBlock> {
  static variable_list forward(AutogradContext* ctx, BLOCK_PARAMS) {
    at::AutoDispatchBelowADInplaceOrView below;
    static auto op = typed_op<BlockFwdSig>("mi355_moe::moe_block_fwd");
    auto [out, counts, kept] = op.call(BLOCK_ARGS);
    statistics_written(histogram, aux_acc, totals);
    ctx->save_for_backward({x, gate_w, some(gate_b), w1, w3, w2, some(sg), some(su), some(sd), kept, some(mask)});
    ctx->saved_data["config"] = std::vector<int64_t>{K, score_func, route_norm, lo, hi, align, overlap_shared,
                                                     some(aux_denominator).defined(), some(expert_b).defined()};
    ctx->saved_data["route_scale"] = route_scale;
    ctx->set_materialize_grads(false);
    ctx->mark_non_differentiable({counts});
    return {out, counts};
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    variable_list out(27);
    if (!grads[0].defined()) return out;
    const auto s = ctx->get_saved_variables();
    const auto c = ctx->saved_data["config"].toIntVector();
    // needs_input_grad counts the tensors among the arguments: an absent one has no index
    const int gb = 2, w = gb + (s[2].defined() ? 1 : 0) + (c.back() ? 1 : 0), sh = w + 3;
    auto wants = [&](int i) { return ctx->needs_input_grad(i); };
    const bool shared = s[6].defined();
    // A pass that is itself differentiated (create_graph) leaves the gradients with a node that raises: there
    // is no derivative of the backward, and without one a gradient penalty would leave the block out unnoticed.
    std::optional<at::AutoDispatchBelowADInplaceOrView> below;
    if (!at::GradMode::is_enabled()) below.emplace();
    static auto op = typed_op<BlockBwdSig>("mi355_moe::moe_block_bwd");
    auto [dx, dgate_w, dgate_b, dw1, dw3, dw2, dsg, dsu, dsd] =
        op.call(grads[0], s[0], s[1], opt(s[2]), s[3], s[4], s[5], opt(s[6]), opt(s[7]), opt(s[8]), s[9], opt(s[10]), c[0],
                c[1], c[2] != 0, ctx->saved_data["route_scale"].toDouble(), c[3], c[4], c[5], c[6] != 0, c[7] != 0,
                wants(0), wants(1), s[2].defined() && wants(gb), wants(w) || wants(w + 1) || wants(w + 2),
                shared && (wants(sh) || wants(sh + 1) || wants(sh + 2)));
    auto put = [&](int argument, int tensor, const Tensor& t) {
      if (t.defined() && wants(tensor)) out[argument] = t;
    };
    put(0, 0, dx);
    put(1, 1, dgate_w);
    out[2] = dgate_b;  // (undefined unless it was asked for)
    put(4, w, dw1);
    put(5, w + 1, dw3);
    put(6, w + 2, dw2);
    if (shared) {
      put(7, sh, dsg);
      put(8, sh + 1, dsu);
      put(9, sh + 2, dsd);
    }
    return out;
  }
};

void check_weights(const Block& b) {
  const Tensor &x = b.x, &w1 = b.w1, &w2 = b.w2;
  TORCH_CHECK_VALUE(x.dim() == 2 && x.size(0) >= 1 && b.gate_w.dim() == 2 && b.gate_w.size(1) == x.size(1), "gate weight ",
                    b.gate_w.sizes(), " does not match input ", x.sizes());
  TORCH_CHECK_VALUE(w1.dim() == 3 && w1.size(2) == x.size(1) && b.w3.sizes() == w1.sizes() && w2.dim() == 3 &&
                        w2.size(0) == w1.size(0) && w2.size(1) == w1.size(2) && w2.size(2) == w1.size(1),
                    "expert weight shapes do not match (E,F,D)/(E,F,D)/(E,D,F)");
  TORCH_CHECK_VALUE(b.c.lo >= 0 && b.c.hi - b.c.lo == w1.size(0) && b.c.hi <= b.gate_w.size(0) && b.c.align >= 1,
                    "local expert range [", b.c.lo, ",", b.c.hi, ") does not match the weights");
  const auto type = x.scalar_type();
  TORCH_CHECK_TYPE((type == at::kFloat || type == at::kBFloat16) && w1.scalar_type() == type &&
                       b.w3.scalar_type() == type && w2.scalar_type() == type,
                   "expert weights and rows must share one dtype, float32 or bfloat16");
  TORCH_CHECK_VALUE((!b.gate_b.defined() || b.gate_b.numel() == b.gate_w.size(0)) &&
                        (!b.expert_b.defined() || b.expert_b.numel() == b.gate_w.size(0)),
                    "a bias does not match the number of experts");
  const Tensor &sg = b.sg, &su = b.su, &sd = b.sd;
  TORCH_CHECK_VALUE(sg.defined() == su.defined() && sg.defined() == sd.defined(), "shared expert: three weights or none");
  if (sg.defined()) {
    TORCH_CHECK_VALUE(sg.dim() == 2 && sg.size(1) == x.size(1) && su.sizes() == sg.sizes() && sd.dim() == 2 &&
                          sd.size(0) == x.size(1) && sd.size(1) == sg.size(0),
                      "shared expert weight shapes do not match (F,D)/(F,D)/(D,F)");
    TORCH_CHECK_TYPE(sg.scalar_type() == type && su.scalar_type() == type && sd.scalar_type() == type,
                     "shared expert weights and tokens must share one dtype");
  }
  for (const Tensor* t : {&b.gate_w, &b.gate_b, &b.expert_b, &b.w1, &b.w3, &b.w2, &sg, &su, &sd})
    TORCH_CHECK(!t->defined() || t->device() == x.device(), "moe_block: tensors on different devices: ", x.device(),
                " and ", t->device());
  TORCH_CHECK_VALUE(!b.mask.defined() || (b.mask.scalar_type() == at::kBool && b.mask.numel() == x.size(0) &&
                                          b.mask.device() == x.device()),
                    "padding mask: one bool per token on the tokens' device");
}

void check_stats(const Block& b, const Stats& st) {
  TORCH_CHECK_VALUE(!st.histogram.defined() ||
                        (st.histogram.scalar_type() == at::kLong && st.histogram.is_contiguous() &&
                         st.histogram.dim() == 2 && st.histogram.size(0) == b.gate_w.size(0) &&
                         st.histogram.device() == b.x.device() && b.expert_b.defined()),
                    "histogram: contiguous int64 (experts, bins) beside an expert bias");
  TORCH_CHECK_VALUE(!st.totals.defined() || (st.totals.scalar_type() == at::kFloat && st.totals.is_contiguous() &&
                                             st.totals.numel() == b.gate_w.size(0) && st.totals.device() == b.x.device()),
                    "totals: contiguous fp32, one per expert");
  auto scalar = [&](const Tensor& t) { return !t.defined() || (t.numel() == 1 && t.device() == b.x.device()); };
  TORCH_CHECK_VALUE(scalar(st.aux_acc) && scalar(st.aux_denominator) &&
                        (!st.aux_denominator.defined() || st.aux_denominator.scalar_type() == at::kFloat) &&
                        (!st.aux_acc.defined() || st.aux_acc.scalar_type() == at::kFloat ||
                         st.aux_acc.scalar_type() == at::kBFloat16),
                    "auxiliary loss: scalars on the tokens' device, the denominator fp32, the metric fp32 or bf16");
}

// The block of a forward call, checked.
std::pair<Block, Stats> block_of(BLOCK_PARAMS) {
  const Stats st{some(histogram), some(aux_acc), some(aux_denominator), aux_coeff, some(totals)};
  Block b{dense(x), dense(gate_w), dense(gate_b), dense(expert_b), dense(w1), dense(w3), dense(w2), dense(sg), dense(su),
          dense(sd), dense(mask),
          Config{K, score_func, route_norm, num_groups, num_limited, lo, hi, align, round_terms, overlap_shared,
                 st.aux_denominator.defined(), route_scale}};
  check_weights(b);
  check_stats(b, st);
  b.sizes();
  return {b, st};
}

std::tuple<Tensor, Tensor> moe_block(BLOCK_PARAMS) {
  const auto [b, st] = block_of(BLOCK_ARGS);
  if (few_choices(b, st)) return choices_forward(b, st.totals);
  auto [out, counts, kept] = block_forward(b, st, false);
  return {out, counts};
}

std::tuple<Tensor, Tensor, Tensor> moe_block_fwd(BLOCK_PARAMS) {
  const auto [b, st] = block_of(BLOCK_ARGS);
  return block_forward(b, st, true);
}

// shapes only (fake and meta tensors)
std::tuple<Tensor, Tensor, Tensor> moe_block_fwd_meta(BLOCK_PARAMS) {
  const auto [b, st] = block_of(BLOCK_ARGS);
  Carver measure{nullptr};
  Kept{}.layout(measure, b, true);
  return {at::empty({b.T, b.D}, b.x.options()), at::empty({b.E}, b.x.options().dtype(at::kInt)), bytes(measure.at, b.x)};
}

#define BLOCK_BWD_PARAMS                                                                                              \
  const Tensor &dout, const Tensor &x, const Tensor &gate_w, const OptTensor &gate_b, const Tensor &w1,               \
      const Tensor &w3, const Tensor &w2, const OptTensor &sg, const OptTensor &su, const OptTensor &sd,              \
      const Tensor &kept, const OptTensor &mask, int64_t K, int64_t score_func, bool route_norm, double route_scale,  \
      int64_t lo, int64_t hi, int64_t align, bool overlap_shared, bool aux, bool need_x, bool need_gate_w,            \
      bool need_gate_b, bool need_experts, bool need_shared
#define BLOCK_BWD_ARGS                                                                                                \
  dout, x, gate_w, gate_b, w1, w3, w2, sg, su, sd, kept, mask, K, score_func, route_norm, route_scale, lo, hi, align, \
      overlap_shared, aux, need_x, need_gate_w, need_gate_b, need_experts, need_shared

// The block and what is asked of a backward call, checked.
std::pair<Block, Needs> block_bwd_of(BLOCK_BWD_PARAMS) {
  Block b{dense(x), dense(gate_w), dense(gate_b), Tensor(), dense(w1), dense(w3), dense(w2), dense(sg), dense(su), dense(sd),
          dense(mask),
          Config{K, score_func, route_norm, 0, 0, lo, hi, align, 0, overlap_shared, aux, route_scale}};
  check_weights(b);
  b.sizes();
  Carver measure{nullptr};
  Kept{}.layout(measure, b, true);
  TORCH_CHECK_VALUE(kept.scalar_type() == at::kByte && kept.is_contiguous() && kept.numel() >= measure.at &&
                        kept.device() == b.x.device(),
                    "moe_block_bwd: not what moe_block_fwd kept for this block");
  TORCH_CHECK_VALUE(dout.sizes() == b.x.sizes() && dout.device() == b.x.device(), "moe_block_bwd: gradient ", dout.sizes(),
                    " does not match the output ", b.x.sizes());
  return {b, Needs{need_x, need_gate_w, need_gate_b && b.gate_b.defined(), need_experts, need_shared && b.Fs > 0}};
}

NineTensors moe_block_bwd(BLOCK_BWD_PARAMS) {
  const auto [b, need] = block_bwd_of(BLOCK_BWD_ARGS);
  Grads g = block_backward(b, dense(kept), dout, need);  // (a saved-tensor hook may hand back a view)
  return {g.x, g.gate_w, g.gate_b, g.w1, g.w3, g.w2, g.sg, g.su, g.sd};
}

NineTensors moe_block_bwd_meta(BLOCK_BWD_PARAMS) {
  const auto [b, need] = block_bwd_of(BLOCK_BWD_ARGS);
  auto like = [](bool wanted, const Tensor& t) { return wanted ? at::empty(t.sizes(), t.options()) : Tensor(); };
  return {like(need.x, b.x),           like(need.gate_w, b.gate_w), like(need.gate_b, b.gate_b),
          like(need.experts, b.w1),    like(need.experts, b.w3),    like(need.experts, b.w2),
          like(need.shared, b.sg),     like(need.shared, b.su),     like(need.shared, b.sd)};
}

// Where no Autograd kernel is in front (inference mode, a caller below it), the versions are raised here.
template <typename Sig>
auto writing(const char* name, BLOCK_PARAMS) {
  static auto op = typed_op<Sig>(name);
  at::AutoDispatchBelowADInplaceOrView below;
  auto r = op.call(BLOCK_ARGS);
  statistics_written(histogram, aux_acc, totals);
  return r;
}
std::tuple<Tensor, Tensor> moe_block_writing(BLOCK_PARAMS) { return writing<BlockSig>("mi355_moe::moe_block", BLOCK_ARGS); }
std::tuple<Tensor, Tensor, Tensor> moe_block_fwd_writing(BLOCK_PARAMS) {
  return writing<BlockFwdSig>("mi355_moe::moe_block_fwd", BLOCK_ARGS);
}

std::tuple<Tensor, Tensor> moe_block_autograd(BLOCK_PARAMS) {
  if (torch::autograd::compute_requires_grad(x, gate_w, gate_b, w1, w3, w2, sg, su, sd)) {
    auto r = MoeBlock::apply(BLOCK_ARGS);
    return {r[0], r[1]};
  }
  return writing<BlockSig>("mi355_moe::moe_block", BLOCK_ARGS);
}

}  // namespace

TORCH_LIBRARY_FRAGMENT(mi355_moe, m) {
  const std::string args =
      "(Tensor x, Tensor gate_w, Tensor? gate_bias, Tensor? expert_bias, Tensor w1, Tensor w3, Tensor w2, "
      "Tensor? shared_gate, Tensor? shared_up, Tensor? shared_down, int top_k, int score_func, bool route_norm, "
      "float route_scale, int num_groups, int num_limited, int local_lo, int local_hi, int align, bool round_terms, "
      "bool overlap_shared, Tensor? padding_mask, Tensor(a!)? histogram, Tensor? aux_denominator, float aux_coeff, "
      "Tensor(b!)? aux_acc, Tensor(c!)? totals=None)";
  m.def(("moe_block" + args + " -> (Tensor, Tensor)").c_str());
  m.def(("moe_block_fwd" + args + " -> (Tensor, Tensor, Tensor)").c_str());
  // a gradient that is not asked for is undefined (None)
  m.def(
      "moe_block_bwd(Tensor dout, Tensor x, Tensor gate_w, Tensor? gate_bias, Tensor w1, Tensor w3, Tensor w2, "
      "Tensor? shared_gate, Tensor? shared_up, Tensor? shared_down, Tensor kept, Tensor? padding_mask, int top_k, "
      "int score_func, bool route_norm, float route_scale, int local_lo, int local_hi, int align, bool overlap_shared, "
      "bool aux, bool need_x, bool need_gate_w, bool need_gate_bias, bool need_experts, bool need_shared) -> "
      "(Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor, Tensor)");
}
TORCH_LIBRARY_IMPL(mi355_moe, CUDA, m) {
  m.impl("moe_block", moe_block);
  m.impl("moe_block_fwd", moe_block_fwd);
  m.impl("moe_block_bwd", moe_block_bwd);
}
TORCH_LIBRARY_IMPL(mi355_moe, Meta, m) {
  m.impl("moe_block_fwd", moe_block_fwd_meta);
  m.impl("moe_block_bwd", moe_block_bwd_meta);
}
TORCH_LIBRARY_IMPL(mi355_moe, ADInplaceOrView, m) {
  m.impl("moe_block", moe_block_writing);
  m.impl("moe_block_fwd", moe_block_fwd_writing);
}
TORCH_LIBRARY_IMPL(mi355_moe, Autograd, m) {
  m.impl("moe_block", moe_block_autograd);
  m.impl("moe_block_bwd", torch::autograd::autogradNotImplementedFallback());
}
