// Grouped products of any width that is a multiple of four, fp32 and bf16 (grouped_any.hip).
#pragma once
#include "common.h"

namespace mi355 {

struct AnySeg {
  const int32_t *seg_offsets, *seg_counts, *tile_expert, *tile_row0, *num_tiles;
  int64_t tile_capacity, El;
};
// The tokens' rows in place of copies in row order: row r of x (rows) or, scaled by row_scale[r], of the output gradient (dy) is
// row token_of_row[r] of a matrix of `tokens` rows.
struct AnyFold {
  const int32_t* token_of_row;
  int64_t tokens;
  const float* row_scale;  // (backward)
};
// The router gate's weight gradient, to be formed beside the experts' products (with a fold): dlogits (tokens, E) fp32, x the tokens, of the rows' dtype.
struct AnyGate {
  const float* dlogits;
  const void* x;
  float* partial;
  int64_t E;
};
// The selection's backward with the experts' rows y (select_bwd.h), which gives dlogits (tokens, E), to be formed beside dH (with a fold).
struct AnySelect {
  const float* logits;
  const int64_t* ids;
  const void *dout, *y;
  const int32_t* row_of_slot;
  const float *aux_f, *aux_scale;
  const uint8_t* padding;
  float* dlogits;
  int64_t E, K;
  int score_func, route_norm;
  float route_scale;
};
constexpr int kSelectBesideE = 64;  // experts at most
struct AnyGrad {  // c (El, M, N) = per segment a^T (rows, M) . b (rows, N)
  const void *a, *b;
  void* c;
  int64_t M, N;
  int through;  // with a fold: 1 a is the output gradient's, 2 b is the tokens'
};

bool any_path_ok(int dtype, int64_t D, int64_t F, int64_t R, std::initializer_list<const void*> matrices);
int any_gateup(const AnySeg& g, int dtype, const void* rows, const void* w1, const void* w3, void* gate, void* up, void* h,
               int64_t D, int64_t F, int64_t R, const AnyFold* fold, hipStream_t s);
// y (R, O) = x (R, I) . w (El, O, I)^T, and its input gradient
int any_linear(const AnySeg& g, int dtype, const void* x, const void* w, void* y, int64_t I, int64_t O, int64_t R,
               hipStream_t s);
int any_linear_dx(const AnySeg& g, int dtype, const void* dy, const void* w, void* dx, int64_t I, int64_t O, int64_t R,
                  hipStream_t s);
int any_dh(const AnySeg& g, int dtype, const void* dy, const void* w2, const void* gate, const void* up, void* dgate,
           void* dup, int64_t D, int64_t F, int64_t R, const AnyFold* fold, const AnyGate* router, const AnySelect* select,
           hipStream_t s);  // (with a fold: the gate's weight gradient or the selection's backward beside it)
// drows (null: not wanted) = dgate . w1 + dup . w3, and at most three weight gradients
int any_backward(const AnySeg& g, int dtype, const void* dgate, const void* dup, const void* w1, const void* w3, void* drows,
                 int64_t D, int64_t F, const AnyGrad* grads, int count, int64_t R, const AnyFold* fold, const AnyGate* router,
                 hipStream_t s);  // (router: only where it is one launch)
bool any_backward_is_one_launch(const AnySeg& g, int dtype, const void* drows, int64_t D, const AnyGrad* grads, int count, int64_t R);

}  // namespace mi355
