// Expert selection, shared by the router's own kernels (router.hip) and the fused selection +
// permutation plan (route.hip): DPP reductions and the selection of one token by a row of 16 lanes.
#pragma once
#include <type_traits>

#include "common.h"

namespace mi355 {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float softplus_f32(float x) {
  return x > 20.0f ? x : log1pf(expf(x));  // torch's threshold=20, beta=1
}

// Wave reductions of this file run on DPP row operations (VALU rate) plus four lane reads, not on
// shuffles: a shuffle is an LDS permute, and a token's selection needs about a hundred of them --
// with one wavefront per token the LDS pipe of a CU, not memory, was what the select kernels waited
// for.  The four controls below exchange within a row of 16 lanes (pairs, quads, halves, the row),
// so after them every lane holds its row's result; lanes 0, 16, 32, 48 then give the four rows.
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false);
}
constexpr int kDppPairs = 0xB1, kDppQuads = 0x4E, kDppHalfMirror = 0x141, kDppRowMirror = 0x140;

__device__ __forceinline__ float lane_f32(float v, int l) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// sum over the wave, left in every lane
__device__ __forceinline__ float wave_sum_dpp(float v) {
  v += dpp_f32<kDppPairs>(v);
  v += dpp_f32<kDppQuads>(v);
  v += dpp_f32<kDppHalfMirror>(v);
  v += dpp_f32<kDppRowMirror>(v);
  return (lane_f32(v, 0) + lane_f32(v, 16)) + (lane_f32(v, 32) + lane_f32(v, 48));
}
__device__ __forceinline__ float wave_max_dpp(float v) {
  v = fmaxf(v, dpp_f32<kDppPairs>(v));
  v = fmaxf(v, dpp_f32<kDppQuads>(v));
  v = fmaxf(v, dpp_f32<kDppHalfMirror>(v));
  v = fmaxf(v, dpp_f32<kDppRowMirror>(v));
  return fmaxf(fmaxf(lane_f32(v, 0), lane_f32(v, 16)), fmaxf(lane_f32(v, 32), lane_f32(v, 48)));
}

// the better of two (value, index) candidates: the larger value, ties to the lower index
__device__ __forceinline__ void take_better(float& v, int& idx, float ov, int oi) {
  if (ov > v || (ov == v && oi < idx)) { v = ov; idx = oi; }
}

// (value, index) arg-max across the wave, left in every lane; ties go to the lower index.
__device__ __forceinline__ void wave_argmax(float& v, int& idx) {
  { const float ov = dpp_f32<kDppPairs>(v); const int oi = dpp_i32<kDppPairs>(idx); take_better(v, idx, ov, oi); }
  { const float ov = dpp_f32<kDppQuads>(v); const int oi = dpp_i32<kDppQuads>(idx); take_better(v, idx, ov, oi); }
  { const float ov = dpp_f32<kDppHalfMirror>(v); const int oi = dpp_i32<kDppHalfMirror>(idx); take_better(v, idx, ov, oi); }
  { const float ov = dpp_f32<kDppRowMirror>(v); const int oi = dpp_i32<kDppRowMirror>(idx); take_better(v, idx, ov, oi); }
  float a = lane_f32(v, 0), b = lane_f32(v, 32);
  int ai = __builtin_amdgcn_readlane(idx, 0), bi = __builtin_amdgcn_readlane(idx, 32);
  take_better(a, ai, lane_f32(v, 16), __builtin_amdgcn_readlane(idx, 16));
  take_better(b, bi, lane_f32(v, 48), __builtin_amdgcn_readlane(idx, 48));
  take_better(a, ai, b, bi);
  v = a;
  idx = ai;
}

// the two largest of {a1 >= a2} and {b1 >= b2}, equal values counted as often as they occur
__device__ __forceinline__ void merge_top2(float& a1, float& a2, float b1, float b2) {
  const float lo = fminf(a1, b1);
  a1 = fmaxf(a1, b1);
  a2 = fmaxf(lo, fmaxf(a2, b2));
}
template <int CTRL>
__device__ __forceinline__ void top2_dpp(float& m1, float& m2) {
  const float o1 = dpp_f32<CTRL>(m1), o2 = dpp_f32<CTRL>(m2);
  merge_top2(m1, m2, o1, o2);
}
// The two largest values held by the `width` lanes (a power of two, 2..64; wave-uniform) of every
// aligned run of lanes, left in all of them.  Each step exchanges between two halves that already
// agree among themselves, so the mirrors of the DPP controls are as good as a butterfly.
__device__ __forceinline__ void run_top2(float& m1, float& m2, int width) {
  top2_dpp<kDppPairs>(m1, m2);
  if (width >= 4) top2_dpp<kDppQuads>(m1, m2);
  if (width >= 8) top2_dpp<kDppHalfMirror>(m1, m2);
  if (width >= 16) top2_dpp<kDppRowMirror>(m1, m2);
  if (width >= 32) {
    // lane ^ 16 within each half of the wave (swizzle bit mode: and 0x1f, or 0, xor 0x10)
    const float o1 = __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(m1), 0x401f));
    const float o2 = __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(m2), 0x401f));
    merge_top2(m1, m2, o1, o2);
  }
  if (width >= 64) {
    float a1 = lane_f32(m1, 0), a2 = lane_f32(m2, 0);
    merge_top2(a1, a2, lane_f32(m1, 32), lane_f32(m2, 32));
    m1 = a1;
    m2 = a2;
  }
}

// ---- selection with one token per row of 16 lanes ----------------------------------------------
// For E <= 256, K <= 16 and 1, 2, 4, 8 or 16 expert groups (or none): four tokens per
// wavefront, lane l of a row keeps experts l*VPR .. l*VPR + VPR - 1, so a group is a run of
// 16 / num_groups whole lanes.  Every reduction is four
// DPP steps inside the row and serves four tokens at once, where the wave-per-token kernel
// spends the same steps plus eight lane reads on one: the selection is bound by instruction
// issue, not by memory, and this form issues about a third of the instructions per token.  The
// choice (larger value, ties to the lower expert index) does not depend on the order of the
// comparisons, so both kernels pick the same experts.  FULL: E == 16 * VPR; else the lanes past
// the last expert hold -inf and are never chosen (no groups then).
__device__ __forceinline__ float row_max(float v) {
  v = fmaxf(v, dpp_f32<kDppPairs>(v));
  v = fmaxf(v, dpp_f32<kDppQuads>(v));
  v = fmaxf(v, dpp_f32<kDppHalfMirror>(v));
  return fmaxf(v, dpp_f32<kDppRowMirror>(v));
}
__device__ __forceinline__ float row_sum(float v) {
  v += dpp_f32<kDppPairs>(v);
  v += dpp_f32<kDppQuads>(v);
  v += dpp_f32<kDppHalfMirror>(v);
  return v + dpp_f32<kDppRowMirror>(v);
}
__device__ __forceinline__ uint32_t row_max_u32(uint32_t v) {
  v = max(v, static_cast<uint32_t>(dpp_i32<kDppPairs>(static_cast<int>(v))));
  v = max(v, static_cast<uint32_t>(dpp_i32<kDppQuads>(static_cast<int>(v))));
  v = max(v, static_cast<uint32_t>(dpp_i32<kDppHalfMirror>(static_cast<int>(v))));
  return max(v, static_cast<uint32_t>(dpp_i32<kDppRowMirror>(static_cast<int>(v))));
}
// floats as integers of the same order (the two zeros equal, NaN above or below everything), never 0
__device__ __forceinline__ uint32_t order_key(float v) {
  const uint32_t u = __float_as_uint(v + 0.0f);
  return max(u & 0x80000000u ? ~u : u | 0x80000000u, 1u);
}
__device__ __forceinline__ float from_order_key(uint32_t k) {
  return __uint_as_float(k & 0x80000000u ? k & 0x7fffffffu : ~k);
}

struct SelectArgs {
  const float* expert_bias;  // (E) or null
  int E, K, score_func, route_norm;
  float route_scale;
  int num_groups, num_limited;
};
struct RowChoice {
  float weight;    // lane k < K: the k-th choice's routing weight
  int id;          // ... and expert
  unsigned taken;  // this lane's chosen experts, one bit each (FULL false: also its experts >= E)
};

// x: the row's logits, this lane's VPR of them (-inf past E).  s: their score function, filled when
// want_scores is set or the choice needs it.
// want_cutoff: also the best choice value left after the K winners, and no choice by logit (the
// cutoff is a score).
//
// Bound by instruction issue.  The K rounds work on integer keys of the choice values' order, of which a
// row's maximum is four single instructions; the lowest lane that holds it, found in a ballot, is the
// winner (lanes hold ascending experts, so ties go to the lower index), and its expert travels to
// lane k by a permute nothing waits for.  Where the choice is by logit, the winner's logit is in
// the key, so only the K winners' score functions are evaluated.  Per token of 128 experts and K = 8 about half
// the instructions of the (value, index, score) triples compared and carried before: the selection of 8192
// tokens as a kernel of its own 8.7 -> 5.9 us.
template <int VPR, bool FULL>
__device__ __forceinline__ RowChoice select_row(const SelectArgs& p, const float (&x)[VPR], int l, bool want_scores,
                                                bool want_cutoff, float (&s)[VPR], float& cutoff) {
  const int e0 = l * VPR;
  // choice values: the logit itself when nothing but a monotone score function stands between
  // it and the choice (exact: two exp() implementations can order two nearly equal scores
  // differently, never two logits), else score (+ bias)
  const bool by_logit = !p.expert_bias && p.num_groups == 0 && !want_cutoff;
  float top = 0.0f, sum = 1.0f;  // of a softmax
  if (p.score_func == MI355_SCORE_SOFTMAX) {
    float m = x[0];
#pragma unroll
    for (int j = 1; j < VPR; ++j) m = fmaxf(m, x[j]);
    top = row_max(m);
    sum = 0.0f;
#pragma unroll
    for (int j = 0; j < VPR; ++j) {
      s[j] = expf(x[j] - top);
      sum += s[j];
    }
    sum = row_sum(sum);
  }
  if (want_scores || !by_logit) {
    if (p.score_func == MI355_SCORE_SOFTMAX) {
#pragma unroll
      for (int j = 0; j < VPR; ++j) s[j] = s[j] / sum;
    } else if (p.score_func == MI355_SCORE_SIGMOID) {
#pragma unroll
      for (int j = 0; j < VPR; ++j) s[j] = 1.0f / (1.0f + expf(-x[j]));
    } else {
#pragma unroll
      for (int j = 0; j < VPR; ++j) s[j] = sqrtf(softplus_f32(x[j]));
    }
  }
  float c[VPR];
  if (p.expert_bias) {
#pragma unroll
    for (int j = 0; j < VPR; ++j) c[j] = s[j] + ((FULL || e0 + j < p.E) ? p.expert_bias[e0 + j] : 0.0f);
  } else {
#pragma unroll
    for (int j = 0; j < VPR; ++j) c[j] = by_logit ? x[j] : s[j];
  }
  if (p.num_groups > 0) {
    // group score = sum of the group's two best choice values: each lane folds its own, the lanes
    // of a group join them; every lane then counts the groups that beat its own (a higher score,
    // or the same score and a lower index), seeing each other group's score by a row rotation,
    // and a group beaten by num_limited others or more is masked
    const int m = 16 / p.num_groups;  // lanes per group
    float m1 = -INFINITY, m2 = -INFINITY;
#pragma unroll
    for (int j = 0; j < VPR; ++j) merge_top2(m1, m2, c[j], -INFINITY);
    if (m >= 2) top2_dpp<kDppPairs>(m1, m2);
    if (m >= 4) top2_dpp<kDppQuads>(m1, m2);
    if (m >= 8) top2_dpp<kDppHalfMirror>(m1, m2);
    if (m >= 16) top2_dpp<kDppRowMirror>(m1, m2);
    const float gs = m1 + m2;
    const int gid = l / m;
    int beaten_by = 0;
    auto other = [&](auto n_t) {
      constexpr int n = decltype(n_t)::value;
      if (n % m != 0) return;  // wave-uniform
      const float og = dpp_f32<0x120 + n>(gs);  // row rotation by n lanes
      const int oi = dpp_i32<0x120 + n>(gid);
      beaten_by += (og > gs || (og == gs && oi < gid)) ? 1 : 0;
    };
    other(std::integral_constant<int, 1>{}); other(std::integral_constant<int, 2>{});
    other(std::integral_constant<int, 3>{}); other(std::integral_constant<int, 4>{});
    other(std::integral_constant<int, 5>{}); other(std::integral_constant<int, 6>{});
    other(std::integral_constant<int, 7>{}); other(std::integral_constant<int, 8>{});
    other(std::integral_constant<int, 9>{}); other(std::integral_constant<int, 10>{});
    other(std::integral_constant<int, 11>{}); other(std::integral_constant<int, 12>{});
    other(std::integral_constant<int, 13>{}); other(std::integral_constant<int, 14>{});
    other(std::integral_constant<int, 15>{});
    if (beaten_by >= p.num_limited) {
#pragma unroll
      for (int j = 0; j < VPR; ++j) c[j] = -INFINITY;
    }
  }

  uint32_t key[VPR];  // 0: taken, or past E
#pragma unroll
  for (int j = 0; j < VPR; ++j) key[j] = FULL || e0 + j < p.E ? order_key(c[j]) : 0u;
  const int lane = __lane_id(), row0 = lane & 48;
  float my_w = 0.0f;
  int my_id = 0;
  auto lane_max = [&]() {
    uint32_t m = key[0];
#pragma unroll
    for (int j = 1; j < VPR; ++j) m = max(m, key[j]);
    return m;
  };
  for (int k = 0; k < p.K; ++k) {
    const uint32_t m = lane_max(), best = row_max_u32(m);
    const int winner = __ffs(static_cast<uint32_t>(__ballot(m == best) >> row0) & 0xffffu) - 1;
    int at = 0;  // the lane's first expert with its own maximum
    float score = 0.0f;
#pragma unroll
    for (int j = VPR - 1; j >= 0; --j) {
      const bool here = key[j] == m;
      at = here ? j : at;
      score = here ? s[j] : score;
    }
    const int id = __builtin_amdgcn_ds_bpermute((row0 + winner) << 2, e0 + at);
    const float w = by_logit ? from_order_key(best)
                             : __int_as_float(__builtin_amdgcn_ds_bpermute((row0 + winner) << 2, __float_as_int(score)));
    if (l == k) {
      my_id = id;
      my_w = w;
    }
    const int gone = winner == l ? at : -1;
#pragma unroll
    for (int j = 0; j < VPR; ++j) key[j] = j == gone ? 0u : key[j];
  }
  unsigned taken = 0;
#pragma unroll
  for (int j = 0; j < VPR; ++j) taken |= key[j] ? 0u : 1u << j;
  // the best choice value left after the K winners: the (K+1)-th of a sorted top-(K+1)
  if (want_cutoff) cutoff = from_order_key(row_max_u32(lane_max()));
  if (by_logit) {  // my_w is the logit
    if (p.score_func == MI355_SCORE_SOFTMAX) my_w = expf(my_w - top) / sum;
    else if (p.score_func == MI355_SCORE_SIGMOID) my_w = 1.0f / (1.0f + expf(-my_w));
    else my_w = sqrtf(softplus_f32(my_w));
  }
  if (p.route_norm) {
    const float chosen = row_sum(l < p.K ? my_w : 0.0f);
    my_w = my_w / (chosen + 1e-20f);
  }
  my_w = my_w * p.route_scale;
  return {my_w, my_id, taken};
}

// this lane's logits of the row at `src` (E of them); FULL rows of four or more per lane are read 16 bytes at a time
template <int VPR, bool FULL>
__device__ __forceinline__ void load_row(const float* __restrict__ src, int l, int E, float (&x)[VPR]) {
  if constexpr (FULL && VPR >= 4) {
#pragma unroll
    for (int q = 0; q < VPR / 4; ++q) {
      const f32x4 v = reinterpret_cast<const f32x4*>(src + l * VPR)[q];
      x[q * 4] = v[0]; x[q * 4 + 1] = v[1]; x[q * 4 + 2] = v[2]; x[q * 4 + 3] = v[3];
    }
  } else {
#pragma unroll
    for (int j = 0; j < VPR; ++j) x[j] = (FULL || l * VPR + j < E) ? src[l * VPR + j] : -INFINITY;
  }
}

// experts per lane for E <= 256: a power of two
inline int row_vpr(int64_t E) { return E <= 16 ? 1 : E <= 32 ? 2 : E <= 64 ? 4 : E <= 128 ? 8 : 16; }

// calls f(integral_constant VPR, bool_constant FULL) for E <= 256
template <typename Fn>
void with_row_shape(int64_t E, Fn f) {
  auto go = [&](auto vpr) {
    if (E == 16 * decltype(vpr)::value) f(vpr, std::true_type{});
    else f(vpr, std::false_type{});
  };
  switch (row_vpr(E)) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 8: go(std::integral_constant<int, 8>{}); break;
    default: go(std::integral_constant<int, 16>{}); break;
  }
}

// what select_row covers
inline bool select_row_covers(int64_t E, int64_t K, int num_groups, int mode) {
  return mode == MI355_SELECT_TOPK && K <= 16 && E <= 256 &&
         (num_groups == 0 || (num_groups <= 16 && 16 % num_groups == 0 && E == 16 * row_vpr(E)));
}

}  // namespace
}  // namespace mi355
