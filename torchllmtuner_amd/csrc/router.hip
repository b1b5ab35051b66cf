// Router: fp32 gate projection and the fused score / top-k / gather / norm pass.
//
// Selection kernels: a token is owned by one row of 16 lanes (E <= 256: four tokens per
// wavefront, lane l keeps consecutive experts) or by one 64-lane wavefront (any E up to 512:
// lane l keeps experts l, l+64, l+128, ...).  The scores stay in registers, the softmax max /
// sum and every arg-max are DPP reductions, and the K winners are written by lanes 0..K-1.  No
// LDS, no atomics; HBM traffic is the (T,E) logits once plus the (T,K) outputs.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gemm_generic.h"
#include "select_bwd.h"

namespace mi355 {
namespace {

constexpr int kMaxVPL = 8;  // experts per lane -> E <= 512

template <int VPL>
__device__ __forceinline__ float pick(const float (&a)[VPL], int j) {
  float r = a[0];
#pragma unroll
  for (int q = 1; q < VPL; ++q) r = (j == q) ? a[q] : r;
  return r;
}

template <int VPL>
__global__ __launch_bounds__(256) void select_fwd_kernel(
    const float* __restrict__ logits, const float* __restrict__ expert_bias,
    float* __restrict__ weights, int64_t* __restrict__ ids, float* __restrict__ scores_out,
    uint8_t* __restrict__ map_out, float* __restrict__ cutoff_out, int T, int E, int K, int score_func,
    int route_norm,
    float route_scale, int num_groups, int num_limited, int mode) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;

  float s[VPL], x[VPL];
  compute_scores<VPL>(logits + static_cast<int64_t>(t) * E, E, lane, score_func, s, x);
  if (scores_out) {
#pragma unroll
    for (int j = 0; j < VPL; ++j)
      if (lane + j * kWave < E) scores_out[static_cast<int64_t>(t) * E + lane + j * kWave] = s[j];
  }

  float my_w = 0.0f;
  int my_id = 0;

  if (mode == MI355_SELECT_TOPK) {
    // Choice values.  Without a bias and without groups the choice is the plain top-k of the
    // scores, and every score function here is non-decreasing in the logit: the experts are
    // then chosen by LOGIT, which is exact -- two implementations of exp() that differ in the
    // last ulp can order two nearly equal scores differently, but never two logits.
    // (not when the caller asks for the cutoff: that is a choice VALUE, the (K+1)-th score)
    const bool by_logit = !expert_bias && num_groups == 0 && !cutoff_out;
    float c[VPL];
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int e = lane + j * kWave;
      c[j] = e < E ? (by_logit ? x[j] : (expert_bias ? s[j] + expert_bias[e] : s[j])) : -INFINITY;
    }
    unsigned taken = 0;
#pragma unroll
    for (int j = 0; j < VPL; ++j)
      if (lane + j * kWave >= E) taken |= 1u << j;  // never selectable

    if (num_groups > 0) {
      // group score = sum of the group's two best choice scores; keep the best
      // num_limited groups (ties to the lower group), mask the rest to -inf.
      const int P = E / num_groups;
      float gscore = -INFINITY;  // lane g (< num_groups) keeps group g's score
      if (P < kWave && kWave % P == 0) {
        // a group is an aligned run of P lanes of one register: the registers' runs are reduced side
        // by side (independent chains), then lane g fetches the sum of its group's run
        const int runs = kWave / P;  // groups per register
        float sum[VPL];
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
          float m1 = c[j], m2 = -INFINITY;
          run_top2(m1, m2, P);
          sum[j] = m1 + m2;
        }
        const int from = (lane % runs) * P;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
          const float got = __int_as_float(__builtin_amdgcn_ds_bpermute(from << 2, __float_as_int(sum[j])));
          if (lane / runs == j) gscore = got;
        }
      } else if (P % kWave == 0) {
        // a group is P / 64 whole registers: each lane folds its own values, then one wave-wide step
        const int regs = P / kWave;
        float m1 = -INFINITY, m2 = -INFINITY;
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
          merge_top2(m1, m2, c[j], -INFINITY);
          if ((j + 1) % regs == 0) {
            run_top2(m1, m2, kWave);
            if (lane == j / regs) gscore = m1 + m2;
            m1 = m2 = -INFINITY;
          }
        }
      } else {
        for (int g = 0; g < num_groups; ++g) {
          float top2 = 0.0f;
          unsigned used = 0;
          for (int r = 0; r < 2; ++r) {
            float bv = -INFINITY;
            int bi = 0x7fffffff;
#pragma unroll
            for (int j = 0; j < VPL; ++j) {
              const int e = lane + j * kWave;
              const bool in = e < E && e / P == g && !((used >> j) & 1u);
              if (in && (c[j] > bv || bi == 0x7fffffff)) { bv = c[j]; bi = e; }
            }
            wave_argmax(bv, bi);
            top2 += bv;
            if ((bi & 63) == lane) used |= 1u << (bi >> 6);
          }
          if (lane == g) gscore = top2;
        }
      }
      // a group is kept when fewer than num_limited groups beat it (a higher score, or the same
      // score and a lower index): the groups a repeated arg-max would pick, without the repeats
      const float mine = lane < num_groups ? gscore : -INFINITY;
      int beaten_by = 0;
      for (int g = 0; g < num_groups; ++g) {
        const float sg = lane_f32(gscore, g);
        beaten_by += (sg > mine || (sg == mine && g < lane)) ? 1 : 0;
      }
      const unsigned long long keep = __ballot(lane < num_groups && beaten_by < num_limited);
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        const int e = lane + j * kWave;
        if (e < E && !((keep >> (e / P)) & 1ull)) c[j] = -INFINITY;
      }
    }

    for (int k = 0; k < K; ++k) {
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        if ((taken >> j) & 1u) continue;
        if (bi == 0x7fffffff || c[j] > bv) { bv = c[j]; bi = lane + j * kWave; }
      }
      wave_argmax(bv, bi);
      const int owner = __builtin_amdgcn_readfirstlane(bi & 63), slot = bi >> 6;
      float sv = 0.0f;
      if (lane == owner) {
        taken |= 1u << slot;
        sv = pick<VPL>(s, slot);
      }
      sv = lane_f32(sv, owner);  // owner is wave-uniform: a lane read, not a shuffle
      if (lane == k) { my_w = sv; my_id = bi; }
    }
    if (cutoff_out) {
      // the best choice score left after the K winners: the (K+1)-th of a sorted top-(K+1)
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < VPL; ++j) {
        if ((taken >> j) & 1u) continue;
        if (bi == 0x7fffffff || c[j] > bv) { bv = c[j]; bi = lane + j * kWave; }
      }
      wave_argmax(bv, bi);
      if (lane == 0) cutoff_out[t] = bv;
    }
  } else {
    // fixed: (t + k) % E ; balanced: (t*K + k) % E ; lane k owns slot k (K <= 64)
    const int64_t base = mode == MI355_SELECT_FIXED ? static_cast<int64_t>(t) + lane
                                                    : static_cast<int64_t>(t) * K + lane;
    my_id = static_cast<int>(base % E);
    // gather the unbiased score of each slot's expert from its owner lane
    for (int k = 0; k < K; ++k) {
      const int want = __builtin_amdgcn_readlane(my_id, k);
      const float got = lane_f32(pick<VPL>(s, want >> 6), __builtin_amdgcn_readfirstlane(want & 63));
      if (lane == k) my_w = got;
    }
  }

  if (mode == MI355_SELECT_FIXED) {
    my_w = 1.0f / static_cast<float>(K);
  } else {
    if (route_norm) {
      const float sum = wave_sum_dpp(lane < K ? my_w : 0.0f);
      my_w = my_w / (sum + 1e-20f);
    }
    my_w = my_w * route_scale;
  }
  if (lane < K) {
    weights[static_cast<int64_t>(t) * K + lane] = my_w;
    ids[static_cast<int64_t>(t) * K + lane] = my_id;
  }
  if (map_out) {
    // one-hot routing map of the token, one byte per expert
    unsigned chosen = 0;
    for (int k = 0; k < K; ++k) {
      const int idk = __builtin_amdgcn_readlane(my_id, k);
      if ((idk & 63) == lane) chosen |= 1u << (idk >> 6);
    }
#pragma unroll
    for (int j = 0; j < VPL; ++j)
      if (lane + j * kWave < E) map_out[static_cast<int64_t>(t) * E + lane + j * kWave] = (chosen >> j) & 1u;
  }
}

// ---- the same selection with one token per row of 16 lanes (select_rows.h) ----------------------
template <int VPR, bool FULL>
__global__ __launch_bounds__(256) void select_rows_kernel(
    const float* __restrict__ logits, SelectArgs p, float* __restrict__ weights,
    int64_t* __restrict__ ids, float* __restrict__ scores_out, uint8_t* __restrict__ map_out,
    float* __restrict__ cutoff_out, int T) {
  const int E = p.E, K = p.K;
  const int l = threadIdx.x & 15;
  const int t_raw = blockIdx.x * 16 + (threadIdx.x >> 4);
  const bool live = t_raw < T;
  const int t = live ? t_raw : T - 1;  // a row past the end redoes the last token and stores nothing
  const int e0 = l * VPR;
  float x[VPR], s[VPR], cutoff = 0.0f;
  load_row<VPR, FULL>(logits + static_cast<int64_t>(t) * E, l, E, x);
  const RowChoice c = select_row<VPR, FULL>(p, x, l, scores_out != nullptr, cutoff_out != nullptr, s, cutoff);
  if (!live) return;
  if (scores_out) {
    float* dst = scores_out + static_cast<int64_t>(t) * E + e0;
    if constexpr (FULL && VPR >= 4) {
#pragma unroll
      for (int q = 0; q < VPR / 4; ++q) {
        const f32x4 v = {s[q * 4], s[q * 4 + 1], s[q * 4 + 2], s[q * 4 + 3]};
        reinterpret_cast<f32x4*>(dst)[q] = v;
      }
    } else {
#pragma unroll
      for (int j = 0; j < VPR; ++j)
        if (FULL || e0 + j < E) dst[j] = s[j];
    }
  }
  if (cutoff_out && l == 0) cutoff_out[t] = cutoff;
  if (l < K) {
    weights[static_cast<int64_t>(t) * K + l] = c.weight;
    ids[static_cast<int64_t>(t) * K + l] = c.id;
  }
  if (map_out) {
    // one-hot routing map of the token, one byte per expert: this lane's VPR experts
    uint8_t* dst = map_out + static_cast<int64_t>(t) * E + e0;
    if constexpr (FULL && VPR >= 4) {
#pragma unroll
      for (int q = 0; q < VPR / 4; ++q) {
        const unsigned b = c.taken >> (q * 4);
        reinterpret_cast<uint32_t*>(dst)[q] = (b & 1u) | ((b & 2u) << 7) | ((b & 4u) << 14) | ((b & 8u) << 21);
      }
    } else {
#pragma unroll
      for (int j = 0; j < VPR; ++j)
        if (FULL || e0 + j < E) dst[j] = (c.taken >> j) & 1u;
    }
  }
}

// whether select_rows_kernel serves this call
inline bool select_rows_ok(const float* logits, const float* scores, const uint8_t* map, int64_t E, int64_t K,
                           int num_groups, int mode) {
  return select_row_covers(E, K, num_groups, mode) && aligned16(logits) && aligned16(scores) &&
         reinterpret_cast<uintptr_t>(map) % 4 == 0;
}
int launch_select_rows(const SelectArgs& p, const float* logits, float* weights, int64_t* ids, float* scores,
                       uint8_t* map, float* cutoff, int64_t T, hipStream_t s, const char* what) {
  with_row_shape(p.E, [&](auto vpr, auto full) {
    hipLaunchKernelGGL((select_rows_kernel<decltype(vpr)::value, decltype(full)::value>), dim3((unsigned)((T + 15) / 16)),
                       dim3(256), 0, s, logits, p, weights, ids, scores, map, cutoff, (int)T);
  });
  return check_launch(what);
}

template <int VPL, typename T = void>
__global__ __launch_bounds__(256) void select_bwd_kernel(SelectBwd p) {
  extern __shared__ float lds[];
  select_bwd_part<VPL, T>(p, blockIdx.x, lds);
}

int check_router_args(int64_t T, int64_t E, int64_t K) {
  MI355_REQUIRE(T >= 0 && T < (1ll << 31), "router: T=%lld out of range", (long long)T);
  MI355_REQUIRE(E >= 1 && E <= kMaxVPL * kWave, "router: E=%lld must be in [1,%d]", (long long)E,
                kMaxVPL * kWave);
  MI355_REQUIRE(K >= 1 && K <= E, "router: K=%lld must be in [1,E]", (long long)K);
  return MI355_OK;
}

}  // namespace
}  // namespace mi355

using namespace mi355;

// Scratch of the forward for whatever dtypes follow: the weight pieces, then the partial sums.
extern "C" int64_t mi355_router_gate_fwd_workspace_bytes(int64_t T, int64_t D, int64_t E) {
  if (T < 0 || D < 1 || E < 1) return 0;
  const int64_t pieces = router_fwd_pieces_bytes(MI355_BF16, MI355_F32, T, D, E);
  const int splits = std::max(router_fwd_splits(MI355_BF16, MI355_F32, T, D, E),
                              router_fwd_splits(MI355_F32, MI355_F32, T, D, E));
  return pieces + (splits > 1 ? splits * T * E * 4 : 0);
}

extern "C" int mi355_router_gate_fwd(const void* x, int x_dtype, const void* w, int w_dtype,
                                     const float* logit_bias, float* logits, void* workspace,
                                     int64_t T, int64_t D, int64_t E, void* stream) {
  MI355_REQUIRE(T >= 0 && D >= 1 && E >= 1, "router_gate_fwd: bad shape T=%lld D=%lld E=%lld",
                (long long)T, (long long)D, (long long)E);
  MI355_REQUIRE(T < (1ll << 31) && D < (1ll << 31), "router_gate_fwd: shape exceeds int32");
  if (T == 0) return MI355_OK;
  MI355_REQUIRE(x && w && logits, "router_gate_fwd: null pointer");
  const int splits = aligned16({x, w, logit_bias, logits, workspace}) ? router_fwd_splits(x_dtype, w_dtype, T, D, E) : 0;
  const int64_t pieces = splits ? router_fwd_pieces_bytes(x_dtype, w_dtype, T, D, E) : 0;
  if (splits > 0 && (workspace || (splits == 1 && pieces == 0))) {
    float* partial = splits > 1 ? reinterpret_cast<float*>(static_cast<char*>(workspace) + pieces) : logits;
    if (int rc = router_fwd_partial(x, x_dtype, static_cast<const float*>(w), logit_bias, partial, workspace, nullptr, T, D, E,
                                    as_stream(stream)))
      return rc;
    return splits > 1 ? router_logits_reduce(partial, logit_bias, logits, T, E, splits, as_stream(stream)) : MI355_OK;
  }
  GemmArgs g{};
  g.A = x; g.B = w; g.C = logits; g.bias = logit_bias;
  g.a_rs = D; g.a_cs = 1;
  g.b_rs = 1; g.b_cs = D;  // B(k=d, n=e) = w[e][d]
  g.ldc = E; g.M = (int)T; g.N = (int)E; g.K = (int)D;
  g.mode = GEMM_DENSE; g.ksplit = 1;
  return launch_gemm(g, x_dtype, w_dtype, MI355_F32, gemm_grid_dense(g.M, g.N, 1), as_stream(stream));
}

static int gate_bwd_ksplit(int64_t T, int64_t D, int64_t E) {
  const int64_t tiles = ((E + 63) / 64) * ((D + 63) / 64);
  int64_t split = (1024 + tiles - 1) / tiles;
  const int64_t max_split = (T + 255) / 256;
  if (split > max_split) split = max_split;
  if (split < 1) split = 1;
  if (split > 64) split = 64;
  return (int)split;
}

extern "C" int64_t mi355_router_gate_bwd_workspace_bytes(int64_t T, int64_t D, int64_t E) {
  if (T < 0 || D < 1 || E < 1) return 0;
  const int s = gate_bwd_ksplit(T, D, E);
  const int64_t strided = s > 1 ? (int64_t)s * E * D * 4 : 0;
  const int64_t x3 = router_x3_ok(MI355_BF16, MI355_F32, D, E) ? router_x3_bwd_workspace(T, D, E) : 0;
  const int64_t few = router_few_bwd_ok(MI355_F32, MI355_F32, T, D, E) ? router_few_bwd_workspace(T, D, E) : 0;
  return std::max({strided, x3, few});
}

extern "C" int mi355_router_gate_add_bwd(const float* dlogits, const void* x, int x_dtype, const void* w, int w_dtype,
                                         const void* pieces, const void* addend, void* dx, void* dw, void* workspace,
                                         int64_t T, int64_t D, int64_t E, void* stream) {
  MI355_REQUIRE(T >= 0 && D >= 1 && E >= 1 && T < (1ll << 31) && D < (1ll << 31),
                "router_gate_bwd: bad shape");
  hipStream_t s = as_stream(stream);
  // (both of these fetch and store 16 bytes at a time; the strided kernel looks for itself)
  const bool vec = workspace && aligned16({dlogits, x, w, pieces, addend, dx, dw, workspace});
  if (vec && router_x3_ok(x_dtype, w_dtype, D, E)) {
    MI355_REQUIRE(dlogits && w && (x || !dw), "router_gate_bwd: null pointer");
    return router_x3_bwd(dlogits, x, static_cast<const float*>(w), pieces, RowSum{addend}, dx, static_cast<float*>(dw),
                         workspace, T, D, E, s);
  }
  if (vec && T > 0 && router_few_bwd_ok(x_dtype, w_dtype, T, D, E) && (dx || dw)) {
    MI355_REQUIRE(dlogits && w && (x || !dw), "router_gate_bwd: null pointer");
    return router_few_bwd(dlogits, x, x_dtype, static_cast<const float*>(w), RowSum{addend}, dx, static_cast<float*>(dw), workspace,
                          T, D, E, s);
  }
  if (dx && T > 0) {
    GemmArgs g{};
    g.A = dlogits; g.B = w; g.C = dx; g.addend = addend;
    g.a_rs = E; g.a_cs = 1;
    g.b_rs = D; g.b_cs = 1;  // B(k=e, n=d) = w[e][d]
    g.ldc = D; g.M = (int)T; g.N = (int)D; g.K = (int)E;
    g.mode = GEMM_DENSE; g.ksplit = 1;
    int rc = launch_gemm(g, MI355_F32, w_dtype, x_dtype, gemm_grid_dense(g.M, g.N, 1), s);
    if (rc) return rc;
  }
  if (dw) {
    const int split = gate_bwd_ksplit(T, D, E);
    MI355_REQUIRE(split == 1 || workspace, "router_gate_bwd: workspace required");
    GemmArgs g{};
    g.A = dlogits; g.B = x;
    g.a_rs = 1; g.a_cs = E;  // A(m=e, k=t) = dlogits[t][e]
    g.b_rs = D; g.b_cs = 1;  // B(k=t, n=d) = x[t][d]
    g.ldc = D; g.M = (int)E; g.N = (int)D; g.K = (int)T;
    g.mode = GEMM_DENSE; g.ksplit = split;
    g.C = split > 1 ? workspace : dw;
    int rc = launch_gemm(g, MI355_F32, x_dtype, w_dtype, gemm_grid_dense(g.M, g.N, split), s);
    if (rc) return rc;
    if (split > 1)
      return launch_splitk_reduce(static_cast<const float*>(workspace), dw, w_dtype, E * D, split, s);
  }
  return MI355_OK;
}

extern "C" int mi355_router_gate_sum_bwd_covers(int x_dtype, int w_dtype, int64_t D, int64_t E, int64_t K) {
  return E >= 1 && K >= 1 && K <= 16 && x_dtype == MI355_BF16 &&
                 (router_x3_ok(x_dtype, w_dtype, D, E) || router_few_ok(x_dtype, w_dtype, D, E))
             ? 1
             : 0;
}

extern "C" int mi355_router_gate_sum_bwd(const float* dlogits, const void* x, int x_dtype, const float* w, const void* pieces,
                                         const void* drows, const int32_t* row_of_slot, int64_t row_capacity, int64_t K,
                                         const void* addend, void* dx, float* dw, void* workspace, int64_t T, int64_t D,
                                         int64_t E, void* stream) {
  MI355_REQUIRE(T >= 1 && T < (1ll << 31) && D >= 1 && D < (1ll << 31) && row_capacity >= 0 && row_capacity < (1ll << 31),
                "router_gate_sum_bwd: bad shape");
  if (!mi355_router_gate_sum_bwd_covers(x_dtype, MI355_F32, D, E, K))
    return fail(MI355_EUNSUP, "router_gate_sum_bwd: not covered; use mi355_permute_rows_add_bwd and mi355_router_gate_add_bwd");
  MI355_REQUIRE(dlogits && x && w && drows && row_of_slot && dx && workspace &&
                    aligned16({dlogits, x, w, pieces, drows, addend, dx, dw, workspace}),
                "router_gate_sum_bwd: null or misaligned pointer");
  const RowSum sum{addend, drows, row_of_slot, K, row_capacity};
  if (router_few_ok(x_dtype, MI355_F32, D, E))
    return router_few_bwd(dlogits, x, x_dtype, w, sum, dx, dw, workspace, T, D, E, as_stream(stream));
  return router_x3_bwd(dlogits, x, w, pieces, sum, dx, dw, workspace, T, D, E, as_stream(stream));
}

extern "C" int mi355_router_gate_rows_bwd_covers(int x_dtype, int w_dtype, int64_t D, int64_t E) {
  return E >= 1 && router_few_ok(x_dtype, w_dtype, D, E) ? 1 : 0;
}

extern "C" int mi355_router_gate_rows_bwd(const float* dlogits, int x_dtype, const float* w, const void* drows,
                                          const int32_t* row_of_slot, int64_t row_capacity, int64_t K, const void* addend,
                                          void* dx, const float* dw_partial, float* dw, int64_t T, int64_t D, int64_t E,
                                          void* stream) {
  MI355_REQUIRE(T >= 1 && T < (1ll << 31) && D >= 1 && D < (1ll << 31) && E >= 1 && K >= 1 && K <= 64 && row_capacity >= 0 &&
                    row_capacity < (1ll << 31),
                "router_gate_rows_bwd: bad shape");
  if (!router_few_ok(x_dtype, MI355_F32, D, E))
    return fail(MI355_EUNSUP, "router_gate_rows_bwd: not covered; use mi355_permute_rows_add_bwd and mi355_router_gate_add_bwd");
  MI355_REQUIRE(!dx || (dlogits && w && drows && row_of_slot), "router_gate_rows_bwd: null pointer");
  MI355_REQUIRE(!dw || dw_partial, "router_gate_rows_bwd: null pointer");
  MI355_REQUIRE(aligned16({dlogits, w, drows, addend, dx, dw_partial, dw}), "router_gate_rows_bwd: misaligned pointer");
  return router_rows_bwd(dlogits, x_dtype, w, drows, row_of_slot, row_capacity, K, addend, dx, dw_partial, dw, T, D, E,
                         as_stream(stream));
}

extern "C" int mi355_router_gate_bwd(const float* dlogits, const void* x, int x_dtype,
                                     const void* w, int w_dtype, void* dx, void* dw,
                                     void* workspace, int64_t T, int64_t D, int64_t E,
                                     void* stream) {
  return mi355_router_gate_add_bwd(dlogits, x, x_dtype, w, w_dtype, nullptr, nullptr, dx, dw, workspace, T, D, E, stream);
}

extern "C" int mi355_router_gate_fwd_splits(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  return router_fwd_splits(x_dtype, w_dtype, T, D, E);
}

extern "C" int64_t mi355_router_gate_fwd_pieces_bytes(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  return T >= 1 && D >= 1 && E >= 1 ? router_fwd_pieces_bytes(x_dtype, w_dtype, T, D, E) : 0;
}

extern "C" int64_t mi355_router_gate_fwd_kept_bytes(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  return T >= 1 && D >= 1 && E >= 1 ? router_fwd_kept_bytes(x_dtype, w_dtype, T, D, E) : 0;
}

static int gate_fwd_partial(const void* x, int x_dtype, const float* w, const float* logit_bias, float* partial, void* pieces, void* keep,
                            int64_t T, int64_t D, int64_t E, void* stream) {
  MI355_REQUIRE(T >= 1 && D >= 1 && E >= 1 && T < (1ll << 31) && D < (1ll << 31), "router_gate_fwd_partial: bad shape");
  if (router_fwd_splits(x_dtype, MI355_F32, T, D, E) < 1)
    return fail(MI355_EUNSUP, "router_gate_fwd_partial: dtype / width not covered; use mi355_router_gate_fwd");
  MI355_REQUIRE(x && w && partial && aligned16(x) && aligned16(w) && aligned16(partial),
                "router_gate_fwd_partial: null or misaligned pointer");
  MI355_REQUIRE(pieces || router_fwd_pieces_bytes(x_dtype, MI355_F32, T, D, E) == 0,
                "router_gate_fwd_partial: scratch for the weight pieces required");
  return router_fwd_partial(x, x_dtype, w, logit_bias, partial, pieces, keep, T, D, E, as_stream(stream));
}
extern "C" int mi355_router_gate_fwd_partial(const void* x, int x_dtype, const float* w, const float* logit_bias,
                                             float* partial, void* pieces, int64_t T, int64_t D, int64_t E,
                                             void* stream) {
  return gate_fwd_partial(x, x_dtype, w, logit_bias, partial, pieces, nullptr, T, D, E, stream);
}
extern "C" int mi355_router_gate_fwd_keeping(const void* x, int x_dtype, const float* w, const float* logit_bias, float* partial,
                                             void* pieces, int64_t T, int64_t D, int64_t E, void* stream) {
  MI355_REQUIRE(aligned16(pieces) && (pieces || mi355_router_gate_fwd_kept_bytes(x_dtype, MI355_F32, T, D, E) == 0),
                "router_gate_fwd_keeping: aligned room for the weight pieces required");
  void* keep = mi355_router_gate_fwd_kept_bytes(x_dtype, MI355_F32, T, D, E) > 0 ? pieces : nullptr;
  return gate_fwd_partial(x, x_dtype, w, logit_bias, partial, pieces, keep, T, D, E, stream);
}

#define DISPATCH_VPL(E, ...)                           \
  do {                                                 \
    const int vpl_ = (int)(((E) + 63) / 64);           \
    if (vpl_ <= 1) { constexpr int VPL = 1; __VA_ARGS__; } \
    else if (vpl_ <= 2) { constexpr int VPL = 2; __VA_ARGS__; } \
    else if (vpl_ <= 4) { constexpr int VPL = 4; __VA_ARGS__; } \
    else { constexpr int VPL = 8; __VA_ARGS__; }       \
  } while (0)

extern "C" int mi355_router_select_fwd(const float* logits, const float* expert_bias,
                                       float* weights, int64_t* ids, float* scores_TE,
                                       uint8_t* routing_map_TE, int64_t T, int64_t E, int64_t K,
                                       int score_func, int route_norm, float route_scale, int num_groups,
                                       int num_limited, int select_mode, void* stream) {
  if (int rc = check_router_args(T, E, K)) return rc;
  MI355_REQUIRE(score_func >= 0 && score_func <= 2, "router_select_fwd: unknown score_func %d", score_func);
  MI355_REQUIRE(select_mode >= 0 && select_mode <= 2, "router_select_fwd: unknown select_mode %d", select_mode);
  MI355_REQUIRE(K <= 64, "router_select_fwd: top_k > 64 unsupported");
  if (num_groups > 0) {
    MI355_REQUIRE(num_groups <= 64 && E % num_groups == 0 && E / num_groups >= 2 &&
                      num_limited >= 1 && num_limited <= num_groups &&
                      K <= (int64_t)num_limited * (E / num_groups),
                  "router_select_fwd: bad group config G=%d L=%d", num_groups, num_limited);
  }
  if (T == 0) return MI355_OK;
  MI355_REQUIRE(logits && weights && ids, "router_select_fwd: null pointer");
  if (select_rows_ok(logits, scores_TE, routing_map_TE, E, K, num_groups, select_mode))
    return launch_select_rows({expert_bias, (int)E, (int)K, score_func, route_norm, route_scale, num_groups, num_limited},
                              logits, weights, ids, scores_TE, routing_map_TE, nullptr, T, as_stream(stream),
                              "router_select_fwd");
  const dim3 grid((unsigned)((T + 3) / 4));
  DISPATCH_VPL(E, hipLaunchKernelGGL(select_fwd_kernel<VPL>, grid, dim3(256), 0, as_stream(stream),
                                     logits, expert_bias, weights, ids, scores_TE, routing_map_TE,
                                     static_cast<float*>(nullptr), (int)T, (int)E, (int)K, score_func,
                                     route_norm, route_scale, num_groups, num_limited, select_mode));
  return check_launch("router_select_fwd");
}

extern "C" int mi355_router_select_cutoff_fwd(const float* logits, const float* expert_bias,
                                              float* weights, int64_t* ids, float* scores_TE,
                                              float* cutoff_T, int64_t T, int64_t E, int64_t K,
                                              int score_func, int route_norm, float route_scale,
                                              void* stream) {
  if (int rc = check_router_args(T, E, K)) return rc;
  MI355_REQUIRE(score_func >= 0 && score_func <= 2, "router_select_cutoff_fwd: unknown score_func %d", score_func);
  MI355_REQUIRE(K <= 64, "router_select_cutoff_fwd: top_k > 64 unsupported");
  MI355_REQUIRE(K < E, "router_select_cutoff_fwd: top_k (%lld) must leave a (K+1)-th expert of %lld",
                (long long)K, (long long)E);
  if (T == 0) return MI355_OK;
  MI355_REQUIRE(logits && weights && ids && cutoff_T, "router_select_cutoff_fwd: null pointer");
  if (select_rows_ok(logits, scores_TE, nullptr, E, K, 0, MI355_SELECT_TOPK))
    return launch_select_rows({expert_bias, (int)E, (int)K, score_func, route_norm, route_scale, 0, 0}, logits, weights,
                              ids, scores_TE, nullptr, cutoff_T, T, as_stream(stream), "router_select_cutoff_fwd");
  const dim3 grid((unsigned)((T + 3) / 4));
  DISPATCH_VPL(E, hipLaunchKernelGGL(select_fwd_kernel<VPL>, grid, dim3(256), 0, as_stream(stream),
                                     logits, expert_bias, weights, ids, scores_TE,
                                     static_cast<uint8_t*>(nullptr), cutoff_T, (int)T,
                                     (int)E, (int)K, score_func, route_norm, route_scale, 0, 0,
                                     MI355_SELECT_TOPK));
  return check_launch("router_select_cutoff_fwd");
}

static int select_bwd(const float* logits, const int64_t* ids, const float* dweights, const float* dscores_TE,
                      const DotPieces& dots, const BalanceGrad& bal, float* dlogits, int64_t T, int64_t E, int64_t K,
                      int score_func, int route_norm, float route_scale, int select_mode, void* stream) {
  if (int rc = check_router_args(T, E, K)) return rc;
  MI355_REQUIRE(K <= 64, "router_select_bwd: top_k > 64 unsupported");
  if (T == 0) return MI355_OK;
  MI355_REQUIRE(logits && ids && dlogits, "router_select_bwd: null pointer");
  const SelectBwd p{logits, ids, dweights, dscores_TE, dots, DotRows{}, bal, dlogits, (int)T, (int)E,
                    (int)K, score_func, route_norm, route_scale, select_mode};
  DISPATCH_VPL(E, hipLaunchKernelGGL(select_bwd_kernel<VPL>, dim3((unsigned)select_bwd_parts(p)), dim3(256), select_bwd_lds(E),
                                     as_stream(stream), p));
  return check_launch("router_select_bwd");
}

extern "C" int mi355_router_select_bwd(const float* logits, const int64_t* ids,
                                       const float* dweights, const float* dscores_TE,
                                       float* dlogits, int64_t T, int64_t E, int64_t K,
                                       int score_func, int route_norm, float route_scale,
                                       int select_mode, void* stream) {
  return select_bwd(logits, ids, dweights, dscores_TE, DotPieces{}, BalanceGrad{}, dlogits, T, E, K, score_func, route_norm,
                    route_scale, select_mode, stream);
}

extern "C" int mi355_router_select_dots_bwd(const float* logits, const int64_t* ids, const float* dots,
                                            int64_t pieces, const int32_t* row_of_slot, int64_t row_capacity,
                                            const float* aux_f_E, const float* aux_scale, const uint8_t* padding_mask_T,
                                            float* dlogits, int64_t T, int64_t E, int64_t K, int score_func,
                                            int route_norm, float route_scale, void* stream) {
  MI355_REQUIRE(pieces >= 0 && pieces <= 4096 && row_capacity >= 0 && row_capacity < (1ll << 31),
                "router_select_dots_bwd: bad shape");
  MI355_REQUIRE(T == 0 || (dots && (pieces == 0 || row_of_slot)), "router_select_dots_bwd: null pointer");
  MI355_REQUIRE(!aux_f_E || aux_scale, "router_select_dots_bwd: the loss needs its scale");
  return select_bwd(logits, ids, pieces ? nullptr : dots, nullptr,
                    pieces ? DotPieces{dots, row_of_slot, (int)pieces, (int)row_capacity} : DotPieces{},
                    BalanceGrad{aux_f_E, aux_scale, padding_mask_T}, dlogits, T, E, K, score_func, route_norm, route_scale,
                    MI355_SELECT_TOPK, stream);
}

extern "C" int mi355_router_select_rows_bwd(const float* logits, const int64_t* ids, const void* dout, const void* y, int dtype,
                                            const int32_t* row_of_slot, int64_t row_capacity, int64_t D, const float* aux_f_E,
                                            const float* aux_scale, const uint8_t* padding_mask_T, float* dlogits, int64_t T,
                                            int64_t E, int64_t K, int score_func, int route_norm, float route_scale,
                                            void* stream) {
  if (int rc = check_router_args(T, E, K)) return rc;
  MI355_REQUIRE(K <= 64, "router_select_rows_bwd: top_k > 64 unsupported");
  MI355_REQUIRE(dtype == MI355_F32 || dtype == MI355_BF16, "router_select_rows_bwd: fp32 or bf16 rows");
  MI355_REQUIRE(row_capacity >= 0 && row_capacity < (1ll << 31) && D >= 1 && D < (1ll << 31),
                "router_select_rows_bwd: bad shape");
  if (T == 0) return MI355_OK;
  MI355_REQUIRE(logits && ids && dlogits && dout && y && row_of_slot && aligned16({dout, y}),
                "router_select_rows_bwd: null or misaligned pointer");
  MI355_REQUIRE(!aux_f_E || aux_scale, "router_select_rows_bwd: the loss needs its scale");
  const SelectBwd p{logits, ids, nullptr, nullptr, DotPieces{}, DotRows{dout, y, row_of_slot, (int)D, (int)row_capacity},
                    BalanceGrad{aux_f_E, aux_scale, padding_mask_T}, dlogits, (int)T, (int)E, (int)K, score_func, route_norm,
                    route_scale, MI355_SELECT_TOPK};
  auto launch = [&](auto* kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)select_bwd_parts(p)), dim3(256), select_bwd_lds(E), as_stream(stream), p);
  };
  if (dtype == MI355_F32) { DISPATCH_VPL(E, launch(select_bwd_kernel<VPL, float>)); }
  else { DISPATCH_VPL(E, launch(select_bwd_kernel<VPL, uint16_t>)); }
  return check_launch("router_select_rows_bwd");
}
