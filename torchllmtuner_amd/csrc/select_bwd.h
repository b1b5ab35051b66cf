// The selection's backward, as parts of launches: by itself (router.hip), or beside the experts' dH (grouped_any.hip).
#pragma once
#include <type_traits>

#include "common.h"
#include "row_vec.h"
#include "select_rows.h"

namespace mi355 {
namespace {

template <int VPL>
__device__ __forceinline__ void compute_scores(const float* __restrict__ row, int E, int lane,
                                               int score_func, float (&s)[VPL], float (&x)[VPL]) {
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int e = lane + j * kWave;
    x[j] = e < E ? row[e] : -INFINITY;
  }
  if (score_func == MI355_SCORE_SOFTMAX) {
    float m = x[0];
#pragma unroll
    for (int j = 1; j < VPL; ++j) m = fmaxf(m, x[j]);
    m = wave_max_dpp(m);
    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      s[j] = (lane + j * kWave < E) ? expf(x[j] - m) : 0.0f;
      sum += s[j];
    }
    sum = wave_sum_dpp(sum);
#pragma unroll
    for (int j = 0; j < VPL; ++j) s[j] = s[j] / sum;
  } else if (score_func == MI355_SCORE_SIGMOID) {
#pragma unroll
    for (int j = 0; j < VPL; ++j) s[j] = 1.0f / (1.0f + expf(-x[j]));
  } else {
#pragma unroll
    for (int j = 0; j < VPL; ++j) s[j] = sqrtf(softplus_f32(x[j]));
  }
}

// The weights' gradient as the folded expert backward leaves it: the sum, in order, of `pieces`
// partial dot products of the slot's row (zero for a slot without one).  Added up here, by the one
// reader, instead of by a launch of its own.
struct DotPieces {
  const float* partial;  // (rows, pieces) or null: dweights holds the sums
  const int32_t* row_of_slot;
  int pieces, rows;
};
__device__ __forceinline__ float slot_dweight(const DotPieces& d, const float* dweights, int64_t slot) {
  if (!d.partial) return dweights[slot];
  const int row = d.row_of_slot[slot];
  float sum = 0.0f;
  if (row >= 0 && row < d.rows)
    for (int i = 0; i < d.pieces; ++i) sum += d.partial[static_cast<int64_t>(row) * d.pieces + i];
  return sum;
}

// ... or as nothing has left it yet: the output gradient and the experts' rows, whose dot products the wave of the token
// forms itself (T of the kernel below; void: no such rows).
struct DotRows {
  const void *dout, *y;
  const int32_t* row_of_slot;
  int D, rows;
};

// The load-balance loss's part of the score gradient (aux.hip's formula), for the tokens that are not padding.
struct BalanceGrad {
  const float* f;  // (E) or null: no loss
  const float* scale;
  const uint8_t* padding;
};

struct SelectBwd {
  const float* logits;
  const int64_t* ids;
  const float *dweights, *dscores;
  DotPieces dots;
  DotRows rows;
  BalanceGrad bal;
  float* dlogits;
  int T, E, K, score_func, route_norm;
  float route_scale;
  int mode;
};
inline int64_t select_bwd_parts(const SelectBwd& p) { return (static_cast<int64_t>(p.T) + 3) / 4; }
inline size_t select_bwd_lds(int64_t E) { return 4 * 2 * E * sizeof(float); }

// Four tokens, a wave each; lds: per wave sc[E], ds[E].
template <int VPL, typename T>
__device__ __forceinline__ void select_bwd_part(const SelectBwd& p, int part, float* lds) {
  const float* __restrict__ logits = p.logits;
  const int64_t* __restrict__ ids = p.ids;
  const float* __restrict__ dweights = p.dweights;
  const float* __restrict__ dscores = p.dscores;
  float* __restrict__ dlogits = p.dlogits;
  const DotPieces& dots = p.dots;
  const DotRows& rows = p.rows;
  const BalanceGrad& bal = p.bal;
  const int T_ = p.T, E = p.E, K = p.K, score_func = p.score_func, route_norm = p.route_norm, mode = p.mode;
  const float route_scale = p.route_scale;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t_raw = part * 4 + wave;
  const bool active = t_raw < T_;
  const int t = active ? t_raw : T_ - 1;  // inactive waves shadow the last token, store nothing
  float* sc = lds + static_cast<size_t>(wave) * 2 * E;
  float* ds = sc + E;

  const float* row = logits + static_cast<int64_t>(t) * E;
  float s[VPL];
  float xs[VPL];
  compute_scores<VPL>(row, E, lane, score_func, s, xs);
  float bal_mean = 0.0f, bal_inv = 0.0f;
  if (bal.f && !(bal.padding && bal.padding[t])) {
    float sum = 0.0f, dot = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int e = lane + j * kWave;
      sum += e < E ? s[j] : 0.0f;
      dot += e < E ? s[j] * bal.f[e] : 0.0f;
    }
    sum = wave_sum_dpp(sum);
    dot = wave_sum_dpp(dot);
    // below the clamp the normalised score is s / eps and the sum no longer enters
    const float inv = 1.0f / fmaxf(sum, 1e-12f);
    bal_mean = sum < 1e-12f ? 0.0f : dot * inv;
    bal_inv = *bal.scale * inv;
  }
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int e = lane + j * kWave;
    if (e < E) {
      sc[e] = s[j];
      float d = dscores ? dscores[static_cast<int64_t>(t) * E + e] : 0.0f;
      if (bal.f) d += (bal.f[e] - bal_mean) * bal_inv;
      ds[e] = d;
    }
  }
  __syncthreads();

  constexpr bool kRows = !std::is_void_v<T>;
  if (mode != MI355_SELECT_FIXED && (kRows || dweights || dots.partial)) {
    // lanes 0..K-1 own one selected expert each (K <= 64)
    int id = lane < K ? static_cast<int>(ids[static_cast<int64_t>(t) * K + lane]) : 0;
    id = min(max(id, 0), E - 1);
    const float sk = lane < K ? sc[id] : 0.0f;
    float dw;
    if constexpr (kRows) {
      const int row = lane < K ? rows.row_of_slot[static_cast<int64_t>(t) * K + lane] : -1;
      dw = row_dots<T>(static_cast<const T*>(rows.dout) + static_cast<int64_t>(t) * rows.D, static_cast<const T*>(rows.y),
                       row < rows.rows ? row : -1, K, rows.D);
    } else {
      dw = lane < K ? slot_dweight(dots, dweights, static_cast<int64_t>(t) * K + lane) : 0.0f;
    }
    float g;
    if (route_norm) {
      const float denom = wave_sum_dpp(sk) + 1e-20f;
      const float dot = wave_sum_dpp(dw * sk);
      g = route_scale * (dw / denom - dot / (denom * denom));
    } else {
      g = route_scale * dw;
    }
    // scatter-add into the dense score gradient, serially so a repeated id adds up
    for (int k = 0; k < K; ++k) {
      const int idk = __builtin_amdgcn_readlane(id, k);
      const float gk = lane_f32(g, k);
      if (lane == 0) ds[idk] += gk;
    }
  }
  __syncthreads();

  float d[VPL];
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int e = lane + j * kWave;
    d[j] = e < E ? ds[e] : 0.0f;
  }
  if (score_func == MI355_SCORE_SOFTMAX) {
    float dot = 0.0f;
#pragma unroll
    for (int j = 0; j < VPL; ++j) dot += (lane + j * kWave < E) ? s[j] * d[j] : 0.0f;
    dot = wave_sum_dpp(dot);
#pragma unroll
    for (int j = 0; j < VPL; ++j) d[j] = s[j] * (d[j] - dot);
  } else if (score_func == MI355_SCORE_SIGMOID) {
#pragma unroll
    for (int j = 0; j < VPL; ++j) d[j] = d[j] * s[j] * (1.0f - s[j]);
  } else {
#pragma unroll
    for (int j = 0; j < VPL; ++j) {
      const int e = lane + j * kWave;
      const float x = e < E ? row[e] : 0.0f;
      const float sig = 1.0f / (1.0f + expf(-x));
      const float dsp = x > 20.0f ? 1.0f : sig;  // d softplus / dx
      d[j] = s[j] > 0.0f ? d[j] * dsp / (2.0f * s[j]) : 0.0f;
    }
  }
#pragma unroll
  for (int j = 0; j < VPL; ++j) {
    const int e = lane + j * kWave;
    if (e < E && active) dlogits[static_cast<int64_t>(t) * E + e] = d[j];
  }
}

}  // namespace
}  // namespace mi355
