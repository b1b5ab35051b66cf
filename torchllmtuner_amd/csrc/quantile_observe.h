// The required-bias histogram through LDS, a workgroup's part of it, for the kernel of quantile.hip and for the plan's second
// launch (route.hip), which has CUs to spare and the scores.
#pragma once
#include "common.h"

namespace mi355 {

// min and max of bias[0..E) in every thread of a workgroup of LANES; red: 2 LANES / 64 floats of LDS
template <int LANES>
__device__ __forceinline__ void bias_range(const float* __restrict__ bias, int E, float* red, float& mn, float& mx) {
  constexpr int W = LANES / kWave;
  float lo = INFINITY, hi = -INFINITY;
  for (int e = threadIdx.x; e < E; e += LANES) {
    lo = fminf(lo, bias[e]);
    hi = fmaxf(hi, bias[e]);
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o, kWave));
    hi = fmaxf(hi, __shfl_xor(hi, o, kWave));
  }
  if ((threadIdx.x & (kWave - 1)) == 0) {
    red[threadIdx.x / kWave] = lo;
    red[W + threadIdx.x / kWave] = hi;
  }
  __syncthreads();
  mn = red[0];
  mx = red[W];
#pragma unroll
  for (int w = 1; w < W; ++w) {
    mn = fminf(mn, red[w]);
    mx = fmaxf(mx, red[W + w]);
  }
}

// scores (T, E), cutoff (T), padding (T) or null, hist (E, B); a workgroup has `eg` neighbouring experts and a run of `tokens` tokens
struct Observe {
  const float *scores, *cutoff, *bias;
  const uint8_t* padding;
  unsigned long long* hist;
  int T, E, B, eg, tokens;
};

// How the pairs are dealt: experts a workgroup (what 32 KiB of LDS bins hold, at most 4, for more workgroups) and tokens; about 256 workgroups,
// each with at least 256 tokens so that the LDS bins pay off.  eg = 0: not through LDS.
inline void observe_shape(int64_t T, int64_t E, int64_t B, int& eg, int& tokens, unsigned& groups, unsigned& chunks) {
  eg = T >= 256 ? static_cast<int>(std::min<int64_t>(std::min<int64_t>(4, E), (32 * 1024) / (B * 4))) : 0;
  tokens = 0, groups = chunks = 0;
  if (eg < 1) return;
  groups = static_cast<unsigned>((E + eg - 1) / eg);
  const int64_t n = std::max<int64_t>(1, std::min<int64_t>(T / 256, (256 + groups - 1) / groups));
  tokens = static_cast<int>((T + n - 1) / n);
  chunks = static_cast<unsigned>((T + tokens - 1) / tokens);
}

// A workgroup owns `eg` neighbouring experts and a run of tokens, counts their pairs in 32-bit LDS bins (a call adds fewer
// than 2^31 pairs to a bin) and then adds its non-empty bins to the 64-bit histogram.  The required biases of
// one expert cluster in a few dozen bins, so this replaces most of the global atomics, which queue up on those few addresses, by LDS ones.
// bins: eg * B words of LDS; red as above.
template <int LANES>
__device__ __forceinline__ void observe_part(const Observe& o, int group, int chunk, unsigned* bins, float* red) {
#pragma clang fp contract(off)
  float mn, mx;
  bias_range<LANES>(o.bias, o.E, red, mn, mx);
  const float lower = mn - 1.0f;
  const float width = ((mx - mn) + 2.0f) / static_cast<float>(o.B);
  const float top = static_cast<float>(o.B - 1);
  const int e0 = group * o.eg;
  const int ne = min(o.eg, o.E - e0);
  const int t0 = chunk * o.tokens;
  const int nt = min(o.tokens, o.T - t0);
  for (int i = threadIdx.x; i < o.eg * o.B; i += LANES) bins[i] = 0u;
  __syncthreads();
  for (int i = threadIdx.x; i < nt * o.eg; i += LANES) {
    const int t = t0 + i / o.eg, j = i % o.eg;
    if (j >= ne || (o.padding && o.padding[t])) continue;
    const float required = o.cutoff[t] - o.scores[static_cast<int64_t>(t) * o.E + e0 + j];
    float q = floorf((required - lower) / width);
    q = fminf(fmaxf(q, 0.0f), top);
    atomicAdd(bins + j * o.B + static_cast<int>(q), 1u);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < ne * o.B; i += LANES) {
    const unsigned c = bins[i];
    if (c) atomicAdd(o.hist + static_cast<int64_t>(e0) * o.B + i, static_cast<unsigned long long>(c));
  }
}

}  // namespace mi355
