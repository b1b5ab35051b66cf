// Both gradients of a router gate of up to 32 experts (by themselves 64), as parts of launches: by themselves (router_gemm.hip), or the weight's beside
// the experts' products (grouped_any.hip) and the input's together with the sum over a token's rows.
//   dW = dlogits^T . x and dx = dlogits . W read or write a (T, D) matrix against a handful of rows, too thin for
// matrix tiles, and the vector units keep up with memory.  A thread owns four columns.  dW parts: eight experts,
// 256 columns and a slice of the tokens, the four waves on every fourth token, joined through LDS in wave
// order; the slices' sums are added by whoever comes next.  dx parts: 32 tokens x 256 columns, dlogits in LDS.
// 1531 tokens, 320 x 16, bf16: 12 us with the sum, 47 with strided GEMMs.
#pragma once
#include "bf16_tiles.h"
#include "common.h"

namespace mi355 {

constexpr int S_EB = 8, S_COLS = 256, S_TOK = 32, S_MAX_E = 32;

struct GateDw {
  const float* dlogits;
  const void* x;
  float* partial;  // (splits, E, D)
  int T, D, E, splits, rows_per_split;
};
// of the dW parts: how many, and the slices of the tokens -- about two parts per CU, at least 32 tokens each
inline int gate_dw_splits(int64_t T, int64_t D, int64_t E) {
  const int64_t tiles = ((D + S_COLS - 1) / S_COLS) * ((E + S_EB - 1) / S_EB);
  int64_t s = 512 / tiles;
  if ((T + 31) / 32 < s) s = (T + 31) / 32;
  if (s > 64) s = 64;
  return static_cast<int>(s < 1 ? 1 : s);
}
inline GateDw gate_dw_job(const float* dlogits, const void* x, float* partial, int64_t T, int64_t D, int64_t E) {
  const int splits = gate_dw_splits(T, D, E);
  return {dlogits, x, partial, (int)T, (int)D, (int)E, splits, (int)((T + splits - 1) / splits)};
}
inline int64_t gate_dw_parts(const GateDw& j) {
  return (int64_t)((j.D + S_COLS - 1) / S_COLS) * j.splits * ((j.E + S_EB - 1) / S_EB);
}

namespace {

__device__ __forceinline__ f32x4 load_cols(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 load_cols(const uint16_t* p) {
  const u32x2 v = *reinterpret_cast<const u32x2*>(p);
  return {__uint_as_float(v[0] << 16), __uint_as_float(v[0] & 0xffff0000u), __uint_as_float(v[1] << 16),
          __uint_as_float(v[1] & 0xffff0000u)};
}
__device__ __forceinline__ void store_cols(float* p, const f32x4& v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void store_cols(uint16_t* p, const f32x4& v) {
  *reinterpret_cast<u32x2*>(p) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

// one dW part, 256 lanes; lds: S_EB / 2 experts of the four waves, 16 KiB
constexpr int kGateDwLds = 4 * (S_EB / 2) * S_COLS;
template <typename TX>
__device__ __forceinline__ void gate_dw_part(const GateDw& j, int part, float* lds) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int D = j.D, E = j.E, col_blocks = (D + S_COLS - 1) / S_COLS;
  const TX* x = static_cast<const TX*>(j.x);
  const int cb = part % col_blocks, rest = part / col_blocks, split = rest % j.splits, e0 = rest / j.splits * S_EB;
  const int n = min(cb * S_COLS + lane * 4, D - 4);  // (D % 4 == 0; lanes past the end repeat the last columns)
  const int t0 = split * j.rows_per_split, t1 = min(j.T, t0 + j.rows_per_split);
  f32x4 acc[S_EB];
#pragma unroll
  for (int e = 0; e < S_EB; ++e) acc[e] = f32x4{0, 0, 0, 0};
  constexpr int U = 4;  // tokens requested together
  for (int t = t0 + wave; t < t1; t += 4 * U) {
    f32x4 xv[U];
    float dl[U][S_EB];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int tt = t + 4 * u;
      const bool live = tt < t1;
      xv[u] = load_cols(x + static_cast<int64_t>(live ? tt : t) * D + n);
#pragma unroll
      for (int e = 0; e < S_EB; ++e)
        dl[u][e] = live && e0 + e < E ? j.dlogits[static_cast<int64_t>(tt) * E + e0 + e] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < S_EB; ++e)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[e][i] = fmaf(dl[u][e], xv[u][i], acc[e][i]);
  }
  constexpr int H = S_EB / 2;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    if (half) __syncthreads();
#pragma unroll
    for (int e = 0; e < H; ++e) *reinterpret_cast<f32x4*>(lds + (wave * H + e) * S_COLS + lane * 4) = acc[half * H + e];
    __syncthreads();
    const int e = e0 + half * H + wave;
    f32x4 v = *reinterpret_cast<const f32x4*>(lds + wave * S_COLS + lane * 4);
#pragma unroll
    for (int w = 1; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(lds + (w * H + wave) * S_COLS + lane * 4);
    if (e < E && cb * S_COLS + lane * 4 < D)
      store_cols(j.partial + (static_cast<int64_t>(split) * E + e) * D + cb * S_COLS + lane * 4, v);
  }
}

}  // namespace
}  // namespace mi355
