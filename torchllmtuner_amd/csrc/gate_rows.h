// logits(T,E) = x(T,D) . W(E,D)^T for a tile of 32 tokens x 32 experts: by itself (router_gemm.hip) or in front of the
// selection (route.hip).
#pragma once
#include <type_traits>

#include "bf16_tiles.h"
#include "common.h"

namespace mi355 {

constexpr int R_BM = 32, R_BN = 32, R_WAVES = 8, R_STEP = 32;

// contraction per wave of one of `splits` slices
inline int gate_rows_k(int64_t D, int splits) {
  const int64_t per_wave = (D + splits * R_WAVES - 1) / (splits * R_WAVES);
  return (int)((per_wave + R_STEP - 1) / R_STEP * R_STEP);
}

namespace {

// 8 consecutive fp32 -> three 16-byte chunks of bf16 pieces (hi, mid, lo)
__device__ __forceinline__ void split8(const f32x4& a, const f32x4& b, u32x4& hi, u32x4& mid, u32x4& lo) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float v0 = i < 2 ? a[2 * i] : b[2 * i - 4], v1 = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
    float h0 = v0, h1 = v1;
    hi[i] = round_bf16x2(h0, h1);
    const float r0 = v0 - h0, r1 = v1 - h1;
    h0 = r0, h1 = r1;
    mid[i] = round_bf16x2(h0, h1);
    lo[i] = pack_bf16x2(r0 - h0, r1 - h1);
  }
}

template <typename TX>
__device__ __forceinline__ void load16_masked(const TX* p, int k, int k_end, f32x4 (&v)[4]) {
  // fp32: four pieces of four, each inside the row or zero (D % 4 == 0)
#pragma unroll
  for (int j = 0; j < 4; ++j)
    v[j] = k + 4 * j < k_end ? *reinterpret_cast<const f32x4*>(p + k + 4 * j) : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
}
__device__ __forceinline__ void load16_masked(const uint16_t* p, int k, int k_end, u32x4 (&v)[2]) {
#pragma unroll
  for (int j = 0; j < 2; ++j)
    v[j] = k + 8 * j < k_end ? *reinterpret_cast<const u32x4*>(p + k + 8 * j) : u32x4{0, 0, 0, 0};
}

// One slice of the contraction, by the 64 R_WAVES lanes of a workgroup (ends behind a barrier).  Lanes below 8 BN: the sum of
// token lane & 31 and the experts q * 8 + (lane >> 5) * 4 + 0..3 of the tile, q their wave.  BN below 32: the tile's first BN experts
// alone, the same sums in the same order (an element of the matrix instruction's result depends on its own row and column).
// KEEP: the first two pieces of the tile's weights are left at `keep`, E * D apart, unless that is null (bf16 tokens; D % 8 == 0).  (Another kernel: the test in the
// loop took 0.3 of the 24.1 us of a forward of one token.)
template <typename TX, int BN = R_BN, bool KEEP = false>
__device__ __forceinline__ f32x4 gate_rows_tile(const TX* __restrict__ x, const float* __restrict__ w, int T, int D, int E,
                                                int t0, int n0, int split, int k_per_wave, float (&red)[R_WAVES][4][64][4] /* wave, q, lane, i */,
                                                uint16_t* keep = nullptr) {
  constexpr bool BF = sizeof(TX) == 2;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int half = lane >> 5;
  const TX* xp = x + static_cast<int64_t>(min(t0 + (lane & 31), T - 1)) * D;
  const float* wp = w + static_cast<int64_t>(min(n0 + (lane & 31), E - 1)) * D;
  const int k0 = (split * R_WAVES + wave) * k_per_wave;
  const int k1 = min(k0 + k_per_wave, D);
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  const int w_end = (lane & 31) < BN ? k1 : 0;  // (what the other lanes hold is not read)
  constexpr int B = 4;  // steps requested together: 128 of the contraction, 24 KiB (bf16 x, 32 experts) per wave
  for (int kb = k0; kb < k1; kb += B * R_STEP) {
    f32x4 wv[B][4];
    std::conditional_t<BF, u32x4[B][2], f32x4[B][4]> xv;
#pragma unroll
    for (int b = 0; b < B; ++b) {
      const int k = kb + b * R_STEP + 16 * half;
      load16_masked(wp, k, w_end, wv[b]);
      load16_masked(xp, k, k1, xv[b]);
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
      if (kb + b * R_STEP >= k1) break;  // wave-uniform
      if constexpr (BF) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          u32x4 hi, mid, lo;
          split8(wv[b][2 * j], wv[b][2 * j + 1], hi, mid, lo);
          if (KEEP && keep) {
            const int k = kb + b * R_STEP + 16 * half + 8 * j, n = n0 + (lane & 31);
            if (k < w_end && n < E) {
              uint16_t* at = keep + static_cast<int64_t>(n) * D + k;
              *reinterpret_cast<u32x4*>(at) = hi;
              *reinterpret_cast<u32x4*>(at + static_cast<int64_t>(E) * D) = mid;
            }
          }
          const bf16x8 a = __builtin_bit_cast(bf16x8, xv[b][j]);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, hi), a, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, mid), a, acc, 0, 0, 0);
          acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, lo), a, acc, 0, 0, 0);
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[b][j][i], xv[b][j][i], acc, 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < BN / 8; ++q) {
    const f32x4 v = {acc[q * 4], acc[q * 4 + 1], acc[q * 4 + 2], acc[q * 4 + 3]};
    *reinterpret_cast<f32x4*>(red[wave][q][lane]) = v;
  }
  __syncthreads();
  const int q = (tid >> 6) & (BN / 8 - 1);
  f32x4 v = *reinterpret_cast<const f32x4*>(red[0][q][lane]);
#pragma unroll
  for (int i = 1; i < R_WAVES; ++i) v += *reinterpret_cast<const f32x4*>(red[i][q][lane]);
  return v;
}

}  // namespace
}  // namespace mi355
