// Rows 16 bytes at a time, for the kernels that give a token a wave: a piece as fp32 values, and the dot products of a
// token's output gradient with its experts' rows.
#pragma once
#include "common.h"

namespace mi355 {
namespace {

template <typename T>
struct Vec {
  static constexpr int N = 16 / sizeof(T);
  __device__ static void unpack(const uint4& v, float (&f)[N]);
  __device__ static uint4 pack(const float (&f)[N]);
};
template <>
__device__ inline void Vec<float>::unpack(const uint4& v, float (&f)[4]) {
  f[0] = __uint_as_float(v.x); f[1] = __uint_as_float(v.y);
  f[2] = __uint_as_float(v.z); f[3] = __uint_as_float(v.w);
}
template <>
__device__ inline uint4 Vec<float>::pack(const float (&f)[4]) {
  return make_uint4(__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]),
                    __float_as_uint(f[3]));
}
template <>
__device__ inline void Vec<uint16_t>::unpack(const uint4& v, float (&f)[8]) {
  f[0] = __uint_as_float(v.x << 16); f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16); f[3] = __uint_as_float(v.y & 0xffff0000u);
  f[4] = __uint_as_float(v.z << 16); f[5] = __uint_as_float(v.z & 0xffff0000u);
  f[6] = __uint_as_float(v.w << 16); f[7] = __uint_as_float(v.w & 0xffff0000u);
}
template <>
__device__ inline uint4 Vec<uint16_t>::pack(const float (&f)[8]) {
  return make_uint4(pack_bf16x2(f[0], f[1]), pack_bf16x2(f[2], f[3]), pack_bf16x2(f[4], f[5]),
                    pack_bf16x2(f[6], f[7]));
}

// <g, y[row of slot k]> for the K <= 64 slots of one token, by one wave: lane k receives slot k's (zero without a row),
// `row` is lane k's row or negative.  The products are added in the order of combine_bwd_kernel, which
// writes the scaled gradient rows besides: the same bits.  Four rows are requested together.
template <typename T>
__device__ __forceinline__ float row_dots(const T* __restrict__ g, const T* __restrict__ y, int row, int K, int D) {
  const int lane = threadIdx.x & 63;
  constexpr int V = Vec<T>::N, G = 4, B = 4;
  float my_dot = 0.0f;
  if (D % V == 0) {
    const int nv = D / V;
    for (int base = 0; base < nv; base += G * kWave) {
      float gf[G][V];
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const int i = base + q * kWave + lane;
        Vec<T>::unpack(i < nv ? reinterpret_cast<const uint4*>(g)[i] : make_uint4(0, 0, 0, 0), gf[q]);
      }
      for (int k0 = 0; k0 < K; k0 += B) {
        uint4 v[B][G];
        int r[B];
#pragma unroll
        for (int j = 0; j < B; ++j) {
          r[j] = k0 + j < K ? __builtin_amdgcn_readlane(row, min(k0 + j, 63)) : -1;
          const uint4* src = reinterpret_cast<const uint4*>(y + static_cast<int64_t>(max(r[j], 0)) * D);
#pragma unroll
          for (int q = 0; q < G; ++q) {
            const int i = base + q * kWave + lane;
            v[j][q] = r[j] >= 0 && i < nv ? load_stream(src + i) : make_uint4(0, 0, 0, 0);
          }
        }
#pragma unroll
        for (int j = 0; j < B; ++j) {
          if (r[j] < 0) continue;  // wave-uniform
          float dot = 0.0f;
#pragma unroll
          for (int q = 0; q < G; ++q) {
            float yf[V];
            Vec<T>::unpack(v[j][q], yf);
#pragma unroll
            for (int c = 0; c < V; ++c) dot += yf[c] * gf[q][c];
          }
          dot = wave_sum(dot);
          if (lane == k0 + j) my_dot += dot;
        }
      }
    }
  } else {
    for (int k = 0; k < K; ++k) {
      const int r = __builtin_amdgcn_readlane(row, k);
      if (r < 0) continue;
      const T* yr = y + static_cast<int64_t>(r) * D;
      float dot = 0.0f;
      for (int i = lane; i < D; i += kWave) dot += load_as_f32(yr + i) * load_as_f32(g + i);
      dot = wave_sum(dot);
      if (lane == k) my_dot = dot;
    }
  }
  return my_dot;
}

}  // namespace
}  // namespace mi355
