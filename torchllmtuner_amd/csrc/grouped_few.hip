// Forward expert products for a handful of rows per expert (generation: one token to a few dozen).
//
// Such a product is one read of the touched experts' weights and nothing else: a weight row meets at
// most 16 activation rows, so no operand is worth staging.  The 256-row kernels of grouped_bf16.hip
// stream the same weights through LDS in 1 MB work items, one workgroup per CU in lockstep: at one
// token 48 items for 256 CUs, at 33 tokens 2.6 rounds of them.  Here a workgroup is four waves that
// split the contraction of 16 output columns (of gate and up, or 32 of the down projection) of one
// expert; every wave loads its weights straight into MFMA fragments, 16 KiB requested ahead, up
// to sixteen waves to a CU, and the four partial tiles are added in wave order through LDS.
//   Bound by HBM: 709 MB of gate and up weights (33 tokens of 128 experts, 2048 x 768) in 116 us, 6.1 TB/s
// where a plain read in this pattern reaches 6.15 (145 us before); one token, 50 MB, 13 us (31 before).
// Waves along the contraction rather than side by side: at one token 12-25 us less in all, at 33 the
// same.  32 or 64 rows per wave instead of 16 need registers that the requests in flight want: slower.
//   A contraction step is 64 wide: lane group g = lane / 16 holds k = 16 g .. 16 g + 15 of it (two
// 16-byte loads, so that a row's 128 bytes are one request) for both operands alike.
#include <algorithm>

#include "bf16_tiles.h"
#include "common.h"

namespace mi355 {
namespace {

struct FewArgs {
  const uint16_t* a;     // GATEUP: rows or (with a_src) tokens, K wide; else h
  const int32_t* a_src;  // row -> row of a, or null
  int a_rows;
  const uint16_t *b0, *b1;  // (El, N, K) each; DOWN: b1 = b0
  uint16_t *gate, *up, *out;  // gate, up may be null
  const int32_t *seg_offsets, *seg_counts, *tile_expert, *tile_row0, *num_tiles;
  int K, N, col_groups;
};

__device__ __forceinline__ float few_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

// raw buffer resource over a wave-uniform base: a 32-bit offset per lane and a scalar one per step
__device__ __forceinline__ __amdgpu_buffer_rsrc_t few_rsrc(const void* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, -1, 0x00020000);
}

template <bool GATEUP>
__global__ __launch_bounds__(256, 4) void few_rows_kernel(FewArgs p) {
  constexpr int kPairs = 4;  // 64-wide contraction steps requested together
  __shared__ f32x4 part[4][2][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int t = blockIdx.x / p.col_groups, cg = blockIdx.x - t * p.col_groups;
  if (t >= *p.num_tiles) return;
  const int e = __builtin_amdgcn_readfirstlane(p.tile_expert[t]), row0 = __builtin_amdgcn_readfirstlane(p.tile_row0[t]);
  const int cnt = p.seg_counts[e], seg0 = p.seg_offsets[e];
  const int rows = min(even_tile_rows(cnt, 256), seg0 + cnt - row0);
  const int K = p.K, N = p.N;
  // this wave's share of the contraction
  const int steps = K >> 6, s0 = steps * wave >> 2, s1 = steps * (wave + 1) >> 2;
  // weight rows: 16 columns of gate and the same of up, or 32 columns of the one matrix (N % 32 == 0)
  const int n0 = cg * (GATEUP ? 16 : 32);
  const int64_t we = static_cast<int64_t>(e) * N * K;
  const auto rs0 = few_rsrc(p.b0 + we), rs1 = few_rsrc(p.b1 + we), rsA = few_rsrc(p.a);
  const uint32_t off0 = static_cast<uint32_t>((n0 + r16) * K + g * 16) * 2u;
  const uint32_t off1 = GATEUP ? off0 : off0 + static_cast<uint32_t>(32 * K);
  for (int sub = 0; sub < rows; sub += 16) {
    const int row = row0 + min(sub + r16, rows - 1);
    const int index = p.a_src ? p.a_src[row] : row;
    f32x4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    u32x4 b0[kPairs][2], b1[kPairs][2], a[kPairs][2];
    uint32_t offA;
    auto request_w = [&](int i, int step) {
      const int k = step * 128;  // bytes
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        b0[i][h] = __builtin_amdgcn_raw_buffer_load_b128(rs0, off0 + 16 * h, k, 0);
        b1[i][h] = __builtin_amdgcn_raw_buffer_load_b128(rs1, off1 + 16 * h, k, 0);
      }
    };
    auto request_a = [&](int i, int step) {
#pragma unroll
      for (int h = 0; h < 2; ++h) a[i][h] = __builtin_amdgcn_raw_buffer_load_b128(rsA, offA + 16 * h, step * 128, 0);
    };
    auto multiply = [&](int i) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const bf16x8 af = __builtin_bit_cast(bf16x8, a[i][h]);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b0[i][h]), af, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, b1[i][h]), af, acc1, 0, 0, 0);
      }
    };
    // the first weights go out before the row's index is back (past the end: the last step again, not used)
#pragma unroll
    for (int i = 0; i < kPairs; ++i) request_w(i, min(s0 + i, s1 - 1));
    __builtin_amdgcn_sched_barrier(0);
    const int src = p.a_src ? min(max(index, 0), p.a_rows - 1) : row;
    offA = (static_cast<uint32_t>(src) * static_cast<uint32_t>(K) + g * 16) * 2u;
#pragma unroll
    for (int i = 0; i < kPairs; ++i) request_a(i, min(s0 + i, s1 - 1));
    int s = s0;
    for (; s + 2 * kPairs <= s1; s += kPairs) {
#pragma unroll
      for (int i = 0; i < kPairs; ++i) {
        multiply(i);
        request_w(i, s + kPairs + i);
        request_a(i, s + kPairs + i);
      }
    }
    // at most 2 kPairs - 1 steps are left, kPairs of them requested
#pragma unroll
    for (int i = 0; i < kPairs; ++i) {
      if (s + i < s1) multiply(i);
      if (s + kPairs + i < s1) {
        request_w(i, s + kPairs + i);
        request_a(i, s + kPairs + i);
      }
    }
#pragma unroll
    for (int i = 0; i < kPairs; ++i)
      if (s + kPairs + i < s1) multiply(i);
    part[wave][0][lane] = acc0;
    part[wave][1][lane] = acc1;
    __syncthreads();
    // lane = activation row lane & 15, its four values = columns 4 g .. 4 g + 3 of a 16-column tile
    auto sum = [&](int tile) {
      f32x4 v = part[0][tile][lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) v += part[w][tile][lane];
      return v;
    };
    if (wave < (GATEUP ? 1 : 2) && sub + r16 < rows) {
      const int64_t at = static_cast<int64_t>(row) * N + n0 + 16 * wave + 4 * g;
      if constexpr (GATEUP) {
        const f32x4 v = sum(0), u = sum(1);
        float gv[4], uv[4], hv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          gv[i] = round_bf16(v[i]);
          uv[i] = round_bf16(u[i]);
          hv[i] = round_bf16(gv[i] * few_sigmoid(gv[i])) * uv[i];
        }
        if (p.gate) {
          *reinterpret_cast<u32x2*>(p.gate + at) = u32x2{pack2(gv[0], gv[1]), pack2(gv[2], gv[3])};
          *reinterpret_cast<u32x2*>(p.up + at) = u32x2{pack2(uv[0], uv[1]), pack2(uv[2], uv[3])};
        }
        *reinterpret_cast<u32x2*>(p.out + at) = u32x2{pack2(hv[0], hv[1]), pack2(hv[2], hv[3])};
      } else {
        const f32x4 v = sum(wave);
        *reinterpret_cast<u32x2*>(p.out + at) = u32x2{pack2(v[0], v[1]), pack2(v[2], v[3])};
      }
    }
    if (sub + 16 < rows) __syncthreads();
  }
}

}  // namespace

// gate/up (stage 1) or down (stage 2) of the forward; the arguments of bf16_grouped_fwd.
int few_rows_fwd(int stage, const void* a, const int32_t* a_src, int64_t a_rows, const void* b0, const void* b1,
                 void* gate, void* up, void* out, const int32_t* seg_offsets, const int32_t* seg_counts,
                 const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* num_tiles, int64_t tiles, int64_t K,
                 int64_t N, hipStream_t s) {
  FewArgs p{};
  p.a = (const uint16_t*)a; p.a_src = a_src; p.a_rows = (int)a_rows;
  p.b0 = (const uint16_t*)b0; p.b1 = (const uint16_t*)b1;
  p.gate = (uint16_t*)gate; p.up = (uint16_t*)up; p.out = (uint16_t*)out;
  p.seg_offsets = seg_offsets; p.seg_counts = seg_counts; p.tile_expert = tile_expert; p.tile_row0 = tile_row0;
  p.num_tiles = num_tiles; p.K = (int)K; p.N = (int)N;
  p.col_groups = (int)(N / (stage == 1 ? 16 : 32));
  const dim3 grid((unsigned)(tiles * p.col_groups));
  if (stage == 1) hipLaunchKernelGGL(few_rows_kernel<true>, grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL(few_rows_kernel<false>, grid, dim3(256), 0, s, p);
  return check_launch("grouped forward, few rows");
}

}  // namespace mi355
