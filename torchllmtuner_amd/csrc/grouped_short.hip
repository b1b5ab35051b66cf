// Forward expert products of a dozen to some dozens of rows per expert: a batch of generation, a short prompt, an expert-parallel
// rank's share of either.
//
// Such a product is still one read of the touched experts' weights, but a weight row meets up to 64 or 128 activation rows, so the
// rows are worth sharing.  A workgroup is four waves side by side over 64 columns of gate and of up (or 128 of the down projection): each
// wave streams its own 32 weight rows through LDS, two contraction steps of 64 ahead, and all read the tile's rows there.  Two steps of 64
// (128) rows and the weights are 48 (64) KiB, so three (two) workgroups fit a CU and fill each other's gaps: lookups, first operands,
// barriers, ends.  The 256-row kernels have one workgroup to a CU, whose 2 to 12 us of those per tile nothing fills: at few rows they
// are a fifth of the launch.  grouped_few.hip, 16 rows a pass, reads the weights again for every 16.
//   An expert of more rows has as many passes, workgroups of their own that read the same weights side by side, from L2: with the passes one after the other in one
// workgroup a router that prefers some experts made a training step of 300 tokens of the first block below 10 % longer (805 us for 735; 722 now).
//   Where they are chosen: grouped_bf16.hip (many rows of few experts want the row tiles, which these loads do not have).
//   Bound by HBM: block forward of three sets of weights in turn, us, row tiles / 64-row passes / 128-row passes.  128 experts of 2048 x 768, eight a
// token, 200 tokens 219 / 214 / 212, 500 239 / 232 / 235 (1.2 GB of weights in 190), 700 250 / 245 / 249, 1000 261 / 300 / 267; 64 of 1024 x 512, six each, 300 71 / 65 / 66;
// 60 of 1728 x 960, six each, 120 130 / 121 / 124, 300 135 / 128 / 131, 450 143 / 137 / 142; 16 of 2048 x 1024, four each, 48 68 / 60 / 60, 180 72 / 64 / 65; 16 of 512 x
// 384 32 / 28 / 29, 34 / 30 / 32; 32 of 256 of 7168 x 2048, eight each, 80 382 / 319, 128 402 / 347, 256 420 / 411 / 422, 430 451 / 455 / 455, 512 455 / 461 / 470.  The few-row
// kernels / these: 64 tokens of the last 305 / 322, 100 325 / 327; 40 and 100 of the first 193 / 196, 211 / 208; 60 of the third 116 / 120.
// 32 rows a pass bring nothing more, 96 the same as 128; a third step of weights in LDS 1-2 % slower.
#include <algorithm>
#include <type_traits>

#include "bf16_tiles.h"
#include "common.h"
#include "tile_list.h"

namespace mi355 {
namespace {

struct ShortArgs {
  const uint16_t* a;     // GATEUP: rows or (with a_src) tokens, K wide; else h
  const int32_t* a_src;  // row -> row of a, or null
  int a_rows;
  const uint16_t *b0, *b1;    // (El, N, K) each; DOWN: b1 = b0
  uint16_t *gate, *up, *out;  // gate, up may be null
  const int32_t *seg_offsets, *seg_counts;
  TileList list;
  int El, K, N, col_groups, last_row;  // last_row: of the row arrays
  int turn;    // a workgroup's contraction starts at a step of its own
  int stream;  // weights that one pass alone reads: with the non-temporal hint
};

__device__ __forceinline__ float short_sigmoid(float x) { return __builtin_amdgcn_rcpf(1.0f + __expf(-x)); }

typedef const int32_t __attribute__((address_space(4))) * const_i32;

constexpr int short_lds(int RB) { return 2 * (RB * 2048 + 16384); }

template <bool GATEUP, int RB>
__global__ __launch_bounds__(256, RB > 4 ? 2 : 3) void short_rows_kernel(ShortArgs p) {
  constexpr int NA = RB / 2, NB = 4;  // requests of a wave for one contraction step
  constexpr int ROWS = 16 * RB;       // of a pass
  constexpr uint32_t A_STAGE = RB * 2048, B_STAGE = 16384, B_AT = 2 * A_STAGE;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_cptr)smem));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int K = p.K, N = p.N, steps = K >> 6;
  // Which expert, pass and columns: every wave adds up the experts' passes itself, from one load of their counts (a list in memory would be a second one behind
  // it, and both stand in front of the first weights).  An XCD has a run of (expert, column group, pass): passes that share weights are neighbours in
  // one L2, and so are an expert's column groups, which share its rows.
  int count[4], to[4], total = 0, unlisted = -p.list.size();
#pragma unroll
  for (int b = 0; b < 4; ++b) count[b] = 64 * b + lane < p.El ? p.seg_counts[64 * b + lane] : 0;
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    to[b] = total + wave_scan((count[b] + ROWS - 1) / ROWS);
    total = __builtin_amdgcn_readlane(to[b], 63);
    unlisted += __builtin_amdgcn_readlane(wave_scan(listed_tiles(count[b])), 63);
  }
  const int chunk = (total * p.col_groups + 7) >> 3, within = blockIdx.x >> 3, id = (blockIdx.x & 7) * chunk + within;
  if (within >= chunk || id >= total * p.col_groups) return;
  const int pass_of_all = id / p.col_groups;
  int e = 0, cnt = 0, before = 0;
#pragma unroll
  for (int b = 3; b >= 0; --b) {
    const unsigned long long past = __ballot(to[b] > pass_of_all);
    if (past) {
      const int l = __ffsll(past) - 1;
      e = 64 * b + l;
      cnt = __builtin_amdgcn_readlane(count[b], l);
      before = __builtin_amdgcn_readlane(to[b], l) - (cnt + ROWS - 1) / ROWS;
    }
  }
  const int passes = (cnt + ROWS - 1) / ROWS, q = id - before * p.col_groups, cg = q / passes, pass = q - cg * passes;
  const bool stream = p.stream && passes == 1;
  // weight rows: 16 columns of gate and the same of up, or 32 columns of the one matrix
  const int n0 = GATEUP ? cg * 64 + 16 * wave : cg * 128 + 32 * wave;
  const int nb = GATEUP ? n0 : min(n0, N - 32);  // (a wave past the last column reads the last ones and stores nothing)
  const int64_t we = (static_cast<int64_t>(e) * N + nb) * K;
  const uint64_t w0 = reinterpret_cast<uint64_t>(p.b0 + we);
  const uint64_t w1 = reinterpret_cast<uint64_t>(GATEUP ? p.b1 + we : p.b0 + we + static_cast<int64_t>(16) * K);
  const int k_start = p.turn ? (5 * e + 3 * cg) % steps : 0;
  const int r8 = lane >> 3, c_lo = (lane & 7) ^ (r8 >> 1), c_hi = c_lo ^ 4;
  const uint32_t off_lo = static_cast<uint32_t>(r8 * K + c_lo * 8) * 2u, off_hi = static_cast<uint32_t>((r8 + 8) * K + c_hi * 8) * 2u;
  const uint32_t to_a = lds0 + wave * (NA * 1024u), to_b = lds0 + B_AT + wave * 4096u;
  auto kofs = [&](int s) {
    const int k = s + k_start;
    return static_cast<uint32_t>(k < steps ? k : k - steps) * 128u;
  };
  auto request_b = [&](int s) {
    const uint32_t k = kofs(s), to = to_b + (s & 1) * B_STAGE;
    if (stream) {
      lds_load16<true>(w0, off_lo, k, to);
      lds_load16<true>(w0, off_hi, k, to + 1024);
      lds_load16<true>(w1, off_lo, k, to + 2048);
      lds_load16<true>(w1, off_hi, k, to + 3072);
    } else {
      lds_load16(w0, off_lo, k, to);
      lds_load16(w0, off_hi, k, to + 1024);
      lds_load16(w1, off_lo, k, to + 2048);
      lds_load16(w1, off_hi, k, to + 3072);
    }
  };
  const int seg0 = ((const_i32)p.seg_offsets)[e];
  int row0 = seg0 + pass * ROWS, left = min(cnt - pass * ROWS, ROWS);
  if (unlisted != 0 && !listed_rows(p.list, e, seg0, cnt, row0, left)) return;
  const int act = (left + 15) >> 4;
  const int l15 = lane & 15, l4 = lane >> 4;
  const uint32_t cpos = static_cast<uint32_t>((l4 ^ (l15 >> 1)) * 16);  // k 0..31; k 32..63: ^ 64
  const uint32_t ra = lds0 + l15 * 128u + cpos, rb = lds0 + B_AT + wave * 4096u + l15 * 128u + cpos;

  if (p.a_src) {
    // the row indices into the wave's own part of the second stage, whose rows are requested behind them
#pragma unroll
    for (int i = 0; i < (RB + 3) / 4; ++i)
      lds_load4(reinterpret_cast<uint64_t>(p.a_src), static_cast<uint32_t>(min(row0 + 64 * i + lane, p.last_row)) * 4u, 0,
                to_a + A_STAGE + i * 256u);
  }
  request_b(0);
  request_b(1);
  uint32_t off_a[NA];
  if (p.a_src) lds_wait<2 * NB>();
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int blk = wave * NA + i, r = min(8 * blk + r8, left - 1);
    const int src = p.a_src ? min(max(lds_read_i32(to_a + A_STAGE + r * 4u), 0), p.a_rows - 1) : r;
    off_a[i] = (static_cast<uint32_t>(src) * static_cast<uint32_t>(K) + (blk & 1 ? c_hi : c_lo) * 8u) * 2u;
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  const uint64_t act_base = reinterpret_cast<uint64_t>(p.a_src ? p.a : p.a + static_cast<int64_t>(row0) * K);
  auto request_a = [&](int s) {
    const uint32_t k = kofs(s), to = to_a + (s & 1) * A_STAGE;
#pragma unroll
    for (int i = 0; i < NA; ++i) lds_load16(act_base, off_a[i], k, to + i * 1024u);
  };
  request_a(0);
  request_a(1);
  f32x4 acc[RB][2];
#pragma unroll
  for (int mi = 0; mi < RB; ++mi) acc[mi][0] = acc[mi][1] = f32x4{0, 0, 0, 0};
  for (int s = 0; s < steps; ++s) {
    if (s == 0) lds_wait<NA>();
    else if (s + 1 < steps) lds_wait<NA + NB>();
    else lds_wait<0>();
    lds_sync<63>();
    const uint32_t at = (s & 1) * A_STAGE, bt = (s & 1) * B_STAGE;
    bf16x8 b0[2], b1[2], a[RB][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      b0[h] = lds_read16(((rb + bt) ^ (h * 64u)));
      b1[h] = lds_read16(((rb + bt) ^ (h * 64u)) + 2048);
    }
#pragma unroll
    for (int mi = 0; mi < RB; ++mi)
      if (mi < act)
#pragma unroll
        for (int h = 0; h < 2; ++h) a[mi][h] = lds_read16(((ra + at) ^ (h * 64u)) + mi * 2048u);
    lds_sync<63>();
    if (s + 2 < steps) {
      request_b(s + 2);
      request_a(s + 2);
    }
#pragma unroll
    for (int mi = 0; mi < RB; ++mi)
      if (mi < act)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          acc[mi][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0[h], a[mi][h], acc[mi][0], 0, 0, 0);
          acc[mi][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1[h], a[mi][h], acc[mi][1], 0, 0, 0);
        }
  }
  if (n0 >= N) return;
  // lane = activation row lane & 15, its four values = columns 4 l4 .. 4 l4 + 3 of a 16-column block
#pragma unroll
  for (int mi = 0; mi < RB; ++mi) {
    const int r = 16 * mi + l15;
    if (r >= left) continue;
    const int64_t at = static_cast<int64_t>(row0 + r) * N + n0 + 4 * l4;
    if constexpr (GATEUP) {
      float gv[4], uv[4], hv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        gv[i] = round_bf16(acc[mi][0][i]);
        uv[i] = round_bf16(acc[mi][1][i]);
        hv[i] = round_bf16(gv[i] * short_sigmoid(gv[i])) * uv[i];
      }
      if (p.gate) {
        *reinterpret_cast<u32x2*>(p.gate + at) = u32x2{pack2(gv[0], gv[1]), pack2(gv[2], gv[3])};
        *reinterpret_cast<u32x2*>(p.up + at) = u32x2{pack2(uv[0], uv[1]), pack2(uv[2], uv[3])};
      }
      *reinterpret_cast<u32x2*>(p.out + at) = u32x2{pack2(hv[0], hv[1]), pack2(hv[2], hv[3])};
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j)
        *reinterpret_cast<u32x2*>(p.out + at + 16 * j) =
            u32x2{pack2(acc[mi][j][0], acc[mi][j][1]), pack2(acc[mi][j][2], acc[mi][j][3])};
    }
  }
}

}  // namespace

// gate/up (stage 1) or down (stage 2) of the forward; the arguments of bf16_grouped_fwd.  tall: 128 rows a pass, else 64; turn: each
// tile's contraction starts at a step of its own (`turned` in grouped_bf16.hip).
int short_rows_fwd(int stage, bool tall, const void* a, const int32_t* a_src, int64_t a_rows, const void* b0, const void* b1,
                   void* gate, void* up, void* out, const int32_t* seg_offsets, const int32_t* seg_counts, const int32_t* tile_expert,
                   const int32_t* tile_row0, const int32_t* num_tiles, int64_t tile_capacity, int64_t El, int64_t K, int64_t N,
                   int64_t row_capacity, bool stream, bool turn, hipStream_t s) {
  ShortArgs p{};
  p.a = (const uint16_t*)a; p.a_src = a_src; p.a_rows = (int)a_rows;
  p.b0 = (const uint16_t*)b0; p.b1 = (const uint16_t*)b1;
  p.gate = (uint16_t*)gate; p.up = (uint16_t*)up; p.out = (uint16_t*)out;
  p.seg_offsets = seg_offsets; p.seg_counts = seg_counts;
  p.list = {tile_expert, tile_row0, num_tiles, (int)std::min<int64_t>(tile_capacity, INT32_MAX)};
  p.El = (int)El; p.K = (int)K; p.N = (int)N; p.last_row = (int)row_capacity - 1; p.turn = turn; p.stream = stream;
  const int width = stage == 1 ? 64 : 128;
  p.col_groups = (int)((N + width - 1) / width);
  auto launch = [&](auto gateup, auto rb) {
    constexpr int B = decltype(rb)::value;
    const int64_t passes = std::min(El, row_capacity) + row_capacity / (16 * B);  // at most
    hipLaunchKernelGGL((short_rows_kernel<decltype(gateup)::value, B>), dim3((unsigned)((passes * p.col_groups + 7) / 8 * 8)),
                       dim3(256), short_lds(B), s, p);
  };
  auto of_height = [&](auto gateup) {
    if (tall) launch(gateup, std::integral_constant<int, 8>{});
    else launch(gateup, std::integral_constant<int, 4>{});
  };
  if (stage == 1) of_height(std::true_type{});
  else of_height(std::false_type{});
  return check_launch("grouped forward, short rows");
}

}  // namespace mi355
