// Forward expert products for a handful of rows per expert (generation: one token to a few dozen).
//
// Such a product is one read of the touched experts' weights and nothing else: a weight row meets at
// most 16 activation rows, so no operand is worth staging.  The 256-row kernels of grouped_bf16.hip
// stream the same weights through LDS in 1 MB work items, one workgroup per CU in lockstep: at one
// token 48 items for 256 CUs, at 33 tokens 2.6 rounds of them.  Here a workgroup is four waves that
// split the contraction of 16 output columns (of gate and up, or 32 of the down projection) of one
// expert, and the four partial tiles are added in wave order through LDS.
//   A wave's weights go straight into LDS of its own, two contraction steps of 64 ahead (8 KiB; three workgroups fit a CU's LDS: 96 KiB), in whole 128-byte lines, eight rows an
// instruction, and are read from there as MFMA fragments: no barrier stands in the loop.  Asked for as
// fragments, 64 bytes of 16 rows an instruction with 16 KiB in registers ahead, a line is two requests, and the non-temporal hint makes the
// second one go to memory again (5-11 % slower).  In lines the hint gains what it gains in the 256-row kernels (`streamed` there).
//   Bound by HBM, us, fragments / lines / lines with the hint: gate and up of 33 tokens of 128 experts of 2048 x 768 (709 MB) 120 / 121 / 105 (6.8 TB/s), down
// 57 / 60 / 54; 100 tokens 148 / 145 / 130, 68 / 70 / 65; 32 experts of 7168 x 2048, three rows each 330 / 304 / 271, 150 / 152 / 133; one
// dense segment of it, where half the chip has to do, 16 rows 21 / 13, 8 / 7, 60 rows 77 / 41, 25 / 14; five tokens of the first, 36 / 35, 19 / 19.  One step ahead and twice the workgroups a
// CU: the same within 3 %, but the dense segment 23 and 10; three ahead: 4-6 % slower.
// Waves along the contraction rather than side by side: at one token 12-25 us less in all, at 33 the
// same.  32 or 64 rows per wave instead of 16 need registers that the requests in flight want: slower.
//   A contraction step is 64 wide: lane group g = lane / 16 holds k = 16 g .. 16 g + 15 of it for both operands alike.
#include <algorithm>

#include "bf16_tiles.h"
#include "common.h"
#include "select_rows.h"

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

constexpr int kFewSteps = 2;                          // contraction steps of a wave in LDS
constexpr uint32_t kFewStep = 6144;                   // bytes of one: 16 weight rows, 16 more, 16 activation rows, 128 each
constexpr int kFewLds = 4 * kFewSteps * kFewStep;     // of a workgroup; the partial tiles (8 KiB) take their place

// Column group cg of the product of expert e with the rows that where() names (the first and how many, at least one: looked up once
// the first weights are on their way); a row is source(row) of a, or itself.
struct FewRows {
  int row0, rows;
};
template <bool GATEUP, bool STREAM, typename Source, typename Where>
__device__ __forceinline__ void few_rows_tile(const FewArgs& p, int e, int cg, bool through, Source source, Where where, char* ring) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, g = lane >> 4;
  const int K = p.K, N = p.N;
  // this wave's share of the contraction
  const int steps = K >> 6, s0 = steps * wave >> 2, n = (steps * (wave + 1) >> 2) - s0;
  // weight rows: 16 columns of gate and the same of up, or 32 columns of the one matrix (N % 32 == 0)
  const int n0 = cg * (GATEUP ? 16 : 32);
  const int64_t we = static_cast<int64_t>(e) * N * K + static_cast<int64_t>(n0) * K + s0 * 64;
  const uint64_t w0 = reinterpret_cast<uint64_t>(p.b0 + we);
  const uint64_t w1 = reinterpret_cast<uint64_t>(GATEUP ? p.b1 + we : p.b0 + we + static_cast<int64_t>(16) * K);
  const uint64_t act = reinterpret_cast<uint64_t>(p.a + s0 * 64);
  const uint32_t own = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_cptr)ring)) + wave * (kFewSteps * kFewStep);
  // an instruction's eight rows: this lane's, and its 16 bytes -- chunk c of row r of 16 lies at c ^ (r >> 1)
  const int r8 = lane >> 3, c_lo = (lane & 7) ^ (r8 >> 1), c_hi = c_lo ^ 4;
  const uint32_t off_lo = static_cast<uint32_t>(r8 * K + c_lo * 8) * 2u, off_hi = static_cast<uint32_t>((r8 + 8) * K + c_hi * 8) * 2u;
  auto request_w = [&](int s) {
    const uint32_t k = s * 128u, to = own + (s % kFewSteps) * kFewStep;
    lds_load16<STREAM>(w0, off_lo, k, to);
    lds_load16<STREAM>(w0, off_hi, k, to + 1024);
    lds_load16<STREAM>(w1, off_lo, k, to + 2048);
    lds_load16<STREAM>(w1, off_hi, k, to + 3072);
  };
  auto request_first = [&]() {
#pragma unroll
    for (int i = 0; i < kFewSteps; ++i)
      if (i < n) request_w(i);
  };
  // the first weights go out before the rows are known
  request_first();
  const FewRows at_rows = where();
  const int row0 = at_rows.row0, rows = at_rows.rows;
  for (int sub = 0; sub < rows; sub += 16) {
    if (sub) request_first();
    uint32_t off_a[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int row = row0 + min(sub + r8 + 8 * h, rows - 1);
      const int src = through ? min(max(source(row), 0), p.a_rows - 1) : row;
      off_a[h] = (static_cast<uint32_t>(src) * static_cast<uint32_t>(K) + (h ? c_hi : c_lo) * 8u) * 2u;
    }
    auto request_a = [&](int s) {
      const uint32_t k = s * 128u, to = own + (s % kFewSteps) * kFewStep + 4096;
      lds_load16(act, off_a[0], k, to);
      lds_load16(act, off_a[1], k, to + 1024);
    };
#pragma unroll
    for (int i = 0; i < kFewSteps; ++i)
      if (i < n) request_a(i);
    f32x4 acc0 = {0, 0, 0, 0}, acc1 = {0, 0, 0, 0};
    auto multiply = [&](int s) {
      const uint32_t at = own + (s % kFewSteps) * kFewStep + r16 * 128u;
      bf16x8 b0[2], b1[2], a[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t piece = ((2 * g + h) ^ (r16 >> 1)) * 16u;  // k 16 g + 8 h ..
        b0[h] = lds_read16(at + piece);
        b1[h] = lds_read16(at + piece + 2048);
        a[h] = lds_read16(at + piece + 4096);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the step's place is free for requests then)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0[h], a[h], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b1[h], a[h], acc1, 0, 0, 0);
      }
    };
    // the first steps are waited for together (their weights were requested in front of all their rows), the others in turn
    static_assert(kFewSteps == 2, "the waits below are written out");
    lds_wait<0>();
    int s = 0;
    for (; s + kFewSteps < n; ++s) {
      if (s >= kFewSteps) lds_wait<6>();
      multiply(s);
      request_w(s + kFewSteps);
      request_a(s + kFewSteps);
    }
    if (s < n) {
      lds_wait<6>();
      multiply(s++);
    }
    if (s < n) {
      lds_wait<0>();
      multiply(s);
    }
    f32x4* part = reinterpret_cast<f32x4*>(ring);  // [4][2][64]
    __syncthreads();
    part[(wave * 2 + 0) * 64 + lane] = acc0;
    part[(wave * 2 + 1) * 64 + lane] = acc1;
    __syncthreads();
    // lane = activation row lane & 15, its four values = columns 4 g .. 4 g + 3 of a 16-column tile
    auto sum = [&](int tile) {
      f32x4 v = part[tile * 64 + lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) v += part[(w * 2 + tile) * 64 + lane];
      return v;
    };
    if (wave < (GATEUP ? 1 : 2) && sub + r16 < rows) {
      const int64_t at = static_cast<int64_t>(row0 + sub + r16) * N + n0 + 16 * wave + 4 * g;
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

template <bool GATEUP, bool STREAM>
__global__ __launch_bounds__(256) void few_rows_kernel(FewArgs p) {
  extern __shared__ __attribute__((aligned(16))) char ring[];
  const int t = blockIdx.x / p.col_groups, cg = blockIdx.x - t * p.col_groups;
  // looked up together (an entry past the last tile is not used): every lookup in a row is a round trip in front of the weights
  const int tiles = *p.num_tiles, e = __builtin_amdgcn_readfirstlane(p.tile_expert[t]),
            row0 = __builtin_amdgcn_readfirstlane(p.tile_row0[t]);
  if (t >= tiles) return;
  few_rows_tile<GATEUP, STREAM>(
      p, e, cg, p.a_src != nullptr, [&](int row) { return p.a_src[row]; },
      [&]() -> FewRows {
        const int cnt = p.seg_counts[e], seg0 = p.seg_offsets[e];
        return {row0, min(even_tile_rows(cnt, 256), seg0 + cnt - row0)};
      },
      ring);
}

// ---- a handful of tokens, forward only: no plan ---------------------------------------------------
// One or a few tokens' choices are K rows each, nearly all of different experts, and grouping them saves nothing.  Row t K + k is
// choice k of token t: the first launch selects in every workgroup that needs the choice (a row of 16 lanes, about a
// microsecond, against a launch of its own) and forms gate and up of its row; the second takes the
// down projection of all K choices of a token for 16 columns and combines them, waves along choices and halves of
// the contraction.  With the gate's projection three launches instead of five; every sum in the order of the grouped kernels, the
// same bits.  Up to four tokens (torch_block.cpp), all experts here: block forward of 128 experts of 2048 x 768, eight a token, us,
// grouped / this: one token 39.7 / 28.7, 2 49 / 40, 3 60 / 55, 4 72 / 68, 6 96 / 99, 8 111 / 125 -- the experts that tokens share are read
// once per token here.  On one rank's share (32 of 256 experts) seven in eight workgroups select for nothing: four tokens 118 / 165.
struct ChoiceIn {
  const float *partial, *logit_bias;  // (splits, T, E)
  int splits, T, lo, hi;
  SelectArgs sel;
  float* weights;  // (T, K)
  int32_t* ids;    // (T, K): local expert, -1 elsewhere
  int32_t* counts; // (E)
};

// token t's choices, by a row of 16 lanes each (lane l < K: choice l)
template <int VPR, bool FULL>
__device__ __forceinline__ RowChoice choose(const ChoiceIn& c, int t, int l) {
  const int E = c.sel.E;
  float x[VPR], s[VPR], cutoff;
  load_row<VPR, FULL>(c.partial + static_cast<int64_t>(t) * E, l, E, x);
  for (int z = 1; z < c.splits; ++z) {
    float y[VPR];
    load_row<VPR, FULL>(c.partial + (static_cast<int64_t>(z) * c.T + t) * E, l, E, y);
#pragma unroll
    for (int j = 0; j < VPR; ++j) x[j] += y[j];
  }
  if (c.splits > 1 && c.logit_bias) {
#pragma unroll
    for (int j = 0; j < VPR; ++j)
      if (FULL || l * VPR + j < E) x[j] += c.logit_bias[l * VPR + j];
  }
  return select_row<VPR, FULL>(c.sel, x, l, false, false, s, cutoff);
}

constexpr int kChoiceTokens = 16;  // a row of 16 lanes each in one workgroup of four waves

template <int VPR, bool FULL>
__global__ __launch_bounds__(256) void choice_gateup_kernel(FewArgs p, ChoiceIn c) {
  extern __shared__ __attribute__((aligned(16))) char ring[];
  const int lane = threadIdx.x & 63, K = c.sel.K;
  const int row = blockIdx.x / p.col_groups, cg = blockIdx.x - row * p.col_groups;
  if (row == c.T * K) {
    // the last workgroup: everyone's choices for the second launch, and the experts' loads
    int* count = reinterpret_cast<int*>(ring);
    for (int e = threadIdx.x; e < c.sel.E; e += 256) count[e] = 0;
    __syncthreads();
    const int t = threadIdx.x >> 4, l = lane & 15;
    const RowChoice ch = choose<VPR, FULL>(c, min(t, c.T - 1), l);
    if (t < c.T && l < K) {
      c.weights[t * K + l] = ch.weight;
      c.ids[t * K + l] = ch.id >= c.lo && ch.id < c.hi ? ch.id - c.lo : -1;
      if (ch.id >= 0 && ch.id < c.sel.E) atomicAdd(&count[ch.id], 1);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < c.sel.E; e += 256) c.counts[e] = count[e];
    return;
  }
  const int t = row / K;
  const RowChoice ch = choose<VPR, FULL>(c, t, lane & 15);
  const int id = __builtin_amdgcn_readlane(ch.id, row - t * K);
  if (id < c.lo || id >= c.hi) return;  // (the same for the whole workgroup)
  few_rows_tile<true, false>(
      p, id - c.lo, cg, true, [&](int) { return t; }, [&]() -> FewRows { return {row, 1}; }, ring);
}

struct ChoiceOut {
  const uint16_t *h, *w2, *addend;  // (T K, F), (El, D, F), (T, D) or null
  uint16_t* out;
  const float* weights;
  const int32_t* ids;
  int K, D, F, El, round_terms;
};

// A workgroup is eight columns of one token; a wave takes one choice and two quarters of the contraction at a time, in one
// MFMA: operand rows 0-7 are the columns (and the choice's row) over quarter `pair`, rows 8-15 the same over quarter pair + 2, and of the
// result the two diagonal blocks are what is wanted.  One token, eight choices of 2048 x 768 (25 MB): 7.7 us, where 16 columns
// a workgroup, half the chip, took 12.9 and the grouped product with the combine behind it 11.4.
constexpr int kChoiceCols = 8, kChoiceWaves = 16;

__global__ __launch_bounds__(64 * kChoiceWaves) void choice_down_kernel(ChoiceOut p) {
  constexpr int kAhead = 4;  // 64-wide steps requested together
  __shared__ float part[16][4][kChoiceCols];  // choice, quarter of the contraction, column
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int groups = p.D / kChoiceCols, t = blockIdx.x / groups, n0 = (blockIdx.x - t * groups) * kChoiceCols;
  const int r8 = lane & 7, second = lane >> 3 & 1, g = lane >> 4;
  const int K = p.K, F = p.F, steps = F >> 6;
  const int my_e = lane < K ? p.ids[t * K + lane] : -1;
  const float my_w = lane < K ? p.weights[t * K + lane] : 0.0f;
  for (int u = wave; u < 2 * K; u += waves) {
    const int k = u >> 1, pair = u & 1;
    const int e = __builtin_amdgcn_readlane(my_e, k);
    if (e < 0 || e >= p.El) continue;
    const auto rsB = few_rsrc(p.w2 + (static_cast<int64_t>(e) * p.D + n0) * F), rsA = few_rsrc(p.h + (static_cast<int64_t>(t) * K + k) * F);
    // this lane's quarter
    const int q = pair + 2 * second, s0 = steps * q >> 2, s1 = steps * (q + 1) >> 2;
    const int n = max((steps * (pair + 1) >> 2) - (steps * pair >> 2), (steps * (pair + 3) >> 2) - (steps * (pair + 2) >> 2));
    const uint32_t offB = static_cast<uint32_t>(r8 * F + g * 16) * 2u, offA = static_cast<uint32_t>(g * 16) * 2u;
    f32x4 acc = {0, 0, 0, 0};
    u32x4 b[kAhead][2], a[kAhead][2];
    auto request = [&](int i, int s) {
      const uint32_t at = static_cast<uint32_t>(min(s0 + s, s1 - 1)) * 128u;  // (the shorter quarter's last step again: zeroed below)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        b[i][h] = __builtin_amdgcn_raw_buffer_load_b128(rsB, offB + at + 16 * h, 0, 0);
        a[i][h] = __builtin_amdgcn_raw_buffer_load_b128(rsA, offA + at + 16 * h, 0, 0);
      }
    };
    auto multiply = [&](int i, int s) {
      const bool live = s0 + s < s1;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const u32x4 zero = {0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, live ? b[i][h] : zero),
                                                      __builtin_bit_cast(bf16x8, live ? a[i][h] : zero), acc, 0, 0, 0);
      }
    };
#pragma unroll
    for (int i = 0; i < kAhead; ++i) request(i, min(i, n - 1));
    for (int s = 0; s < n; s += kAhead) {
#pragma unroll
      for (int i = 0; i < kAhead; ++i) {
        if (s + i < n) multiply(i, s + i);
        if (s + i + kAhead < n) request(i, s + i + kAhead);
      }
    }
    // lane = activation row lane & 15, its four values = weight rows 4 g ..: rows 0 (columns 0-7) and 8 (columns 8-15)
    if (r8 == 0 && (g >> 1) == second) *reinterpret_cast<f32x4*>(&part[k][q][4 * (g & 1)]) = acc;
  }
  if (wave != 0) {
    __syncthreads();
    return;
  }
  // the token's terms in ascending order of their experts, as the combine visits their rows
  const bool here = my_e >= 0 && my_e < p.El;
  int pos = 0;
  for (int k = 0; k < K; ++k) {
    const int e = __builtin_amdgcn_readlane(my_e, k);
    pos += e >= 0 && e < my_e ? 1 : 0;
  }
  const int terms = __popcll(__ballot(here));
  const int to = (here ? pos : 63) << 2;
  const int o_k = __builtin_amdgcn_ds_permute(to, lane);
  const float o_w = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(my_w)));
  __syncthreads();
  float sum = 0.0f;
  for (int n = 0; n < terms; ++n) {
    const int k = __builtin_amdgcn_readlane(o_k, n);
    const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(o_w), n));
    const float y = round_bf16(((part[k][0][r8] + part[k][1][r8]) + part[k][2][r8]) + part[k][3][r8]);
    const float term = y * w;
    sum += p.round_terms ? round_bf16(term) : term;
  }
  if (lane >= kChoiceCols) return;
  const int64_t o = static_cast<int64_t>(t) * p.D + n0 + r8;
  if (p.addend) sum = round_bf16(sum) + bf16_to_f32(p.addend[o]);
  p.out[o] = f32_to_bf16(sum);
}

}  // namespace

// gate/up (stage 1) or down (stage 2) of the forward; the arguments of bf16_grouped_fwd.  stream: weights with the non-temporal hint.
int few_rows_fwd(int stage, const void* a, const int32_t* a_src, int64_t a_rows, const void* b0, const void* b1,
                 void* gate, void* up, void* out, const int32_t* seg_offsets, const int32_t* seg_counts,
                 const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* num_tiles, int64_t tiles, int64_t K,
                 int64_t N, bool stream, hipStream_t s) {
  FewArgs p{};
  p.a = (const uint16_t*)a; p.a_src = a_src; p.a_rows = (int)a_rows;
  p.b0 = (const uint16_t*)b0; p.b1 = (const uint16_t*)b1;
  p.gate = (uint16_t*)gate; p.up = (uint16_t*)up; p.out = (uint16_t*)out;
  p.seg_offsets = seg_offsets; p.seg_counts = seg_counts; p.tile_expert = tile_expert; p.tile_row0 = tile_row0;
  p.num_tiles = num_tiles; p.K = (int)K; p.N = (int)N;
  p.col_groups = (int)(N / (stage == 1 ? 16 : 32));
  const dim3 grid((unsigned)(tiles * p.col_groups));
  const auto kernel = stage == 1 ? (stream ? few_rows_kernel<true, true> : few_rows_kernel<true, false>)
                                 : (stream ? few_rows_kernel<false, true> : few_rows_kernel<false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), kFewLds, s, p);
  return check_launch("grouped forward, few rows");
}

}  // namespace mi355

using namespace mi355;

namespace mi355 {
bool bf16_fast_path_ok(int64_t D, int64_t F);
}

extern "C" int mi355_choice_covers(int64_t T, int64_t D, int64_t F, int64_t E, int64_t K, int num_groups) {
  return T >= 1 && T <= kChoiceTokens && E >= 1 && K >= 1 && K <= E && bf16_fast_path_ok(D, F) &&
                 T * K * std::max(D, F) * 2 < (1ll << 31) && select_row_covers(E, K, num_groups, MI355_SELECT_TOPK)
             ? 1 : 0;
}

extern "C" int mi355_choice_gateup_fwd(const float* partial, int splits, const float* logit_bias, const float* expert_bias,
                                       int64_t T, int64_t E, int64_t K, int score_func, int route_norm, float route_scale,
                                       int num_groups, int num_limited, int64_t lo, int64_t hi, const void* x, const void* w1,
                                       const void* w3, void* h, float* weights_TK, int32_t* ids_TK, int32_t* counts_E,
                                       int64_t D, int64_t F, void* stream) {
  if (!mi355_choice_covers(T, D, F, E, K, num_groups))
    return fail(MI355_EUNSUP, "choice_gateup_fwd: not covered; use mi355_route_plan and mi355_grouped_swiglu_fwd");
  MI355_REQUIRE(score_func >= 0 && score_func <= 2, "choice_gateup_fwd: unknown score_func %d", score_func);
  if (num_groups > 0)
    MI355_REQUIRE(E % num_groups == 0 && E / num_groups >= 2 && num_limited >= 1 && num_limited <= num_groups &&
                      K <= (int64_t)num_limited * (E / num_groups),
                  "choice_gateup_fwd: bad group config G=%d L=%d", num_groups, num_limited);
  MI355_REQUIRE(0 <= lo && lo < hi && hi <= E, "choice_gateup_fwd: bad local range [%lld,%lld)", (long long)lo, (long long)hi);
  MI355_REQUIRE(partial && splits >= 1 && x && w1 && w3 && h && weights_TK && ids_TK && counts_E &&
                    aligned16({partial, x, w1, w3, h}),
                "choice_gateup_fwd: null or misaligned pointer");
  FewArgs p{};
  p.a = (const uint16_t*)x; p.a_rows = (int)T;
  p.b0 = (const uint16_t*)w1; p.b1 = (const uint16_t*)w3; p.out = (uint16_t*)h;
  p.K = (int)D; p.N = (int)F; p.col_groups = (int)(F / 16);
  const ChoiceIn c{partial, logit_bias, splits, (int)T, (int)lo, (int)hi,
                   SelectArgs{expert_bias, (int)E, (int)K, score_func, route_norm, route_scale, num_groups, num_limited},
                   weights_TK, ids_TK, counts_E};
  with_row_shape(E, [&](auto vpr, auto full) {
    hipLaunchKernelGGL((choice_gateup_kernel<decltype(vpr)::value, decltype(full)::value>),
                       dim3((unsigned)(T * K * p.col_groups + 1)), dim3(256), kFewLds, as_stream(stream), p, c);
  });
  return check_launch("choice_gateup");
}

extern "C" int mi355_choice_down_fwd(const void* h, const void* w2, const float* weights_TK, const int32_t* ids_TK,
                                     const void* addend, void* out, int64_t T, int64_t K, int64_t El, int64_t D, int64_t F,
                                     int round_terms, void* stream) {
  MI355_REQUIRE(T >= 1 && T <= kChoiceTokens && K >= 1 && K <= 16 && El >= 1 && bf16_fast_path_ok(D, F), "choice_down_fwd: bad shape");
  MI355_REQUIRE(h && w2 && weights_TK && ids_TK && out && aligned16({h, w2}), "choice_down_fwd: null or misaligned pointer");
  const ChoiceOut p{(const uint16_t*)h, (const uint16_t*)w2, (const uint16_t*)addend, (uint16_t*)out, weights_TK, ids_TK,
                    (int)K, (int)D, (int)F, (int)El, round_terms};
  const int waves = (int)std::min<int64_t>(kChoiceWaves, 2 * K);
  hipLaunchKernelGGL(choice_down_kernel, dim3((unsigned)(T * (D / kChoiceCols))), dim3(64 * waves), 0, as_stream(stream), p);
  return check_launch("choice_down");
}
