// Expert choice and permutation plan in one pass: what mi355_router_select_fwd followed by
// mi355_permute_plan compute, for the block's own path, in one launch (up to 64 tokens) or two.
//
//   1. route_rank   a workgroup takes 32 or 64 tokens at a time: each row of 16 lanes adds its
//                   token's partial logits, selects its experts (select_rows.h) and leaves the ids
//                   in LDS, where the workgroup ranks its slots among equal experts in slot order
//                   (the wave's lanes by ballots over the bits of the id, the waves through
//                   per-wave counts).  Emits weights, ids, ranks and the workgroup's histogram.
//   2. route_rows   the same partition: every workgroup sums the histograms below its own for its
//                   slots' offsets (all of them, for the segments), which costs it a read of a few
//                   dozen KiB from L2 and saves the launch of a scan, and writes its slots' rows in
//                   both directions; the first workgroup writes the plan's lists.  What statistics a router keeps are summed,
//                   and its required-bias histogram is counted, by workgroups of their own behind those.
// A single workgroup does both at once.  Bound by launches, instruction issue and dependent latency throughout: at 33
// tokens of 128 experts the four launches this replaces took 29 us of GPU time, at 8192 tokens
// (8 each) 39 us; here 13 and 21.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gate_rows.h"
#include "gemm_generic.h"
#include "quantile_observe.h"
#include "select_rows.h"

namespace mi355 {
namespace {

// A workgroup of LANES takes LANES / 16 tokens at a time; of at most 16 choices they are at most LANES slots,
// one per lane.  Beyond this many workgroups a workgroup takes several such chunks, so that the histograms
// everyone reads stay small.
constexpr int kMaxBlocks = 256;

struct PlanOut {
  int lo, hi, align, tile_m, row_capacity, tile_capacity;
  int32_t *counts_E, *seg_offsets, *seg_counts, *row_of_slot, *slot_of_row, *token_of_row;
  float* row_scale;
  int32_t *tile_expert, *tile_row0, *num_tiles;
};

// What a router that keeps statistics wants besides (all null: nothing).  valid_counts: every expert's slots
// of the tokens that are not padding.  scores, cutoff: for the required-bias histogram.  f, scale, acc:
// the load-balance loss sum_e f_e p_e of aux.hip over the tokens that are not padding: f_e and the
// factor of its gradient for the backward, and the running mean metric it is added to.
struct StatsOut {
  const uint8_t* padding;  // (T), non-zero = padding
  int32_t* valid_counts;
  float *scores, *cutoff;
  float *f, *scale;
  void* acc;
  int acc_dtype;
  const float* denominator;
  float coeff;
  int32_t* block_valid;  // (blocks, E)
  float* block_share;    // (blocks, E)
};

// Integer arrays in LDS for the layout step, E experts.
struct LayoutLds {
  int32_t *count, *before, *seg, *tile, *order, *wave_sums;
  __device__ LayoutLds(int32_t* base, int E)
      : count(base), before(base + E), seg(base + 2 * E), tile(base + 3 * E + 1), order(base + 4 * E + 2),
        wave_sums(base + 5 * E + 2) {}
};
constexpr int layout_words(int E) { return 5 * E + 2 + 8; }

// counts -> padded segment offsets, tiles before each local expert, rank by descending count; left in
// LDS for all lanes (ends on a barrier).  One lane per local expert (at most 256: four waves) scans
// rows and tiles; the ranks, one comparison per pair of experts, are shared by all lanes.
__device__ void plan_layout(const LayoutLds& s, const PlanOut& p, bool lists) {
  const int El = p.hi - p.lo, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, lanes = blockDim.x;
  for (int j = tid; j < El; j += lanes) s.order[j] = 0;
  int rows = 0, tiles = 0, rows_to = 0, tiles_to = 0;
  if (wave < 4) {
    const int c = tid < El ? s.count[p.lo + tid] : 0;
    rows = p.align > 1 ? (c + p.align - 1) / p.align * p.align : c;
    tiles = (c + p.tile_m - 1) / p.tile_m;
    rows_to = wave_scan(rows);
    tiles_to = wave_scan(tiles);
    if (lane == 63) {
      s.wave_sums[wave] = rows_to;
      s.wave_sums[4 + wave] = tiles_to;
    }
  }
  __syncthreads();
  if (wave < 4) {
    for (int w = 0; w < wave; ++w) {
      rows_to += s.wave_sums[w];
      tiles_to += s.wave_sums[4 + w];
    }
    if (tid < El) {
      s.seg[tid] = rows_to - rows;
      s.tile[tid] = tiles_to - tiles;
      if (tid == El - 1) {
        s.seg[El] = rows_to;
        s.tile[El] = tiles_to;
      }
    }
  }
  if (lists) {
    const int shares = max(1, lanes / El), slice = (El + shares - 1) / shares;
    for (int idx = tid; idx < El * shares; idx += lanes) {
      const int j = idx % El, o0 = (idx / El) * slice, o1 = min(El, o0 + slice);
      const int c = s.count[p.lo + j];
      int rank = 0;
#pragma unroll 8
      for (int o = o0; o < o1; ++o) rank += s.count[p.lo + o] > c - (o < j ? 1 : 0) ? 1 : 0;  // more, or as many and before it
      if (rank) atomicAdd(&s.order[j], rank);
    }
  }
  __syncthreads();
}

__device__ void write_lists(const LayoutLds& s, const PlanOut& p, int E) {
  const int El = p.hi - p.lo, tid = threadIdx.x, lanes = blockDim.x;
  for (int e = tid; e < E; e += lanes) p.counts_E[e] = s.count[e];
  for (int j = tid; j <= El; j += lanes) {
    p.seg_offsets[j] = s.seg[j];
    if (j == El) {
      *p.num_tiles = min(s.tile[El], p.tile_capacity);
      break;
    }
    const int c = s.count[p.lo + j];
    p.seg_counts[j] = c;
    p.seg_counts[El + s.order[j]] = j;
    const int nt = s.tile[j + 1] - s.tile[j], rows = even_tile_rows(c, p.tile_m);
    for (int i = 0; i < nt; ++i) {
      const int at = s.tile[j] + i;
      if (at < p.tile_capacity) {
        p.tile_expert[at] = j;
        p.tile_row0[at] = s.seg[j] + i * rows;
      }
    }
  }
}

__device__ __forceinline__ void place_slot(const LayoutLds& s, const PlanOut& p, int slot, int e, int rank, int K,
                                           float weight) {
  int row = -1;
  if (e >= p.lo && e < p.hi) {
    row = s.seg[e - p.lo] + s.before[e] + rank;
    if (row < p.row_capacity) {
      p.slot_of_row[row] = slot;
      p.token_of_row[row] = slot / K;
      if (p.row_scale) p.row_scale[row] = weight;
    } else {
      row = -1;
    }
  }
  p.row_of_slot[slot] = row;
}

// Every expert's valid slots and score shares of all workgroups, the shares in the workgroups' order; lane e < E has expert e's.  One workgroup of kLanes;
// stage: kStatsWords words of LDS.  All lanes request what they find, a run of workgroups at a time, and hand the shares on through LDS to the
// lane that adds them.  With 32 of either kind in flight in that lane's own registers the kernel had 198 of them at 512 lanes and spilled 70 at 1024 (50 and none
// here), and all its workgroups were one to a CU: the launch at 3000 and 12000 tokens of 64 experts 10.0 / 7.9 us, 59.6 / 13.2.
constexpr int kStatsBatch = 8;
template <int kLanes>
constexpr int kStatsWords = kLanes * kStatsBatch;
template <int kLanes>
__device__ __forceinline__ void sum_blocks(const StatsOut& st, int E, int nb, int32_t* stage, int& valid, float& share) {
  const int tid = threadIdx.x, parts = kLanes / E, run = parts * E;  // E <= 256; lanes at work
  float* shares = reinterpret_cast<float*>(stage);
  int mine = 0;  // of expert tid % E
  for (int b0 = 0; b0 < nb; b0 += parts * kStatsBatch) {
    int v[kStatsBatch];
    float p[kStatsBatch];
#pragma unroll
    for (int i = 0; i < kStatsBatch; ++i) {
      const int at = (b0 + i * parts) * E + tid;
      const bool in = tid < run && at < nb * E;
      v[i] = in ? st.block_valid[at] : 0;
      p[i] = in && st.f ? st.block_share[at] : 0.0f;
    }
#pragma unroll
    for (int i = 0; i < kStatsBatch; ++i) {
      mine += v[i];
      if (tid < run) shares[i * run + tid] = p[i];
    }
    __syncthreads();
    if (st.f && tid < E)
#pragma unroll 8
      for (int j = 0; j < min(parts * kStatsBatch, nb - b0); ++j) share += shares[j * E + tid];
    __syncthreads();
  }
  if (tid < run) stage[tid] = mine;
  __syncthreads();
  if (tid < E)
    for (int q = 0; q < parts; ++q) valid += stage[q * E + tid];
}

// The loss from the valid slots and score shares of lane e < E's expert; one workgroup.
__device__ void finish_loss(const StatsOut& st, int E, int valid, float share, float* red) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr float kEps = 1e-12f;  // F.normalize's clamp
  if (!st.f) return;
  // E <= 256: four waves hold everything
  auto total = [&](float v) {
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0 && wave < 4) red[wave] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
  };
  const float all = total(static_cast<float>(valid));
  const float f = static_cast<float>(valid) * (static_cast<float>(E) / fmaxf(all, kEps));
  const float loss = total(f * share);
  if (tid < E) st.f[tid] = f;
  if (tid == 0) {
    const float scale = 1.0f / fmaxf(*st.denominator, 1.0f);
    *st.scale = st.coeff * scale;
    if (st.acc && st.acc_dtype == MI355_BF16) {
      uint16_t* acc = static_cast<uint16_t*>(st.acc);
      *acc = f32_to_bf16(bf16_to_f32(*acc) + loss * scale);
    } else if (st.acc) {
      *static_cast<float*>(st.acc) += loss * scale;
    }
  }
}

// The gate's operands where its projection rides along (TX: their type; void: the logits are there already): up to 32
// experts are one tile of it, whose 512 lanes are those of 32 tokens' selection.  A launch less: a training step of 512 fp32 tokens
// of 8 x 256 x 512 117 -> 105 us, 30 bf16 tokens of 4 x 200 x 104 122 -> 112; 8000 tokens of 16 x 512 x 512 forward 76.6 -> 74.8.
struct GateIn {
  const void* x;
  const float *w, *bias;
  int D, k_per_wave;
};

template <int VPR, bool FULL, int kLanes, typename TX = void>
__global__ __launch_bounds__(kLanes) void route_rank_kernel(
    GateIn gate, const float* __restrict__ partial, int splits, const float* __restrict__ logit_bias,
    float* __restrict__ logits_out, SelectArgs sel, float* __restrict__ weights, int64_t* __restrict__ ids,
    uint32_t* __restrict__ rank_in_block, int32_t* __restrict__ block_hist, int T, int chunks, int fill, PlanOut p,
    StatsOut st) {
  constexpr int kRows = kLanes / 16, kWaves = kLanes / kWave;
  extern __shared__ int32_t lds[];
  const int E = sel.E, K = sel.K;
  int32_t* run = lds;                       // [E] slots of each expert so far
  int32_t* cnt = lds + E;                   // [waves][E] slots of each expert in each wave of the chunk
  const bool stats = st.valid_counts != nullptr || st.f != nullptr;
  int32_t* valid_run = cnt + kWaves * E;    // with statistics: [E] valid slots, [waves][E] score shares
  float* share = reinterpret_cast<float*>(valid_run + E);
  int32_t* extra = valid_run + (stats ? (1 + kWaves) * E : 0);  // single workgroup: the layout arrays
  __shared__ uint16_t id_sh[kLanes];
  __shared__ float w_sh[kLanes];
  __shared__ float red_sh[4];
  constexpr bool kGate = !std::is_void_v<TX>;
  static_assert(!kGate || (kLanes == 64 * R_WAVES && kRows == R_BM && 16 * VPR <= R_BN), "one tile of the projection a chunk");
  constexpr int kPitch = R_BN + 4;
  __shared__ __attribute__((aligned(16))) float logit_sh[kGate ? R_BM * kPitch : 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l = tid & 15;
  const bool single = gridDim.x == 1;
  // rows that end up without a slot (padding, unused capacity) must read -1 and a zero scale
  if (fill) {
    for (int64_t i = static_cast<int64_t>(blockIdx.x) * kLanes + tid; i < p.row_capacity;
         i += static_cast<int64_t>(gridDim.x) * kLanes) {
      p.slot_of_row[i] = -1;
      p.token_of_row[i] = -1;
      if (p.row_scale) p.row_scale[i] = 0.0f;
    }
    // (A single workgroup writes its own rows below, behind barriers, which order a workgroup's stores.  A fence for the whole device here, which
    // writes L2 back, held the first wave up for 4.6 us at 20 tokens of a share of 256 experts.)
  }
  for (int e = tid; e < E; e += kLanes) run[e] = 0;
  if (stats)
    for (int i = tid; i < (1 + kWaves) * E; i += kLanes) valid_run[i] = 0;  // (also the shares: 0.0f)

  int my_e = -1, my_rank = 0;
  for (int c = 0; c < chunks; ++c) {
    const int t0 = (blockIdx.x * chunks + c) * kRows;
    if (t0 >= T) break;  // workgroup-uniform
    for (int i = tid; i < kWaves * E; i += kLanes) cnt[i] = 0;
    if constexpr (kGate) {
      __shared__ __attribute__((aligned(16))) float tile_sh[R_WAVES][4][64][4];
      f32x4 v = gate_rows_tile<TX>(static_cast<const TX*>(gate.x), gate.w, T, gate.D, E, t0, 0, 0, gate.k_per_wave, tile_sh);
      const int n = wave * 8 + (lane >> 5) * 4;
      if (tid < 256) {
        if (gate.bias) {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (n + i < E) v[i] += gate.bias[n + i];
        }
        *reinterpret_cast<f32x4*>(logit_sh + (lane & 31) * kPitch + n) = v;
      }
      __syncthreads();
    } else {
      if (c == 0 && stats) __syncthreads();  // the shares are zero before a wave adds to its own
    }
    // ---- selection: one token per row of 16 lanes; waves without a token have nothing to select
    if (t0 + (wave << 2) < T) {
      const int t_raw = t0 + (tid >> 4);
      const bool live = t_raw < T;
      const int t = live ? t_raw : T - 1;
      float x[VPR], s[VPR], cutoff;
      if constexpr (kGate) {
#pragma unroll
        for (int j = 0; j < VPR; ++j) x[j] = FULL || l * VPR + j < E ? logit_sh[(tid >> 4) * kPitch + l * VPR + j] : -INFINITY;
      } else {
        load_row<VPR, FULL>(partial + static_cast<int64_t>(t) * E, l, E, x);
      }
      // Partial sums requested together, as many as registers hold: seven slices of 256 experts were four waits for loads and are two.  That and
      // the fence above, one rank's share, forward of 12, 20 and 32 tokens, us: 180 / 177.7, 199.3 / 197.2, 251.4 / 248.8.
      constexpr int kAhead = VPR < 16 ? 4 : kLanes <= 512 ? 6 : 3;
      for (int z0 = 1; z0 < splits; z0 += kAhead) {
        float y[kAhead][VPR];
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
          load_row<VPR, FULL>(partial + (static_cast<int64_t>(min(z0 + i, splits - 1)) * T + t) * E, l, E, y[i]);
#pragma unroll
        for (int i = 0; i < kAhead; ++i)
#pragma unroll
          for (int j = 0; j < VPR; ++j) x[j] = z0 + i < splits ? x[j] + y[i][j] : x[j];
      }
      if (splits > 1 && logit_bias) {
#pragma unroll
        for (int j = 0; j < VPR; ++j)
          if (FULL || l * VPR + j < E) x[j] += logit_bias[l * VPR + j];
      }
      if (logits_out && live) {
#pragma unroll
        for (int j = 0; j < VPR; ++j)
          if (FULL || l * VPR + j < E) logits_out[static_cast<int64_t>(t) * E + l * VPR + j] = x[j];
      }
      const RowChoice ch = select_row<VPR, FULL>(sel, x, l, st.scores || st.f, st.cutoff != nullptr, s, cutoff);
      if (st.scores && live) {
#pragma unroll
        for (int j = 0; j < VPR; ++j)
          if (FULL || l * VPR + j < E) st.scores[static_cast<int64_t>(t) * E + l * VPR + j] = s[j];
      }
      if (st.cutoff && live && l == 0) st.cutoff[t] = cutoff;
      if (st.f) {
        // the token's scores over their sum, added up over the wave's four rows, then the wave's tokens
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < VPR; ++j) sum += s[j];
        sum = row_sum(sum);
        const float inv = live && !(st.padding && st.padding[t]) ? 1.0f / fmaxf(sum, 1e-12f) : 0.0f;
#pragma unroll
        for (int j = 0; j < VPR; ++j) {
          float v = s[j] * inv;
          v += __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x401f));  // lane ^ 16
          v += __shfl_xor(v, 32, kWave);
          if (lane < 16 && (FULL || l * VPR + j < E)) share[wave * E + l * VPR + j] += v;
        }
      }
      if (l < K) {
        const int at = (tid >> 4) * K + l;
        id_sh[at] = static_cast<uint16_t>(live && ch.id >= 0 && ch.id < E ? ch.id : 0xffff);
        w_sh[at] = ch.weight;
        if (live) {
          weights[static_cast<int64_t>(t) * K + l] = ch.weight;
          ids[static_cast<int64_t>(t) * K + l] = ch.id;
        }
      }
    }
    __syncthreads();
    // (the ids of the chunk's missing tokens were not written: their slots are past T * K)
    // ---- rank of each slot among the chunk's earlier slots of its expert
    const int slot = t0 * K + tid;
    const bool slot_here = tid < kRows * K && slot < T * K;
    const int e = slot_here ? id_sh[tid] : 0xffff;
    const bool valid = e != 0xffff;
    unsigned long long same = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; ++b) {
      const bool bit = (e >> b) & 1;
      const unsigned long long set = __ballot(bit);
      same &= bit ? set : ~set;
    }
    const unsigned long long lower = (1ull << lane) - 1;
    const int below = __popcll(same & lower);
    if (valid && below == 0) cnt[wave * E + e] = __popcll(same);  // the lowest lane of each expert
    if (stats) {
      const bool counts = valid && !(st.padding && st.padding[slot / K]);
      const int n = __popcll(same & __ballot(counts));
      if (valid && below == 0 && n) atomicAdd(&valid_run[e], n);
    }
    __syncthreads();
    for (int i = tid; i < E; i += kLanes) {
      int r = run[i], v[kWaves];  // (all read before the first write: the compiler sees one array)
#pragma unroll
      for (int w = 0; w < kWaves; ++w) v[w] = cnt[w * E + i];
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        cnt[w * E + i] = r;
        r += v[w];
      }
      run[i] = r;
    }
    __syncthreads();
    my_e = valid ? e : -1;
    my_rank = valid ? cnt[wave * E + e] + below : 0;
    if (!single && slot_here) rank_in_block[slot] = static_cast<uint32_t>(my_rank);
    if (c + 1 < chunks) __syncthreads();  // cnt and id_sh are reused
  }
  if (stats) {
    __syncthreads();
    for (int e = tid; e < E; e += kLanes) {
      st.block_valid[static_cast<int64_t>(blockIdx.x) * E + e] = valid_run[e];
      float v = 0.0f;
#pragma unroll
      for (int w = 0; w < kWaves; ++w) v += share[w * E + e];
      if (st.f) st.block_share[static_cast<int64_t>(blockIdx.x) * E + e] = v;
    }
  }
  if (!single) {
    for (int e = tid; e < E; e += kLanes) block_hist[static_cast<int64_t>(blockIdx.x) * E + e] = run[e];
    return;
  }
  if (stats) {
    int valid = 0;
    float share = 0.0f;
    if (tid < E) {  // (each lane reads back the counts it wrote)
      valid = st.block_valid[tid];
      share += st.f ? st.block_share[tid] : 0.0f;
      if (st.valid_counts) st.valid_counts[tid] = valid;
    }
    finish_loss(st, E, valid, share, red_sh);
  }
  const LayoutLds s(extra, E);
  for (int e = tid; e < E; e += kLanes) {
    s.count[e] = run[e];
    s.before[e] = 0;
  }
  __syncthreads();
  plan_layout(s, p, true);
  write_lists(s, p, E);
  if (tid < T * K && tid < kRows * K) place_slot(s, p, tid, my_e, my_rank, K, w_sh[tid]);
}

// What a router that keeps statistics has done behind the plan's nb workgroups, by workgroups of their own: one for the sums (counts or loss wanted), the
// histogram's (groups > 0).  Both are chains of latency that nothing here waits for: at 3000 tokens of 64 experts the sums made the first workgroup the
// last to end (16 us for 7), and a launch of its own for the histogram took 10 more; together 395 -> 381 us of a training step of 1024 x 64 x 512.
struct Behind {
  int nb;
  StatsOut st;
  Observe observe;
  int groups;
};
// (a router without statistics, with those arguments and branches / without: 512 tokens of 8 experts 5.5 / 4.4 us, 1531 of 16 5.7 / 4.8, 8192 of 128 12.0 / 10.7)
struct NothingBehind {};

template <int kLanes, typename Extra>
__global__ __launch_bounds__(kLanes) void route_rows_kernel(const float* __restrict__ weights,
                                                            const int64_t* __restrict__ ids,
                                                            const uint32_t* __restrict__ rank_in_block,
                                                            const int32_t* __restrict__ block_hist, int T, int E, int K,
                                                            int tokens /* of a workgroup */, PlanOut p, Extra behind) {
  extern __shared__ int32_t lds[];
  const LayoutLds s(lds, E);
  const int tid = threadIdx.x;
  int nb = gridDim.x;
  if constexpr (std::is_same_v<Extra, Behind>) {
    __shared__ float red_sh[2 * kLanes / kWave];
    nb = behind.nb;
    const StatsOut& st = behind.st;
    int extra = static_cast<int>(blockIdx.x) - nb;
    if (extra >= 0 && (st.valid_counts || st.f)) {
      if (extra == 0) {
        int valid = 0;
        float share = 0.0f;
        sum_blocks<kLanes>(st, E, nb, lds, valid, share);
        if (st.valid_counts && tid < E) st.valid_counts[tid] = valid;
        finish_loss(st, E, valid, share, red_sh);
        return;
      }
      --extra;
    }
    if (extra >= 0) {
      observe_part<kLanes>(behind.observe, extra % behind.groups, extra / behind.groups, reinterpret_cast<unsigned*>(lds), red_sh);
      return;
    }
  }
  for (int e = tid; e < E; e += kLanes) s.count[e] = s.before[e] = 0;
  __syncthreads();
  // every expert's slots in all workgroups and in those before this one, a slice of the histograms
  // per lane, sixteen loads in flight
  const int parts = max(1, kLanes / E), per = (nb + parts - 1) / parts;
  constexpr int kBatch = 16;
  for (int idx = tid; idx < E * parts; idx += kLanes) {
    const int e = idx % E, b0 = (idx / E) * per, b1 = min(nb, b0 + per);
    int all = 0, before = 0;
    for (int b = b0; b < b1; b += kBatch) {
      int v[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) v[i] = b + i < b1 ? block_hist[static_cast<int64_t>(b + i) * E + e] : 0;
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        all += v[i];
        before += b + i < static_cast<int>(blockIdx.x) ? v[i] : 0;
      }
    }
    if (all) atomicAdd(&s.count[e], all);
    if (before) atomicAdd(&s.before[e], before);
  }
  __syncthreads();
  plan_layout(s, p, blockIdx.x == 0);
  if (blockIdx.x == 0) write_lists(s, p, E);
  const int per_block = tokens * K;
  const int first = blockIdx.x * per_block, last = min(T * K, first + per_block);
  for (int slot = first + tid; slot < last; slot += kLanes) {
    const int64_t e = ids[slot];
    place_slot(s, p, slot, e >= 0 && e < E ? static_cast<int>(e) : -1, static_cast<int>(rank_in_block[slot]), K,
               weights[slot]);
  }
}

// Lanes per workgroup.  Selection is bound by instruction issue, so its tokens want to be spread over the
// CUs: 512 lanes, as long as each of at most kMaxBlocks workgroups has one chunk of tokens (8192).  Every workgroup of
// route_rows reads all histograms, so with more than 128 experts the line lies lower.  Up to 64 tokens one
// workgroup does everything, with 512 lanes where they hold the tokens (32): fewer waves to clear counters for and to
// meet at barriers.  All launches together, us, 512 / 1024 lanes:
//   experts, choices   8 tokens    32           33           64           1000         7000         8192         9000
//    64, 6              7.5 / 8.1   8.2 / 8.7   11.3 / 9.6   11.3 / 10.5  11.9 / 14.7  14.2 / 15.5  14.2 / 15.7  17.6 / 15.9
//   128, 8              9.5 / 10.3 10.9 / 11.6  13.8 / 12.2  13.9 / 13.7  14.9 / 18.0  18.8 / 19.9  19.4 / 20.1  24.1 / 21.3
//   256, 8             14.1 / 14.4 16.9 / 17.4  20.3 / 18.7  20.9 / 21.5  21.5 / 26.3  29.0 / 29.8  31.3 / 29.2  37.1 / 31.6
//   Of 65 to 512 tokens four waves, one to a SIMD: two that share one take turns, and there are CUs enough.  (Not with up to 32 experts, whose selection is
// short and has the gate's projection in front, eight waves' work.)  The second launch keeps to 512 lanes.  Block forward, us, eight waves / four: one rank's share of 256 experts of
// 7168 x 2048, 80 tokens 317.3 / 313.6, 128 352.4 / 350.3, 256 419.6 / 413.3, 512 433.1 / 434.1; 64 of 1024 x 512, six each, 100 54.2 / 53.4, 300 56.8 / 56.1, 1000
// 70.2 / 69.9; 128 of 2048 x 768, 256 221.1 / 220.4, 512 to 3000 the same within the spread.
int route_lanes(int64_t T, int64_t E) {
  if (E > 32 && T > 64 && T <= 512) return 256;
  return T <= 32 || (T > 64 && T <= (E > 128 ? 7000 : 8192)) ? 512 : 1024;
}
int route_chunks(int64_t T, int64_t E) {
  const int64_t rows = route_lanes(T, E) / 16, groups = (T + rows - 1) / rows;
  return static_cast<int>((groups + kMaxBlocks - 1) / kMaxBlocks);
}
int64_t route_tokens(int64_t T, int64_t E) { return static_cast<int64_t>(route_chunks(T, E)) * (route_lanes(T, E) / 16); }  // of a workgroup
int64_t route_blocks(int64_t T, int64_t E) {
  const int64_t per = route_tokens(T, E);
  return (T + per - 1) / per;
}
// calls f(integral_constant lanes)
template <typename Fn>
void with_lanes(int64_t T, int64_t E, Fn f) {
  const int lanes = route_lanes(T, E);
  if (lanes == 256) f(std::integral_constant<int, 256>{});
  else if (lanes == 512) f(std::integral_constant<int, 512>{});
  else f(std::integral_constant<int, 1024>{});
}

}  // namespace
}  // namespace mi355

using namespace mi355;

extern "C" int mi355_route_plan_covers(int64_t E, int64_t K, int num_groups, int select_mode) {
  return E >= 1 && K >= 1 && K <= E && select_row_covers(E, K, num_groups, select_mode) ? 1 : 0;
}

extern "C" int64_t mi355_route_plan_workspace_bytes(int64_t T, int64_t K, int64_t E) {
  if (K < 1 || E < 1 || T < 1 || route_blocks(T, E) == 1) return 0;
  return (T * K + route_blocks(T, E) * E) * (int64_t)sizeof(int32_t);
}
extern "C" int64_t mi355_route_stats_workspace_bytes(int64_t T, int64_t E) {
  return T < 1 || E < 1 ? 0 : 2 * route_blocks(T, E) * E * (int64_t)sizeof(int32_t);
}

static int route_plan(const float* partial, int splits, const float* logit_bias, float* logits,
                                const float* expert_bias, int64_t T, int64_t E, int64_t K, int score_func,
                                int route_norm, float route_scale, int num_groups, int num_limited, float* weights,
                                int64_t* ids, int64_t lo, int64_t hi, int64_t align, int64_t tile_m,
                                int32_t* counts_E, int32_t* seg_offsets, int32_t* seg_counts, int32_t* row_of_slot,
                                int32_t* slot_of_row, int32_t* token_of_row, float* row_scale, int64_t row_capacity,
                                int32_t* tile_expert, int32_t* tile_row0, int32_t* num_tiles, int64_t tile_capacity,
                                void* workspace, const StatsOut& st, void* stream, const GateIn& gate = {},
                                int x_dtype = MI355_F32, int64_t* histogram = nullptr, int64_t B = 1) {
  MI355_REQUIRE(T >= 1 && T < (1ll << 26) && E >= 1 && K >= 1 && K <= E && T * K < (1ll << 30),
                "route_plan: bad shape T=%lld E=%lld K=%lld", (long long)T, (long long)E, (long long)K);
  if (!select_row_covers(E, K, num_groups, MI355_SELECT_TOPK))
    return fail(MI355_EUNSUP, "route_plan: E=%lld K=%lld G=%d is not covered; use mi355_router_select_fwd and "
                              "mi355_permute_plan", (long long)E, (long long)K, num_groups);
  MI355_REQUIRE(score_func >= 0 && score_func <= 2, "route_plan: unknown score_func %d", score_func);
  if (num_groups > 0)
    MI355_REQUIRE(E % num_groups == 0 && E / num_groups >= 2 && num_limited >= 1 && num_limited <= num_groups &&
                      K <= (int64_t)num_limited * (E / num_groups),
                  "route_plan: bad group config G=%d L=%d", num_groups, num_limited);
  MI355_REQUIRE(0 <= lo && lo < hi && hi <= E, "route_plan: bad local range [%lld,%lld)", (long long)lo, (long long)hi);
  MI355_REQUIRE(align >= 1 && tile_m >= 1 && align < (1ll << 20) && tile_m < (1ll << 20), "route_plan: align and tile_m must be positive");
  MI355_REQUIRE(row_capacity >= 1 && row_capacity < (1ll << 31) && tile_capacity >= 1 && tile_capacity < (1ll << 31),
                "route_plan: bad capacity");
  MI355_REQUIRE((gate.x || (partial && splits >= 1 && aligned16(partial))) && weights && ids && counts_E && seg_offsets &&
                    seg_counts && row_of_slot && slot_of_row && token_of_row && tile_expert && tile_row0 && num_tiles,
                "route_plan: null or misaligned pointer");
  MI355_REQUIRE(route_blocks(T, E) == 1 || workspace, "route_plan: workspace required");
  hipStream_t s = as_stream(stream);
  const SelectArgs sel{expert_bias, (int)E, (int)K, score_func, route_norm, route_scale, num_groups, num_limited};
  const PlanOut p{(int)lo, (int)hi, (int)align, (int)tile_m, (int)row_capacity, (int)tile_capacity, counts_E,
                  seg_offsets, seg_counts, row_of_slot, slot_of_row, token_of_row, row_scale, tile_expert, tile_row0,
                  num_tiles};
  const int chunks = route_chunks(T, E);
  const int blocks = (int)route_blocks(T, E);
  uint32_t* rank = static_cast<uint32_t*>(workspace);
  int32_t* hist = reinterpret_cast<int32_t*>(rank + (blocks > 1 ? T * K : 0));
  // every row has a slot when all experts are local and nothing is padded
  const int fill = !(lo == 0 && hi == E && align == 1 && row_capacity == T * K);
  const bool stats = st.valid_counts || st.f;
  const int waves = route_lanes(T, E) / kWave;
  const size_t lds = ((1 + waves) * E * (stats ? 2 : 1) + (blocks == 1 ? layout_words((int)E) : 0)) * sizeof(int32_t);
  with_row_shape(E, [&](auto vpr, auto full) {
    if constexpr (decltype(vpr)::value <= 2) {
      if (gate.x) {
        constexpr int V = decltype(vpr)::value;
        constexpr bool F = decltype(full)::value;
        hipLaunchKernelGGL((x_dtype == MI355_BF16 ? route_rank_kernel<V, F, 512, uint16_t> : route_rank_kernel<V, F, 512, float>),
                           dim3(blocks), dim3(512), lds, s, gate, nullptr, 1, nullptr, logits, sel, weights, ids, rank, hist,
                           (int)T, chunks, fill, p, st);
        return;
      }
    }
    with_lanes(T, E, [&](auto lanes) {
      hipLaunchKernelGGL((route_rank_kernel<decltype(vpr)::value, decltype(full)::value, decltype(lanes)::value>), dim3(blocks),
                         dim3(lanes), lds, s, GateIn{}, partial, splits, logit_bias, logits, sel, weights, ids, rank, hist, (int)T,
                         chunks, fill, p, st);
    });
  });
  if (int rc = check_launch("route_rank")) return rc;
  Observe o{st.scores, st.cutoff, expert_bias, st.padding, reinterpret_cast<unsigned long long*>(histogram), (int)T, (int)E, (int)B, 0, 0};
  unsigned groups = 0, token_chunks = 0;
  if (histogram && blocks > 1) observe_shape(T, E, B, o.eg, o.tokens, groups, token_chunks);
  if (blocks > 1) {
    with_lanes(T, E, [&](auto lanes) {
      constexpr int kLanes = std::max(512, decltype(lanes)::value);
      auto rows = [&](auto kernel, unsigned grid, size_t words, auto behind) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(kLanes), words * sizeof(int32_t), s, weights, ids, rank, hist, (int)T, (int)E, (int)K,
                           (int)route_tokens(T, E), p, behind);
      };
      const size_t words = layout_words((int)E);
      if (stats || groups > 0)
        rows(route_rows_kernel<kLanes, Behind>, blocks + (stats ? 1 : 0) + groups * token_chunks,
             std::max<size_t>({words, (size_t)o.eg * o.B, stats ? (size_t)kStatsWords<kLanes> : 0}), Behind{blocks, st, o, (int)groups});
      else
        rows(route_rows_kernel<kLanes, NothingBehind>, blocks, words, NothingBehind{});
    });
    if (int rc = check_launch("route_rows")) return rc;
  }
  if (histogram && groups == 0)
    return mi355_quantile_observe(st.scores, st.cutoff, expert_bias, st.padding, histogram, T, E, B, stream);
  return MI355_OK;
}

extern "C" int mi355_route_plan(const float* partial, int splits, const float* logit_bias, float* logits,
                                const float* expert_bias, int64_t T, int64_t E, int64_t K, int score_func,
                                int route_norm, float route_scale, int num_groups, int num_limited, float* weights,
                                int64_t* ids, int64_t lo, int64_t hi, int64_t align, int64_t tile_m,
                                int32_t* counts_E, int32_t* seg_offsets, int32_t* seg_counts, int32_t* row_of_slot,
                                int32_t* slot_of_row, int32_t* token_of_row, float* row_scale, int64_t row_capacity,
                                int32_t* tile_expert, int32_t* tile_row0, int32_t* num_tiles, int64_t tile_capacity,
                                void* workspace, void* stream) {
  return route_plan(partial, splits, logit_bias, logits, expert_bias, T, E, K, score_func, route_norm, route_scale,
                    num_groups, num_limited, weights, ids, lo, hi, align, tile_m, counts_E, seg_offsets, seg_counts,
                    row_of_slot, slot_of_row, token_of_row, row_scale, row_capacity, tile_expert, tile_row0, num_tiles,
                    tile_capacity, workspace, StatsOut{}, stream);
}

extern "C" int mi355_route_plan_observe(
    const float* partial, int splits, const float* logit_bias, float* logits, const float* expert_bias, int64_t T,
    int64_t E, int64_t K, int score_func, int route_norm, float route_scale, int num_groups, int num_limited,
    float* weights, int64_t* ids, int64_t lo, int64_t hi, int64_t align, int64_t tile_m, int32_t* counts_E,
    int32_t* seg_offsets, int32_t* seg_counts, int32_t* row_of_slot, int32_t* slot_of_row, int32_t* token_of_row,
    float* row_scale, int64_t row_capacity, int32_t* tile_expert, int32_t* tile_row0, int32_t* num_tiles,
    int64_t tile_capacity, void* workspace, const uint8_t* padding_mask_T, int32_t* valid_counts_E, float* scores_TE,
    float* cutoff_T, float* aux_f_E, float* aux_scale, void* aux_acc, int aux_acc_dtype, const float* aux_denominator, float aux_coeff,
    void* stats_workspace, int64_t* histogram_EB, int64_t B, void* stream) {
  MI355_REQUIRE(!histogram_EB || (scores_TE && cutoff_T && expert_bias && B >= 1 && B < (1 << 24)),
                "route_plan_observe: the histogram needs scores, cutoff, the expert bias and 1 <= B < 2^24 (%lld)", (long long)B);
  MI355_REQUIRE(!cutoff_T || K < E, "route_plan_observe: top_k (%lld) must leave a (K+1)-th expert of %lld", (long long)K,
                (long long)E);
  MI355_REQUIRE(!aux_f_E || (aux_scale && aux_denominator), "route_plan_observe: the loss needs scale and denominator");
  MI355_REQUIRE(!aux_acc || aux_acc_dtype == MI355_F32 || aux_acc_dtype == MI355_BF16, "route_plan_observe: aux_acc is fp32 or bf16");
  MI355_REQUIRE((!aux_f_E && !valid_counts_E) || stats_workspace, "route_plan_observe: workspace required");
  int32_t* block_valid = static_cast<int32_t*>(stats_workspace);
  float* block_share = block_valid ? reinterpret_cast<float*>(block_valid + (T >= 1 ? route_blocks(T, E) : 0) * E) : nullptr;
  const StatsOut st{padding_mask_T, valid_counts_E, scores_TE, cutoff_T, aux_f_E, aux_scale, aux_acc, aux_acc_dtype, aux_denominator,
                    aux_coeff, block_valid, block_share};
  return route_plan(partial, splits, logit_bias, logits, expert_bias, T, E, K, score_func, route_norm, route_scale,
                    num_groups, num_limited, weights, ids, lo, hi, align, tile_m, counts_E, seg_offsets, seg_counts,
                    row_of_slot, slot_of_row, token_of_row, row_scale, row_capacity, tile_expert, tile_row0, num_tiles,
                    tile_capacity, workspace, st, stream, {}, MI355_F32, histogram_EB, B);
}

extern "C" int mi355_route_plan_stats(
    const float* partial, int splits, const float* logit_bias, float* logits, const float* expert_bias, int64_t T,
    int64_t E, int64_t K, int score_func, int route_norm, float route_scale, int num_groups, int num_limited,
    float* weights, int64_t* ids, int64_t lo, int64_t hi, int64_t align, int64_t tile_m, int32_t* counts_E,
    int32_t* seg_offsets, int32_t* seg_counts, int32_t* row_of_slot, int32_t* slot_of_row, int32_t* token_of_row,
    float* row_scale, int64_t row_capacity, int32_t* tile_expert, int32_t* tile_row0, int32_t* num_tiles,
    int64_t tile_capacity, void* workspace, const uint8_t* padding_mask_T, int32_t* valid_counts_E, float* scores_TE,
    float* cutoff_T, float* aux_f_E, float* aux_scale, void* aux_acc, int aux_acc_dtype, const float* aux_denominator, float aux_coeff,
    void* stats_workspace, void* stream) {
  return mi355_route_plan_observe(partial, splits, logit_bias, logits, expert_bias, T, E, K, score_func, route_norm, route_scale, num_groups,
                                  num_limited, weights, ids, lo, hi, align, tile_m, counts_E, seg_offsets, seg_counts, row_of_slot,
                                  slot_of_row, token_of_row, row_scale, row_capacity, tile_expert, tile_row0, num_tiles, tile_capacity,
                                  workspace, padding_mask_T, valid_counts_E, scores_TE, cutoff_T, aux_f_E, aux_scale, aux_acc,
                                  aux_acc_dtype, aux_denominator, aux_coeff, stats_workspace, nullptr, 1, stream);
}

// whole chunks of 32 tokens, one to a workgroup, and one slice of the contraction: the bits of the two calls
extern "C" int mi355_route_gate_plan_covers(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E, int64_t K, int num_groups) {
  return E <= R_BN && mi355_route_plan_covers(E, K, num_groups, MI355_SELECT_TOPK) && T >= 1 && T < (1ll << 26) &&
         route_lanes(T, E) == 512 && route_chunks(T, E) == 1 && router_fwd_splits(x_dtype, w_dtype, T, D, E) == 1 ? 1 : 0;
}

extern "C" int mi355_route_gate_plan_stats(
    const void* x, int x_dtype, const float* w, int64_t D, const float* logit_bias, float* logits, const float* expert_bias,
    int64_t T, int64_t E, int64_t K, int score_func, int route_norm, float route_scale, int num_groups, int num_limited,
    float* weights, int64_t* ids, int64_t lo, int64_t hi, int64_t align, int64_t tile_m, int32_t* counts_E,
    int32_t* seg_offsets, int32_t* seg_counts, int32_t* row_of_slot, int32_t* slot_of_row, int32_t* token_of_row,
    float* row_scale, int64_t row_capacity, int32_t* tile_expert, int32_t* tile_row0, int32_t* num_tiles,
    int64_t tile_capacity, void* workspace, const uint8_t* padding_mask_T, int32_t* valid_counts_E, float* scores_TE,
    float* cutoff_T, float* aux_f_E, float* aux_scale, void* aux_acc, int aux_acc_dtype, const float* aux_denominator, float aux_coeff,
    void* stats_workspace, void* stream) {
  if (!mi355_route_gate_plan_covers(x_dtype, MI355_F32, T, D, E, K, num_groups))
    return fail(MI355_EUNSUP, "route_gate_plan_stats: not covered; use mi355_router_gate_fwd_partial and mi355_route_plan_stats");
  MI355_REQUIRE(x && w && aligned16({x, w}), "route_gate_plan_stats: null or misaligned pointer");
  MI355_REQUIRE(!cutoff_T || K < E, "route_gate_plan_stats: top_k (%lld) must leave a (K+1)-th expert of %lld", (long long)K,
                (long long)E);
  MI355_REQUIRE(!aux_f_E || (aux_scale && aux_denominator), "route_gate_plan_stats: the loss needs scale and denominator");
  MI355_REQUIRE(!aux_acc || aux_acc_dtype == MI355_F32 || aux_acc_dtype == MI355_BF16, "route_gate_plan_stats: aux_acc is fp32 or bf16");
  MI355_REQUIRE((!aux_f_E && !valid_counts_E) || stats_workspace, "route_gate_plan_stats: workspace required");
  int32_t* block_valid = static_cast<int32_t*>(stats_workspace);
  float* block_share = block_valid ? reinterpret_cast<float*>(block_valid + (T >= 1 ? route_blocks(T, E) : 0) * E) : nullptr;
  const StatsOut st{padding_mask_T, valid_counts_E, scores_TE, cutoff_T, aux_f_E, aux_scale, aux_acc, aux_acc_dtype, aux_denominator,
                    aux_coeff, block_valid, block_share};
  const GateIn gate{x, w, logit_bias, (int)D, gate_rows_k(D, 1)};
  return route_plan(nullptr, 1, nullptr, logits, expert_bias, T, E, K, score_func, route_norm, route_scale,
                    num_groups, num_limited, weights, ids, lo, hi, align, tile_m, counts_E, seg_offsets, seg_counts,
                    row_of_slot, slot_of_row, token_of_row, row_scale, row_capacity, tile_expert, tile_row0, num_tiles,
                    tile_capacity, workspace, st, stream, gate, x_dtype);
}
