// Router projections on the bf16 matrix cores with fp32 accuracy.
//
// The router gate is an fp32 GEMM over bf16 activations (x) and fp32 weights (W).  A
// bf16 value times a bf16 value is exact in fp32, so an fp32 operand written as the sum of
// three bf16 pieces (hi + mid + lo, 24 mantissa bits) turns the fp32 product into three
// bf16 MFMAs that accumulate in fp32 -- 16x the rate of the fp32 MFMA for 3x the
// instructions, which makes all three projections memory bound:
//   logits = x . W^T            x exact in bf16, W in three pieces
//   dW     = dlogits^T . x      dlogits in three pieces (split while it is staged)
//   dx     = dlogits . W        rounded to bf16 on output, so hi.hi + hi.mid + mid.hi
//                               (relative error 2^-16) is enough
// Shapes: D and E multiples of 64; anything else stays on the strided fp32-MFMA kernels.
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "bf16_tiles.h"
#include "common.h"
#include "gate_rows.h"
#include "gemm_generic.h"
#include "router_few.h"

namespace mi355 {
namespace {

__device__ __forceinline__ int kc_off(int row, int chunk) {
  return row * BK + ((chunk ^ ((row >> 1) & 7)) << 3);
}
template <int COLS>
__device__ __forceinline__ int ks_off(int k, int chunk) {
  return k * COLS + ((chunk ^ ks_key(k)) << 3);
}

// W (n fp32) -> out[s][n] bf16, s < nsplit
__global__ __launch_bounds__(256) void split_kernel(const float* __restrict__ w, uint16_t* __restrict__ out,
                                                    int64_t n, int nsplit) {
  const int64_t i = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  if (i >= n) return;  // n is a multiple of 8 (D % 64 == 0)
  const f32x4 a = *reinterpret_cast<const f32x4*>(w + i);
  const f32x4 b = *reinterpret_cast<const f32x4*>(w + i + 4);
  u32x4 hi, mid, lo;
  split8(a, b, hi, mid, lo);
  *reinterpret_cast<u32x4*>(out + i) = hi;
  *reinterpret_cast<u32x4*>(out + n + i) = mid;
  if (nsplit > 2) *reinterpret_cast<u32x4*>(out + 2 * n + i) = lo;
}

// ---- logits(T,E) = x(T,D) . W(E,D)^T + bias, few tokens or any widths --------------------
// Bound by latency: at one token the product is one read of W (1 MB at 128 x 2048), which wants to
// be in flight all at once and in as few launches as possible.  A workgroup takes 32 tokens x up to 32
// experts and a slice of the contraction; its eight waves split that slice, and every wave reads
// its operands straight into MFMA fragments (no LDS, no barrier in the loop; a weight is used by
// one wave of one workgroup per 32 tokens), the fp32 weights becoming their three bf16 pieces in
// registers on the way.  The eight partial tiles are added in wave order through LDS.  The order
// of k inside a 32-wide step is a permutation (lane half h holds k = 16 h ..) that both operands
// share, so that each lane reads whole 32- or 64-byte pieces of a row.
// This replaces a kernel that walked the whole contraction in 128-expert tiles behind a separate
// weight-splitting launch: 1 token of 2048 x 128 experts 34 -> 8 us, 1000 tokens 43 -> 12 us, 128
// tokens of 7168 x 256 experts 131 -> 12 us (profiled inside the block, the weights from memory).  From 1024 tokens and 192 Mi products on, with widths on its grid, the
// 128-token kernel below reads the weights four times less often and is the faster one.
template <typename TX, int BN, bool KEEP>
__global__ __launch_bounds__(64 * R_WAVES) void gate_rows_kernel(const TX* __restrict__ x,
                                                                 const float* __restrict__ w,
                                                                 const float* __restrict__ bias,
                                                                 float* __restrict__ out, int T, int D, int E,
                                                                 int k_per_wave, uint16_t* __restrict__ keep) {
  __shared__ __attribute__((aligned(16))) float red[R_WAVES][4][64][4];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, q = tid >> 6;
  const int t0 = blockIdx.x * R_BM, n0 = blockIdx.y * BN;
  f32x4 v = gate_rows_tile<TX, BN, KEEP>(x, w, T, D, E, t0, n0, blockIdx.z, k_per_wave, red, blockIdx.x == 0 ? keep : nullptr);
  if (tid >= 8 * BN) return;
  const int t = t0 + (lane & 31), n = n0 + q * 8 + half * 4;
  if (t >= T || n >= E) return;
  float* dst = out + (static_cast<int64_t>(blockIdx.z) * T + t) * E + n;
  if (bias) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < E) v[i] += bias[n + i];
  }
  if (E % 4 == 0) {
    *reinterpret_cast<f32x4*>(dst) = v;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < E) dst[i] = v[i];
  }
}

// Splits of the contraction over workgroups: about 128 of it per wave (one batch of requests)
// while that leaves the launch below four workgroups a CU; each split costs its consumer one
// more read of the (T, E) partial sums.  The number decides the order in which a logit is summed, and so which of two experts whose logits
// are equal to the last bits a token takes: it is not a setting to be moved with the number of tokens.
int rows_splits(int64_t T, int64_t D, int64_t E) {
  const int64_t tiles = ((T + R_BM - 1) / R_BM) * ((E + R_BN - 1) / R_BN);
  const int64_t want = (D + 128 * R_WAVES - 1) / (128 * R_WAVES);
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>({want, 8, 1024 / tiles})));
}

// Experts a workgroup takes: as few of 32, 16 and 8 as leave it a CU of its own.  Fewer of them are less for a wave to wait for, at
// the same sums.  Block forward of 128 experts of 2048 x 768, eight a token, us, 32 / 16 / 8: one token (8 workgroups of 32) 28.5 / 27.2 /
// 26.5, four 67.6 / 66.2 / 65.4, 33 tokens (16) 210.0 / 207.6 / 206.8, 200 (56) 243.9 / 242.0 / 241.3, 500 (128) 255.9 / 254.0 / 258.1, 1000
// (256) 271.8 / 275.7 / 283.7; 300 of 64 of 1536 x 640, four each (40), 117.2 / 115.5 / 114.5; 128 of one rank's share of 256 of
// 7168 x 2048 (224) 454 / 458 / 465.
int rows_experts(int64_t t_tiles, int64_t E, int splits) {
  const int64_t parts = t_tiles * ((E + R_BN - 1) / R_BN) * splits;
  return parts <= 64 ? 8 : parts <= 128 ? 16 : R_BN;
}

// The same product for many tokens: 128 tokens x 128 experts per workgroup, 8 waves as 2 x 4
// (each 64 tokens x 32 experts), the contraction split over gridDim.z so that the grid still
// fills the chip.  The kernel above reads the weights once per 32 tokens -- at T = 8192 that is
// 0.25 GB through L2 and a conversion each time for a 37 MB problem; this one streams the weight
// pieces, split beforehand, once per 128 tokens.  Partial sums go to the workspace and are added
// (with the bias) in split order by logits_reduce_kernel; a single split writes logits itself.
constexpr int G_BM = 128, G_BN = 128, G_NT = 512;
constexpr int G_STAGE = (G_BM + 3 * G_BN) * BK;  // elements, 64 KiB

__global__ __launch_bounds__(G_NT, 2) void gate_fwd_wide_kernel(const uint16_t* __restrict__ x,
                                                                const uint16_t* __restrict__ ws,
                                                                const float* __restrict__ bias,
                                                                float* __restrict__ out, int T, int D, int E,
                                                                int k_per_split) {
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 2) * 64, wn = (wave & 3) * 32;
  const int t0 = blockIdx.x * G_BM, n0 = blockIdx.y * G_BN;
  const int k_begin = blockIdx.z * k_per_split;
  const int ksteps = min(k_per_split, D - k_begin) / BK;
  const int row = tid >> 3, chunk = tid & 7;  // 64 rows per pass
  const int64_t ED = static_cast<int64_t>(E) * D;
  const uint16_t* ap[2];
  const uint16_t* bp[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    ap[i] = x + static_cast<int64_t>(min(t0 + row + 64 * i, T - 1)) * D + k_begin + chunk * 8;
    bp[i] = ws + static_cast<int64_t>(min(n0 + row + 64 * i, E - 1)) * D + k_begin + chunk * 8;
  }
  const int lds0 = kc_off(row, chunk);  // + 64 rows * BK per pass (64 % 16 == 0: same swizzle key)
  u32x4 ra[2], rb[6];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) ra[i] = *reinterpret_cast<const u32x4*>(ap[i] + k0);
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i) rb[p * 2 + i] = *reinterpret_cast<const u32x4*>(bp[i] + p * ED + k0);
  };
  auto park = [&](uint16_t* st) {
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(st + 64 * i * BK + lds0) = ra[i];
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<u32x4*>(st + (G_BM + p * G_BN + 64 * i) * BK + lds0) = rb[p * 2 + i];
  };
  f32x16 acc[2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
  if (ksteps > 0) {
    fetch(0);
    park(smem);
    if (ksteps > 1) fetch(BK);
  }
  __syncthreads();
  for (int ks = 0; ks < ksteps; ++ks) {
    const uint16_t* As = smem + (ks & 1) * G_STAGE;
    if (ks + 1 < ksteps) park(smem + ((ks + 1) & 1) * G_STAGE);
    if (ks + 2 < ksteps) fetch((ks + 2) * BK);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 af[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) af[m] = frag_kc(As, wm + m * 32, kk, lane);
#pragma unroll
      for (int p = 0; p < 3; ++p) {
        const bf16x8 bf = frag_kc(As + (G_BM + p * G_BN) * BK, wn, kk, lane);
#pragma unroll
        for (int m = 0; m < 2; ++m) acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf, af[m], acc[m], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // lane = token row (lane & 31); registers = expert columns (i>>2)*8 + (lane>>5)*4 + (i&3)
  float* dst = out + static_cast<int64_t>(blockIdx.z) * T * E;
  const bool direct = gridDim.z == 1;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const int t = t0 + wm + m * 32 + (lane & 31);
    if (t >= T) continue;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = n0 + wn + q * 8 + (lane >> 5) * 4;
      if (n < E) {  // E % 4 == 0
        f32x4 v = {acc[m][q * 4], acc[m][q * 4 + 1], acc[m][q * 4 + 2], acc[m][q * 4 + 3]};
        if (direct && bias) v += *reinterpret_cast<const f32x4*>(bias + n);
        *reinterpret_cast<f32x4*>(dst + static_cast<int64_t>(t) * E + n) = v;
      }
    }
  }
}

// logits[t][e] = sum over the splits, in order, of partial[z][t][e], plus bias[e]
__global__ __launch_bounds__(256) void logits_reduce_kernel(const float* __restrict__ partial,
                                                            const float* __restrict__ bias,
                                                            float* __restrict__ logits, int64_t TE, int E,
                                                            int splits) {
  const int64_t first = static_cast<int64_t>(blockIdx.x) * 1024;
  if (TE % 4) {  // (then E % 4 != 0 too, and the splits' rows are not 16-byte aligned)
    for (int64_t i = first + threadIdx.x; i < min(first + 1024, TE); i += 256) {
      float acc = partial[i];
      for (int z = 1; z < splits; ++z) acc += partial[z * TE + i];
      logits[i] = bias ? acc + bias[i % E] : acc;
    }
    return;
  }
  const int64_t i = first + threadIdx.x * 4;
  if (i >= TE) return;
  f32x4 acc = *reinterpret_cast<const f32x4*>(partial + i);
  for (int z = 1; z < splits; ++z) acc += *reinterpret_cast<const f32x4*>(partial + z * TE + i);
  if (bias) {
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[j] += bias[(i + j) % E];
  }
  *reinterpret_cast<f32x4*>(logits + i) = acc;
}

// ---- dx(T,D) = dlogits(T,E) . W(E,D), bf16 out ------------------------------------------
// Tile 128 tokens x 128 columns, 8 waves as 2 x 4, each 64 x 32.  Per K step of 64
// experts: dlogits tile split on the fly into hi / mid (KC), W hi / mid tiles KS.
constexpr int X_BM = 128, X_BN = 128, X_NT = 512;
constexpr int X_ELEMS = 2 * X_BM * BK + 2 * BK * X_BN;  // LDS of a tile: 64 KiB

// the sums of two bf16 pairs, rounded
__device__ __forceinline__ uint32_t add_bf16x2(uint32_t a, uint32_t b) {
  return pack_bf16x2(__uint_as_float(a << 16) + __uint_as_float(b << 16),
                     __uint_as_float(a & 0xffff0000u) + __uint_as_float(b & 0xffff0000u));
}

// What comes in front of the product: an addend, and (ROWS) the sum of the experts' input gradients over a token's K slots in
// ascending order, as permute_rows_bwd forms it.
struct GateSum {
  const uint16_t *addend, *rows;
  const int32_t* row_of_slot;
  int K, row_capacity;
};
constexpr int kMaxSumK = 16;

// Tile `part` of dx, column tiles of a row tile one after the other: together they read whole rows, where all row tiles of one
// column tile would read pieces a power of two apart, few memory channels at a time.
template <bool ROWS>
__device__ __forceinline__ void gate_dx_tile(const float* __restrict__ dlogits, const uint16_t* __restrict__ ws,
                                             const GateSum& g, uint16_t* __restrict__ dx, int T, int D, int E, int part,
                                             uint16_t* smem) {
  uint16_t* A_hi = smem;                    // [128][64] KC
  uint16_t* A_mid = A_hi + X_BM * BK;
  uint16_t* B_hi = A_mid + X_BM * BK;       // [64][128] KS
  uint16_t* B_mid = B_hi + BK * X_BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 2) * 64, wn = (wave & 3) * 32;
  const int col_tiles = (D + X_BN - 1) / X_BN;
  const int t0 = part / col_tiles * X_BM;
  const int n0 = min(part % col_tiles * X_BN, D - X_BN);  // D >= 128: a last tile starts early
  const int64_t ED = static_cast<int64_t>(E) * D;
  f32x16 acc[2];
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[m][i] = 0.0f;
  // One LDS stage; the operands of K step k+1 are requested into registers before the MFMAs of
  // step k (with nothing in flight during the MFMAs every step waited out a memory round trip).
  // A: 128 rows x 8 chunks of 8 experts = 1024 units, 2 per thread; B: 64 experts x 16 chunks =
  // 1024 units per piece, 2 per thread.
  f32x4 ra[2][2];
  u32x4 rb[2][2];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + X_NT * i;
      const float* src = dlogits + static_cast<int64_t>(min(t0 + (u >> 3), T - 1)) * E + k0 + (u & 7) * 8;
      ra[i][0] = *reinterpret_cast<const f32x4*>(src);
      ra[i][1] = *reinterpret_cast<const f32x4*>(src + 4);
      const uint16_t* bsrc = ws + static_cast<int64_t>(k0 + (u >> 4)) * D + n0 + (u & 15) * 8;
      rb[i][0] = *reinterpret_cast<const u32x4*>(bsrc);
      rb[i][1] = *reinterpret_cast<const u32x4*>(bsrc + ED);
    }
  };
  fetch(0);
  // this thread's pieces of the output: row (tid >> 4) + 32 i, columns 8 (tid & 15) ..
  const int o_row = tid >> 4, o_col = n0 + (tid & 15) * 8;
  constexpr int kOut = X_BM * X_BN / 8 / X_NT;  // 4
  u32x4 front[ROWS ? kOut : 1];
  if constexpr (ROWS) {
    int32_t* slots = reinterpret_cast<int32_t*>(smem + X_ELEMS);  // [128][K]
    for (int i = tid; i < X_BM * g.K; i += X_NT) slots[i] = t0 + i / g.K < T ? g.row_of_slot[static_cast<int64_t>(t0) * g.K + i] : -1;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOut; ++i) {
      const int r = o_row + 32 * i;
      float sum[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) sum[j] = 0.0f;
      constexpr int B = 8;  // rows requested together
      for (int k0 = 0; k0 < g.K; k0 += B) {
        uint4 v[B];
#pragma unroll
        for (int k = 0; k < B; ++k) {
          const int row = k0 + k < g.K ? slots[r * g.K + min(k0 + k, g.K - 1)] : -1;
          v[k] = row >= 0 && row < g.row_capacity
                     ? load_stream(reinterpret_cast<const uint4*>(g.rows + static_cast<int64_t>(row) * D + o_col))
                     : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int k = 0; k < B; ++k) {
          const uint32_t w[4] = {v[k].x, v[k].y, v[k].z, v[k].w};
#pragma unroll
          for (int j = 0; j < 8; ++j) sum[j] += __uint_as_float(j & 1 ? w[j >> 1] & 0xffff0000u : w[j >> 1] << 16);
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) front[i][j] = pack_bf16x2(sum[2 * j], sum[2 * j + 1]);
      if (g.addend && t0 + r < T) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(g.addend + static_cast<int64_t>(t0 + r) * D + o_col);
#pragma unroll
        for (int j = 0; j < 4; ++j) front[i][j] = add_bf16x2(front[i][j], a[j]);
      }
    }
  }
  for (int k0 = 0; k0 < E; k0 += BK) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + X_NT * i;
      u32x4 hi, mid, lo;
      split8(ra[i][0], ra[i][1], hi, mid, lo);
      *reinterpret_cast<u32x4*>(A_hi + kc_off(u >> 3, u & 7)) = hi;
      *reinterpret_cast<u32x4*>(A_mid + kc_off(u >> 3, u & 7)) = mid;
      *reinterpret_cast<u32x4*>(B_hi + ks_off<X_BN>(u >> 4, u & 15)) = rb[i][0];
      *reinterpret_cast<u32x4*>(B_mid + ks_off<X_BN>(u >> 4, u & 15)) = rb[i][1];
    }
    __syncthreads();
    if (k0 + BK < E) fetch(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      const bf16x8 bh = frag_ks<X_BN>(B_hi, wn, kk, lane);
      const bf16x8 bm = frag_ks<X_BN>(B_mid, wn, kk, lane);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const bf16x8 ah = frag_kc(A_hi, wm + m * 32, kk, lane);
        const bf16x8 am = frag_kc(A_mid, wm + m * 32, kk, lane);
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh, ah, acc[m], 0, 0, 0);
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bm, ah, acc[m], 0, 0, 0);
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bh, am, acc[m], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // through LDS, then whole 256-byte pieces of rows
  constexpr int PITCH = X_BN + 8;
#pragma unroll
  for (int m = 0; m < 2; ++m)
#pragma unroll
    for (int q = 0; q < 4; ++q)
      *reinterpret_cast<u32x2*>(smem + (wm + m * 32 + (lane & 31)) * PITCH + wn + q * 8 + (lane >> 5) * 4) =
          u32x2{pack2(acc[m][q * 4], acc[m][q * 4 + 1]), pack2(acc[m][q * 4 + 2], acc[m][q * 4 + 3])};
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kOut; ++i) {
    const int r = o_row + 32 * i;
    if (t0 + r >= T) continue;
    const int64_t at = static_cast<int64_t>(t0 + r) * D + o_col;
    u32x4 v = *reinterpret_cast<const u32x4*>(smem + r * PITCH + (tid & 15) * 8);
    // the gradient that came back along the tokens' other uses: added here instead of by a pass of
    // its own over three (T, D) tensors (17 us at 8192 x 2048), with that pass's rounding
    if constexpr (ROWS) {
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = add_bf16x2(v[j], front[i][j]);
    } else if (g.addend) {
      const u32x4 a = *reinterpret_cast<const u32x4*>(g.addend + at);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = add_bf16x2(v[j], a[j]);
    }
    *reinterpret_cast<u32x4*>(dx + at) = v;
  }
}

// ---- dW(E,D) = dlogits(T,E)^T . x(T,D), fp32 partials per K split -----------------------
// Tile 128 experts x 128 columns, 8 waves as 4 x 2, each 32 x 64.  Per K step of 64
// tokens: dlogits tile split into three pieces (KS), x tile (KS).
constexpr int W_BM = 128, W_BN = 128, W_NT = 512;

__device__ __forceinline__ void gate_dw_tile(const float* __restrict__ dlogits, const uint16_t* __restrict__ x,
                                             float* __restrict__ partial, int T, int D, int E, int rows_per_split, int part,
                                             uint16_t* smem) {
  uint16_t* A_p = smem;                 // 3 x [64][128] KS
  uint16_t* B_s = smem + 3 * BK * W_BM;  // [64][128] KS
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 64;
  const int col_tiles = (D + W_BN - 1) / W_BN, row_tiles = (E + W_BM - 1) / W_BM;
  const int n0 = min(part % col_tiles * W_BN, D - W_BN);
  const int m0 = part / col_tiles % row_tiles * W_BM;  // E % 64 == 0; a last tile of 64 experts clamps its rows
  const int split = part / (col_tiles * row_tiles);
  const int t_begin = split * rows_per_split, t_end = min(T, t_begin + rows_per_split);
  f32x16 acc[2];
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[n][i] = 0.0f;
  const u32x4 zero = {0, 0, 0, 0};
  // 64 tokens x 16 chunks of 8 experts (A) / 8 columns (B) = 1024 units each, 2 per thread; one LDS
  // stage, the next K step's operands requested into registers before the MFMAs of the current one
  f32x4 ra[2][2];
  u32x4 rb[2];
  auto fetch = [&](int tk) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + W_NT * i;
      const int k = u >> 4, c = u & 15;
      const int tc = min(tk + k, T - 1);
      const float* src = dlogits + static_cast<int64_t>(tc) * E + min(m0 + c * 8, E - 8);
      ra[i][0] = *reinterpret_cast<const f32x4*>(src);
      ra[i][1] = *reinterpret_cast<const f32x4*>(src + 4);
      rb[i] = *reinterpret_cast<const u32x4*>(x + static_cast<int64_t>(tc) * D + n0 + c * 8);
    }
  };
  if (t_begin < t_end) fetch(t_begin);
  for (int tk = t_begin; tk < t_end; tk += BK) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int u = tid + W_NT * i;
      const int k = u >> 4, c = u & 15;
      const bool live = tk + k < t_end;
      u32x4 hi, mid, lo;
      split8(ra[i][0], ra[i][1], hi, mid, lo);
      const int o = ks_off<W_BM>(k, c);
      *reinterpret_cast<u32x4*>(A_p + o) = live ? hi : zero;
      *reinterpret_cast<u32x4*>(A_p + BK * W_BM + o) = live ? mid : zero;
      *reinterpret_cast<u32x4*>(A_p + 2 * BK * W_BM + o) = live ? lo : zero;
      *reinterpret_cast<u32x4*>(B_s + ks_off<W_BN>(k, c)) = rb[i];
    }
    __syncthreads();
    if (tk + BK < t_end) fetch(tk + BK);
#pragma unroll
    for (int kk = 0; kk < BK / 16; ++kk) {
      bf16x8 bf[2];
#pragma unroll
      for (int n = 0; n < 2; ++n) bf[n] = frag_ks<W_BN>(B_s, wn + n * 32, kk, lane);
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const bf16x8 af = frag_ks<W_BM>(A_p + s * BK * W_BM, wm, kk, lane);
#pragma unroll
        for (int n = 0; n < 2; ++n) acc[n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[n], af, acc[n], 0, 0, 0);
      }
    }
    __syncthreads();
  }
  // lane = expert row (lane & 31); registers = 4 consecutive columns
  const int e = m0 + wm + (lane & 31);
  if (e < E) {
    float* dst = partial + (static_cast<int64_t>(split) * E + e) * D + n0 + wn;
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = {acc[n][q * 4], acc[n][q * 4 + 1], acc[n][q * 4 + 2], acc[n][q * 4 + 3]};
        *reinterpret_cast<f32x4*>(dst + n * 32 + q * 8 + (lane >> 5) * 4) = v;
      }
  }
}

// Both in one launch, the dW tiles first.  In a training step they run beside the experts' weight gradients, whose workgroups hold a
// CU each until the product ends: every launch of this chain waits for one of them to finish, so there are few.  With the row sum
// in front (ROWS) the launch reads 2 T D elements less; alone, us, row sum + dx + dW / this: 3000 tokens of 6 x 1024, 64 experts 30 / 19,
// 8192 of 8 x 2048, 128 experts 102 / 86, 16384 194 / 169.  Inside a training step only the short ones gain: 64 experts of 1024 x 512, six a
// token, 300 tokens 233 / 223, 700 263 / 256, 3000 417 / 414, four of 64, 2000 tokens 273 / 264; 128 of 2048 x 768, 2500 tokens 1160 / 1153, 4000
// 1520 / 1529, 16384 skewed 4655 / 4708.
struct GateBwd {
  const float* dlogits;
  const uint16_t *x, *ws;  // ws: the weight's hi and mid pieces
  GateSum sum;
  uint16_t* dx;
  float* partial;
  int T, D, E, rows_per_split, dw_tiles;
};
template <bool ROWS>
__global__ __launch_bounds__(X_NT, 4) void gate_bwd_kernel(GateBwd p) {
  static_assert(X_NT == W_NT, "both tiles on the same workgroup");
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const int block = blockIdx.x;
  if (block < p.dw_tiles) gate_dw_tile(p.dlogits, p.x, p.partial, p.T, p.D, p.E, p.rows_per_split, block, smem);
  else gate_dx_tile<ROWS>(p.dlogits, p.ws, p.sum, p.dx, p.T, p.D, p.E, block - p.dw_tiles, smem);
}

// ---- both gradients for few experts (router_few.h) ---------------------------------------
// What dx parts read besides dlogits and W.  rows: null, or the experts' input gradients, whose sum over the token's K
// slots in ascending order, rounded, comes in front of the addend as permute_rows_bwd's does.
template <typename TX>
struct GateDx {
  const TX *addend, *rows;
  const int32_t* row_of_slot;
  int K, row_capacity;
};

// TW tokens a wave.  With the rows in front (ROWS) two: the launch is the last of a backward, bound by the latency of its row
// reads, and wants many waves (1531 tokens of 4 x 320, 16 experts: 18.0 us with eight a wave, 6.6 with two; 512 fp32 of 2 x 256 7.6, 4.0).
template <typename TX, bool ROWS, int TW, int PITCH = S_MAX_E>  // PITCH: experts at most
__device__ __forceinline__ void gate_dx_part(const float* __restrict__ dlogits, const float* __restrict__ w,
                                             const GateDx<TX>& g, TX* __restrict__ dx, int T, int D, int E, int part,
                                             float* lds) {
  constexpr int TOK = 4 * TW;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col_blocks = (D + S_COLS - 1) / S_COLS;
  const int cb = part % col_blocks, t0 = part / col_blocks * TOK;
  const int tokens = min(TOK, T - t0), n = cb * S_COLS + lane * 4;
  for (int i = tid; i < TOK * PITCH; i += 256) {
    const int t = i / PITCH, e = i % PITCH;
    lds[i] = t < tokens && e < E ? dlogits[static_cast<int64_t>(t0 + t) * E + e] : 0.0f;
  }
  __syncthreads();
  if (n >= D) return;
  f32x4 sum[ROWS ? TW : 1];
  if constexpr (ROWS) {
    // the rows go out first: the product below runs while they arrive
    constexpr int B = 8 / TW;  // slots requested together
#pragma unroll
    for (int t = 0; t < TW; ++t) sum[t] = f32x4{0, 0, 0, 0};
    const int32_t* slots = g.row_of_slot + (static_cast<int64_t>(t0) + wave * TW) * g.K;
    for (int k0 = 0; k0 < g.K; k0 += B) {
      f32x4 v[B][TW];
#pragma unroll
      for (int k = 0; k < B; ++k)
#pragma unroll
        for (int t = 0; t < TW; ++t) {
          const int row = k0 + k < g.K && wave * TW + t < tokens ? slots[t * g.K + k0 + k] : -1;  // wave-uniform
          v[k][t] = row >= 0 && row < g.row_capacity ? load_cols(g.rows + static_cast<int64_t>(row) * D + n) : f32x4{0, 0, 0, 0};
        }
#pragma unroll
      for (int k = 0; k < B; ++k)
#pragma unroll
        for (int t = 0; t < TW; ++t) sum[t] += v[k][t];
    }
  }
  f32x4 acc[TW];
#pragma unroll
  for (int t = 0; t < TW; ++t) acc[t] = f32x4{0, 0, 0, 0};
  constexpr int EB = TW >= 8 ? 4 : 8;  // experts requested together
  for (int e = 0; e < E; e += EB) {
    f32x4 wv[EB];
#pragma unroll
    for (int j = 0; j < EB; ++j) wv[j] = load_cols(w + static_cast<int64_t>(min(e + j, E - 1)) * D + n);
#pragma unroll
    for (int t = 0; t < TW; ++t)
#pragma unroll
      for (int q = 0; q < EB / 4; ++q) {
        const f32x4 d = *reinterpret_cast<const f32x4*>(lds + (wave * TW + t) * PITCH + e + 4 * q);  // zero past E
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][i] = fmaf(d[j], wv[4 * q + j][i], acc[t][i]);
      }
  }
  auto rounded = [](float v) { return sizeof(TX) == 2 ? round_bf16(v) : v; };
#pragma unroll
  for (int t = 0; t < TW; ++t) {
    if (wave * TW + t >= tokens) break;
    const int64_t at = static_cast<int64_t>(t0 + wave * TW + t) * D + n;
    f32x4 v = acc[t];
    // each sum is added to the rounded one before it and rounded again, as separate additions would be
    if (ROWS || g.addend) {
      f32x4 a = g.addend ? load_cols(g.addend + at) : f32x4{0, 0, 0, 0};
      if constexpr (ROWS) {
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i] = g.addend ? rounded(rounded(sum[t][i]) + a[i]) : rounded(sum[t][i]);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = rounded(v[i]) + a[i];
    }
    store_cols(dx + at, v);
  }
}

constexpr int kRowsTok = 8;  // tokens of a dx part with the rows in front

template <typename TX, bool ROWS, int MAX_E = S_MAX_E>
__global__ __launch_bounds__(256) void gate_bwd_few_kernel(GateDw dw, const float* __restrict__ dlogits,
                                                           const float* __restrict__ w, GateDx<TX> g, TX* __restrict__ dx,
                                                           int T, int D, int E, int dw_parts) {
  __shared__ __attribute__((aligned(16))) float lds[kGateDwLds];
  static_assert(S_TOK * MAX_E <= kGateDwLds, "a dx part's gradients");
  const int block = blockIdx.x;
  if (block < dw_parts) gate_dw_part<TX>(dw, block, lds);
  else gate_dx_part<TX, ROWS, (ROWS ? kRowsTok : S_TOK) / 4, MAX_E>(dlogits, w, g, dx, T, D, E, block - dw_parts, lds);
}

// dx with the sum over the token's rows, and beside it the sum of dW's slices, in their order: the two ends of a backward
// whose dW parts ran in an earlier launch.
template <typename TX>
__global__ __launch_bounds__(256) void gate_rows_bwd_kernel(const float* __restrict__ dlogits, const float* __restrict__ w,
                                                            GateDx<TX> g, TX* __restrict__ dx,
                                                            const float* __restrict__ partial, float* __restrict__ dw,
                                                            int splits, int T, int D, int E, int dx_parts) {
  __shared__ __attribute__((aligned(16))) float lds[kRowsTok * S_MAX_E];
  const int block = blockIdx.x;
  if (block < dx_parts) {
    gate_dx_part<TX, true, kRowsTok / 4>(dlogits, w, g, dx, T, D, E, block, lds);
    return;
  }
  const int64_t n = static_cast<int64_t>(E) * D, i = static_cast<int64_t>(block - dx_parts) * 256 + threadIdx.x;
  if (i >= n) return;
  float sum = 0.0f;
  constexpr int B = 8;  // in flight
  for (int z0 = 0; z0 < splits; z0 += B) {
    float v[B];
#pragma unroll
    for (int b = 0; b < B; ++b) v[b] = z0 + b < splits ? partial[(z0 + b) * n + i] : 0.0f;
#pragma unroll
    for (int b = 0; b < B; ++b) sum += v[b];
  }
  dw[i] = sum;
}

template <typename K>
int set_dyn_lds(K kernel, int bytes) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  return e == hipSuccess ? MI355_OK : fail(MI355_ELAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
}

constexpr int G_LDS = 2 * G_STAGE * 2;                         // 131072

// Splits of the contraction for the 128-token forward kernel: enough workgroups for the chip,
// at least four K steps each, whole K steps.
int fwd_splits(int64_t T, int64_t D, int64_t E) {
  const int64_t tiles = ((T + G_BM - 1) / G_BM) * ((E + G_BN - 1) / G_BN);
  int64_t s = 1;
  while (s < 8 && tiles * s < 256 && D % (2 * s * BK) == 0 && D / (2 * s) >= 4 * BK) s *= 2;
  return static_cast<int>(s);
}
constexpr int X_LDS = X_ELEMS * 2;                              // 65536
constexpr int W_LDS = (3 * BK * W_BM + BK * W_BN) * 2;         // 65536

// Splits of the token contraction for dW.  Two workgroups fit a CU, so the launch runs in
// rounds of 512 and its length goes as rounds x tokens per split: one more split than fills a
// round costs a whole extra round.  Each split also adds an (E, D) fp32 partial for the
// reduction to read, priced here at twelve token rows of the kernel (measured: the sum is
// within a few percent of the best split count at 8192 x 2048 x 128, 16384 x 2048 x 128 and
// 4096 x 7168 x 256).  At least four K steps per split.
int dw_splits(int64_t T, int64_t D, int64_t E) {
  const int64_t tiles = ((D + W_BN - 1) / W_BN) * ((E + W_BM - 1) / W_BM);
  const int64_t max_s = std::max<int64_t>(1, std::min<int64_t>(64, (T + 4 * BK - 1) / (4 * BK)));
  int64_t best = 1, best_cost = INT64_MAX;
  for (int64_t s = 1; s <= max_s; ++s) {
    const int64_t rows = ((T + s - 1) / s + BK - 1) / BK * BK;
    const int64_t cost = ((tiles * s + 511) / 512) * rows + 12 * s;
    if (cost < best_cost) { best = s; best_cost = cost; }
  }
  return static_cast<int>(best);
}

}  // namespace

bool router_few_ok(int x_dtype, int w_dtype, int64_t D, int64_t E) {
  return w_dtype == MI355_F32 && (x_dtype == MI355_BF16 || x_dtype == MI355_F32) && D % 4 == 0 && D >= 4 && E <= S_MAX_E;
}
// ... without the rows in front, up to twice as many experts (60, which no matrix tile divides), while the tokens are few: strided products took three launches,
// and beside the experts' weight gradients each waits for a CU.  Alone, us, those / these: 300 x 512, 60 experts 17.3 / 13.7, 1000 x 1024 21.9 / 15.6,
// 2229 x 768 33.8 / 22.3, 3000 x 512, 36 experts 22.9 / 16.0, fp32 tokens, 64 experts 25.3 / 19.5; but 12000 x 1024 66 / 66, 8000 x 2048 79 / 86 (W is read once for
// 32 tokens, x once for eight experts).  A training step: 2229 tokens of 60 experts of 768 x 384, eight each, 288 / 271, 3000 of 1024 x 512 377 / 369,
// 5000 of 1280 x 640 (past the line) 596 / 597.  dx is the same sum in the same order, dW's error against fp64 is 0.3-0.95 times theirs.
bool router_few_bwd_ok(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  return router_few_ok(x_dtype, w_dtype, D, E) ||
         (router_few_ok(x_dtype, w_dtype, D, S_MAX_E) && E <= 2 * S_MAX_E && E % 4 == 0 && T * D <= (int64_t{6} << 20));
}
int64_t router_few_bwd_workspace(int64_t T, int64_t D, int64_t E) { return gate_dw_splits(T, D, E) * E * D * 4; }

int router_few_bwd(const float* dlogits, const void* x, int x_dtype, const float* w, const RowSum& sum, void* dx, float* dw,
                   void* workspace, int64_t T, int64_t D, int64_t E, hipStream_t s) {
  const int splits = gate_dw_splits(T, D, E);
  const GateDw job = gate_dw_job(dlogits, x, splits > 1 ? static_cast<float*>(workspace) : dw, T, D, E);
  const int64_t dw_parts = dw ? gate_dw_parts(job) : 0;
  const int tok = sum.rows ? kRowsTok : S_TOK;
  const int64_t blocks = dw_parts + (dx ? (T + tok - 1) / tok * ((D + S_COLS - 1) / S_COLS) : 0);
  MI355_REQUIRE(blocks < (1ll << 31), "router_gate_bwd: too many tokens");
  auto launch = [&](auto* xp) {
    using TX = std::remove_const_t<std::remove_pointer_t<decltype(xp)>>;
    const GateDx<TX> g{static_cast<const TX*>(sum.addend), static_cast<const TX*>(sum.rows), sum.row_of_slot, (int)sum.K,
                       (int)sum.row_capacity};
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), 0, s, job, dlogits, w, g, static_cast<TX*>(dx), (int)T, (int)D,
                         (int)E, (int)dw_parts);
    };
    if (E > S_MAX_E) run(gate_bwd_few_kernel<TX, false, 2 * S_MAX_E>);
    else if constexpr (sizeof(TX) == 2) run(sum.rows ? gate_bwd_few_kernel<TX, true> : gate_bwd_few_kernel<TX, false>);
    else run(gate_bwd_few_kernel<TX, false>);  // (fp32 tokens: the experts' launches take the parts along)
  };
  if (x_dtype == MI355_BF16) launch(static_cast<const uint16_t*>(x));
  else launch(static_cast<const float*>(x));
  if (int rc = check_launch("router_gate_bwd")) return rc;
  return dw && splits > 1 ? launch_splitk_reduce(job.partial, dw, MI355_F32, E * D, splits, s) : MI355_OK;
}

int router_rows_bwd(const float* dlogits, int x_dtype, const float* w, const void* rows, const int32_t* row_of_slot,
                    int64_t row_capacity, int64_t K, const void* addend, void* dx, const float* partial, float* dw, int64_t T,
                    int64_t D, int64_t E, hipStream_t s) {
  const int splits = gate_dw_splits(T, D, E);
  const int64_t dx_parts = dx ? (T + kRowsTok - 1) / kRowsTok * ((D + S_COLS - 1) / S_COLS) : 0;
  const int64_t blocks = dx_parts + (dw ? (E * D + 255) / 256 : 0);
  MI355_REQUIRE(blocks < (1ll << 31), "router_gate_rows_bwd: too many tokens");
  if (blocks == 0) return MI355_OK;
  auto launch = [&](auto* xp) {
    using TX = std::remove_pointer_t<decltype(xp)>;
    const GateDx<TX> g{static_cast<const TX*>(addend), static_cast<const TX*>(rows), row_of_slot, (int)K, (int)row_capacity};
    hipLaunchKernelGGL(gate_rows_bwd_kernel<TX>, dim3((unsigned)blocks), dim3(256), 0, s, dlogits, w, g, xp, partial, dw,
                       splits, (int)T, (int)D, (int)E, (int)dx_parts);
  };
  if (x_dtype == MI355_BF16) launch(static_cast<uint16_t*>(dx));
  else launch(static_cast<float*>(dx));
  return check_launch("router_gate_rows_bwd");
}

bool router_x3_ok(int x_dtype, int w_dtype, int64_t D, int64_t E) {
  return x_dtype == MI355_BF16 && w_dtype == MI355_F32 && D % 64 == 0 && E % 64 == 0 && D >= 128;
}

int64_t router_x3_bwd_workspace(int64_t T, int64_t D, int64_t E) {
  return 2 * E * D * 2 + static_cast<int64_t>(dw_splits(T, D, E)) * E * D * 4;
}

// Which forward kernel serves a gate: the 128-token one (widths on its grid and tokens enough), the
// 32-token one (fp32 weights, rows of whole 16-byte pieces), or neither (fp64, odd widths).
// The wide one waits for the launch that splits the weights.  Below 192 Mi products that launch is more than the other's repeated reads of the weights cost, also
// with the split in the backward instead.  us, wide / 32 tokens: forward of 3000 tokens, 64 experts of 512 x 512 64.1 / 60.0, 2000 of 1024 x 512 84.0 / 82.0, 3000 110.3 / 108.9, 6000
// 168.8 / 172.5, 2000 of 128 of it 134.9 / 132.8, 1500 of 128 of 2048 x 768 274.5 / 276.6; a training step with router statistics of 1024, 1500, 2000, 3000, 4000 and 6000 tokens, 64 of
// 1024 x 512, 225.8 / 223.4, 290.6 / 282.5, 304.4 / 298.9, 351.4 / 348.5, 454.9 / 456.8, 547.5 / 549.2.
// Error against fp64 (relative 2-norm, 1024-20000 tokens of 128-2048 x 64-128): 1.2e-7 to 1.8e-7 / 0.8e-7 to 1.4e-7.
static bool gate_wide(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  return T >= 1024 && T * E * D > (int64_t{192} << 20) && router_x3_ok(x_dtype, w_dtype, D, E);
}
int router_fwd_splits(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  if (T < 1 || D < 1 || E < 1) return 0;
  if (gate_wide(x_dtype, w_dtype, T, D, E)) return fwd_splits(T, D, E);
  if (w_dtype != MI355_F32 || E > 65535 * R_BN) return 0;
  if ((x_dtype == MI355_BF16 && D % 8 == 0) || (x_dtype == MI355_F32 && D % 4 == 0)) return rows_splits(T, D, E);
  return 0;
}

int64_t router_fwd_pieces_bytes(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  return gate_wide(x_dtype, w_dtype, T, D, E) ? 3 * E * D * 2 : 0;
}

// ... and what a forward leaves for the backward: the 32-token kernel's first workgroups have the first two pieces in registers, and a launch of its own for
// them in the backward is saved.  A training step with router statistics, us, apart / kept: 64 experts of 1024 x 512, 256 tokens 176.2 / 173.8, 400 187.9 / 185.8, 700 211.0 /
// 209.1, 1000 227.9 / 222.6, 1500 287.5 / 285.1, 3000 351.9 / 353.5; 300 of 128 of 512 x 384 155.1 / 153.5.  Larger weights and more tokens have their backward beside the experts' weight
// gradients, where the launch is hidden: 200, 500 and 1000 tokens of 128 of 2048 x 768 678.3 / 679.7, 721.3 / 723.6, 766.2 / 768.3.
int64_t router_fwd_kept_bytes(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E) {
  if (const int64_t wide = router_fwd_pieces_bytes(x_dtype, w_dtype, T, D, E)) return wide;
  return router_x3_ok(x_dtype, w_dtype, D, E) && E * D <= (1 << 17) && T * E * D <= (1 << 27) && router_fwd_splits(x_dtype, w_dtype, T, D, E) > 0 ? 2 * E * D * 2 : 0;
}

int router_fwd_partial(const void* x, int x_dtype, const float* w, const float* bias, float* partial, void* pieces, void* keep,
                       int64_t T, int64_t D, int64_t E, hipStream_t s) {
  const int splits = router_fwd_splits(x_dtype, MI355_F32, T, D, E);
  const float* in_kernel_bias = splits == 1 ? bias : nullptr;
  if (gate_wide(x_dtype, MI355_F32, T, D, E)) {
    static PerDeviceOnce wide_configured;
    if (wide_configured.needed()) {
      if (int rc = set_dyn_lds(gate_fwd_wide_kernel, G_LDS)) return rc;
      wide_configured.done();
    }
    uint16_t* ws = static_cast<uint16_t*>(pieces);
    const int64_t n = E * D;
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, s, w, ws, n, 3);
    const dim3 grid((unsigned)((T + G_BM - 1) / G_BM), (unsigned)((E + G_BN - 1) / G_BN), (unsigned)splits);
    hipLaunchKernelGGL(gate_fwd_wide_kernel, grid, dim3(G_NT), G_LDS, s, static_cast<const uint16_t*>(x), ws,
                       in_kernel_bias, partial, (int)T, (int)D, (int)E, (int)(D / splits));
    return check_launch("router_gate_fwd");
  }
  const int k_per_wave = gate_rows_k(D, splits);
  const int64_t t_tiles = (T + R_BM - 1) / R_BM;
  auto launch = [&](auto* xp, auto bn) {
    constexpr int BN = decltype(bn)::value;
    using TX = std::remove_const_t<std::remove_pointer_t<decltype(xp)>>;
    const dim3 grid((unsigned)t_tiles, (unsigned)((E + BN - 1) / BN), (unsigned)splits);
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(64 * R_WAVES), 0, s, xp, w, in_kernel_bias, partial, (int)T, (int)D, (int)E, k_per_wave,
                         static_cast<uint16_t*>(keep));
    };
    if constexpr (sizeof(TX) == 2) run(keep ? gate_rows_kernel<TX, BN, true> : gate_rows_kernel<TX, BN, false>);
    else run(gate_rows_kernel<TX, BN, false>);
  };
  auto choose = [&](auto* xp) {
    const int bn = rows_experts(t_tiles, E, splits);
    if (bn == 8) launch(xp, std::integral_constant<int, 8>{});
    else if (bn == 16) launch(xp, std::integral_constant<int, 16>{});
    else launch(xp, std::integral_constant<int, 32>{});
  };
  if (x_dtype == MI355_BF16) choose(static_cast<const uint16_t*>(x));
  else choose(static_cast<const float*>(x));
  return check_launch("router_gate_fwd");
}

int router_logits_reduce(const float* partial, const float* bias, float* logits, int64_t T, int64_t E, int splits,
                         hipStream_t s) {
  const int64_t te = T * E;
  hipLaunchKernelGGL(logits_reduce_kernel, dim3((unsigned)((te + 1023) / 1024)), dim3(256), 0, s, partial, bias,
                     logits, te, (int)E, splits);
  return check_launch("router_gate_fwd");
}

int router_x3_bwd(const float* dlogits, const void* x, const float* w, const void* pieces, const RowSum& sum,
                  void* dx, float* dw, void* workspace, int64_t T, int64_t D, int64_t E, hipStream_t s) {
  static PerDeviceOnce configured;
  if (configured.needed()) {
    for (auto* kernel : {gate_bwd_kernel<false>, gate_bwd_kernel<true>})
      if (int rc = set_dyn_lds(kernel, std::max(X_LDS + X_BM * kMaxSumK * 4, W_LDS))) return rc;
    configured.done();
  }
  uint16_t* ws = static_cast<uint16_t*>(workspace);
  const int64_t n = E * D, cols = (D + X_BN - 1) / X_BN;
  const bool want_dx = dx && T > 0;
  // (the forward's pieces, when its caller kept them: hi and mid come first there too)
  if (want_dx && !pieces)
    hipLaunchKernelGGL(split_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, s, w, ws, n, 2);
  const int splits = dw ? dw_splits(T, D, E) : 0;
  const int64_t dw_tiles = cols * ((E + W_BM - 1) / W_BM) * splits;
  const int64_t blocks = dw_tiles + (want_dx ? (T + X_BM - 1) / X_BM * cols : 0);
  MI355_REQUIRE(blocks < (1ll << 31), "router_gate_bwd: too many tokens");
  if (blocks == 0) return MI355_OK;
  const GateBwd p{dlogits, static_cast<const uint16_t*>(x), pieces ? static_cast<const uint16_t*>(pieces) : ws,
                  GateSum{static_cast<const uint16_t*>(sum.addend), static_cast<const uint16_t*>(sum.rows), sum.row_of_slot,
                          (int)sum.K, (int)sum.row_capacity},
                  static_cast<uint16_t*>(dx), reinterpret_cast<float*>(ws + 2 * n), (int)T, (int)D, (int)E,
                  splits ? (int)(((T + splits - 1) / splits + BK - 1) / BK * BK) : 0, (int)dw_tiles};
  if (sum.rows)
    hipLaunchKernelGGL(gate_bwd_kernel<true>, dim3((unsigned)blocks), dim3(X_NT), std::max(X_LDS + X_BM * (int)sum.K * 4, W_LDS), s, p);
  else
    hipLaunchKernelGGL(gate_bwd_kernel<false>, dim3((unsigned)blocks), dim3(X_NT), std::max(X_LDS, W_LDS), s, p);
  if (int rc = check_launch("router_gate_bwd")) return rc;
  return dw ? launch_splitk_reduce(p.partial, dw, MI355_F32, n, splits, s) : MI355_OK;
}

}  // namespace mi355
