// Weighted unpermute-combine and its backward (which also yields the router's
// score gradient).  Both are bandwidth kernels: a wavefront per token (or per 1 KiB of a
// token's row), 16-byte lanes along D, the K row indices and weights held in lanes 0..K-1 and broadcast
// by shuffles.  No atomics: every output element has exactly one writer, so the
// result is deterministic.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "row_vec.h"

namespace mi355 {
namespace {

template <typename T>
__device__ __forceinline__ float round_to(float v);
template <>
__device__ __forceinline__ float round_to<float>(float v) { return v; }
template <>
__device__ __forceinline__ float round_to<uint16_t>(float v) { return round_bf16(v); }

// a = round(a) + v
template <typename T>
__device__ __forceinline__ void plus(float (&a)[Vec<T>::N], const uint4& v) {
  float f[Vec<T>::N];
  Vec<T>::unpack(v, f);
#pragma unroll
  for (int q = 0; q < Vec<T>::N; ++q) a[q] = round_to<T>(a[q]) + f[q];
}

// SMALL_K: K <= 8, the eight-row chunk below is the only one.
//   A token's row is cut into `pieces` of 1 KiB, one wave each, and the workgroups of a token's pieces follow one
// another: few tokens fill the chip, and what runs at one time reads whole rows.  (All tokens' first
// pieces, then all second ones, and so on reads the same KiB of rows that lie a power of two apart, few memory channels
// at a time.)  Eight bf16 rows a token, us, one wave a row in passes of 4 KiB / pieces in that other order / here:
//   8192 tokens of 1024 columns 37 / 29 / 29, of 2048 57 / 71 / 54 (5.6 TB/s), of 4096 112 / 134 / 107, of 7168
//   197 / 193 / 186; 3000 of 2048 21 / 23 / 21; 1000 of 4096 18 / 13 / 13; 128 of 7168 21 / 5.1 / 5.1; 1 of 2048
//   6.6 / 3.7 / 3.7.  Sixteen rows, 8192 of 2048 108 / 137 / 100.  One row in eight present (one rank's share of 8
//   ranks), 4095 of 7168 44 / 33 / 33, 8192 of 2048 22 / 20 / 19.
template <typename T, bool SMALL_K>
__global__ __launch_bounds__(256) void combine_fwd_kernel(
    const T* __restrict__ y, const float* __restrict__ weights,
    const int32_t* __restrict__ row_of_slot, const T* __restrict__ addend, T* __restrict__ out, int T_, int D, int K,
    int round_terms, int pieces, const int32_t* __restrict__ counts, float* __restrict__ totals, int E) {
  const int lane = threadIdx.x & 63;
  // A router's running counts.  As a launch behind this one, a training step, us, apart / here: 512 fp32 tokens of 8 x 256 x 512 128 / 124.5, 225 of 16 x 628 x 832 154.2 /
  // 151.4; bf16 1000 of 16 x 1024 x 512 151.7 / 148.7, 283, 1000 and 3000 of 64 of it 184 / 181, 229 / 225.7, 345 / 342, 300 and 1000 of 128 x 2048 x 768 698 / 692, 766 / 761.
  if (totals && blockIdx.x == 0)
    for (int e = threadIdx.x; e < E; e += 256) totals[e] += static_cast<float>(counts[e]);
  const int tokens = blockIdx.x / pieces, piece = blockIdx.x % pieces;
  const int t = tokens * 4 + (threadIdx.x >> 6);
  if (t >= T_) return;
  const int64_t s0 = static_cast<int64_t>(t) * K;
  const int row = lane < K ? row_of_slot[s0 + lane] : -1;
  const float w = lane < K ? weights[s0 + lane] : 0.0f;
  // addend (the shared expert's output): added to the rounded sum and rounded again, as the separate
  // addition of two tensors of this type would be
  const T* add = addend ? addend + static_cast<int64_t>(t) * D : nullptr;
  // ascending-row visiting order (index_add's order): position of each valid slot
  int pos = 0;
  for (int j = 0; j < K; ++j) {
    const int rj = __builtin_amdgcn_readlane(row, j);  // j is wave-uniform: a lane read, not an LDS permute
    pos += (rj >= 0 && (rj < row || (rj == row && j < lane))) ? 1 : 0;
  }
  const int nvalid = __popcll(__ballot(row >= 0));
  // lane p receives the p-th visited slot: every valid lane sends its (row, weight) to lane
  // `pos` (one cross-lane permute each); the others send to lane 63, which is past the last
  // valid position whenever such a lane exists and is not read then
  const int to = (row >= 0 ? pos : 63) << 2;
  int o_row = __builtin_amdgcn_ds_permute(to, row);
  float o_w = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(w)));
  if (lane >= nvalid) { o_row = -1; o_w = 0.0f; }

  constexpr int V = Vec<T>::N;
  T* dst = out + static_cast<int64_t>(t) * D;
  // Loops are uniform across the wave (shuffles need every lane).
  if (D % V == 0) {
    const int nv = D / V;
    // one vector per lane from eight rows at a time, all requested before the first is used.  Rows and weights
    // are wave-uniform; the terms are added in visiting order.
    constexpr int B = 8;
    auto request = [&](int i, int p0, uint4 (&v)[B], float (&ww)[B]) {
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int p = max(min(p0 + j, nvalid - 1), 0);  // past the end: not loaded, not used
        const int r = __builtin_amdgcn_readlane(o_row, p);  // p is wave-uniform
        ww[j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(o_w), p));
        const uint4* src = reinterpret_cast<const uint4*>(y + static_cast<int64_t>(max(r, 0)) * D);
        v[j] = (p0 + j < nvalid && i < nv) ? load_stream(src + i) : make_uint4(0, 0, 0, 0);
      }
    };
    auto add_terms = [&](float (&a)[V], const uint4& v, float w) {
      float f[V];
      Vec<T>::unpack(v, f);
#pragma unroll
      for (int q = 0; q < V; ++q) {
        const float term = f[q] * w;
        a[q] += round_terms ? round_to<T>(term) : term;
      }
    };
    for (int base = piece * kWave; base < nv; base += pieces * kWave) {
      const int i = base + lane;
      float a[V];
#pragma unroll
      for (int q = 0; q < V; ++q) a[q] = 0.0f;
      for (int p0 = 0; p0 < (SMALL_K ? 1 : nvalid); p0 += B) {
        uint4 v[B];
        float ww[B];
        request(i, p0, v, ww);
#pragma unroll
        for (int j = 0; j < B; ++j)
          if (p0 + j < nvalid) add_terms(a, v[j], ww[j]);
      }
      if (i < nv) {
        if (add) plus<T>(a, reinterpret_cast<const uint4*>(add)[i]);
        reinterpret_cast<uint4*>(dst)[i] = Vec<T>::pack(a);
      }
    }
  } else {
    for (int base = piece * kWave; base < D; base += pieces * kWave) {
      const int i = base + lane;
      const bool on = i < D;
      float a = 0.0f;
      for (int p = 0; p < nvalid; ++p) {
        const int r = __shfl(o_row, p, kWave);
        const float ww = __shfl(o_w, p, kWave);
        if (!on) continue;
        const float term = load_as_f32(y + static_cast<int64_t>(r) * D + i) * ww;
        a += round_terms ? round_to<T>(term) : term;
      }
      if (on) store_from_f32(dst + i, add ? round_to<T>(a) + load_as_f32(add + i) : a);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void combine_bwd_kernel(
    const T* __restrict__ dout, const T* __restrict__ y, const float* __restrict__ weights,
    const int32_t* __restrict__ row_of_slot, const int32_t* __restrict__ slot_of_row,
    const int32_t* __restrict__ total_rows, T* __restrict__ dy, float* __restrict__ dweights,
    int T_, int D, int K, int token_blocks, int row_capacity, int stream_stores) {
  const int lane = threadIdx.x & 63;
  constexpr int V = Vec<T>::N;
  if (static_cast<int>(blockIdx.x) >= token_blocks) {
    // padding rows of dy get zeros
    const int r = (blockIdx.x - token_blocks) * 4 + (threadIdx.x >> 6);
    if (r >= row_capacity || r >= *total_rows || slot_of_row[r] >= 0) return;
    T* dst = dy + static_cast<int64_t>(r) * D;
    for (int i = lane; i < D; i += kWave) dst[i] = T(0);
    return;
  }
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T_) return;
  const int64_t s0 = static_cast<int64_t>(t) * K;
  const int row = lane < K ? row_of_slot[s0 + lane] : -1;
  const float w = lane < K ? weights[s0 + lane] : 0.0f;
  const T* g = dout + static_cast<int64_t>(t) * D;
  float my_dot = 0.0f;  // lane k keeps slot k's dot product
  if (D % V == 0) {
    // The token's gradient row is read ONCE per pass of G vectors per lane (4 KiB of the row per
    // wave: all of it at D = 2048 bf16) and kept in registers while the K expert rows stream by;
    // re-reading it per slot fetched it K times from wherever it had gone meanwhile.
    const int nv = D / V;
    constexpr int G = 4;
    for (int base = 0; base < nv; base += G * kWave) {
      float gf[G][V];
#pragma unroll
      for (int q = 0; q < G; ++q) {
        const int i = base + q * kWave + lane;
        Vec<T>::unpack(i < nv ? reinterpret_cast<const uint4*>(g)[i] : make_uint4(0, 0, 0, 0), gf[q]);
      }
      for (int k = 0; k < K; ++k) {
        const int r = __shfl(row, k, kWave);
        const float ww = __shfl(w, k, kWave);
        if (r < 0) continue;
        const uint4* yr = reinterpret_cast<const uint4*>(y + static_cast<int64_t>(r) * D);
        uint4* dr = reinterpret_cast<uint4*>(dy + static_cast<int64_t>(r) * D);
        uint4 yv[G];
#pragma unroll
        for (int q = 0; q < G; ++q) {
          const int i = base + q * kWave + lane;
          yv[q] = i < nv ? load_stream(yr + i) : make_uint4(0, 0, 0, 0);
        }
        float dot = 0.0f;
#pragma unroll
        for (int q = 0; q < G; ++q) {
          const int i = base + q * kWave + lane;
          float yf[V], o[V];
          Vec<T>::unpack(yv[q], yf);
#pragma unroll
          for (int c = 0; c < V; ++c) {
            dot += yf[c] * gf[q][c];
            o[c] = gf[q][c] * ww;
          }
          if (i < nv) {
            if (stream_stores) store_stream(dr + i, Vec<T>::pack(o));
            else dr[i] = Vec<T>::pack(o);
          }
        }
        dot = wave_sum(dot);
        if (lane == k) my_dot += dot;
      }
    }
  } else {
    for (int k = 0; k < K; ++k) {
      const int r = __shfl(row, k, kWave);
      const float ww = __shfl(w, k, kWave);
      if (r < 0) continue;
      const T* yr = y + static_cast<int64_t>(r) * D;
      T* dr = dy + static_cast<int64_t>(r) * D;
      float dot = 0.0f;
      for (int i = lane; i < D; i += kWave) {
        const float gv = load_as_f32(g + i);
        dot += load_as_f32(yr + i) * gv;
        store_from_f32(dr + i, gv * ww);
      }
      dot = wave_sum(dot);
      if (lane == k) my_dot = dot;
    }
  }
  if (lane < K && dweights) dweights[s0 + lane] = my_dot;
}

// ---- fp64 rows: every product and sum in fp64 (the scores stay fp32 and are widened), one wave
// per token, lanes along D; the terms are added in ascending row order like the kernels above
__global__ __launch_bounds__(256) void combine_fwd_f64_kernel(
    const double* __restrict__ y, const float* __restrict__ weights, const int32_t* __restrict__ row_of_slot,
    double* __restrict__ out, int T_, int D, int K) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T_) return;
  const int64_t s0 = static_cast<int64_t>(t) * K;
  const int row = lane < K ? row_of_slot[s0 + lane] : -1;
  const float w = lane < K ? weights[s0 + lane] : 0.0f;
  int pos = 0;
  for (int j = 0; j < K; ++j) {
    const int rj = __shfl(row, j, kWave);
    pos += (rj >= 0 && (rj < row || (rj == row && j < lane))) ? 1 : 0;
  }
  const int nvalid = __popcll(__ballot(row >= 0));
  const int to = (row >= 0 ? pos : 63) << 2;
  int o_row = __builtin_amdgcn_ds_permute(to, row);
  float o_w = __int_as_float(__builtin_amdgcn_ds_permute(to, __float_as_int(w)));
  if (lane >= nvalid) { o_row = -1; o_w = 0.0f; }
  double* dst = out + static_cast<int64_t>(t) * D;
  for (int base = 0; base < D; base += kWave) {  // uniform trip count: the shuffles need every lane
    const int i = base + lane;
    double a = 0.0;
    for (int p = 0; p < nvalid; ++p) {
      const int r = __shfl(o_row, p, kWave);
      const double ww = static_cast<double>(__shfl(o_w, p, kWave));
      if (i < D) a += y[static_cast<int64_t>(r) * D + i] * ww;
    }
    if (i < D) dst[i] = a;
  }
}

__global__ __launch_bounds__(256) void combine_bwd_f64_kernel(
    const double* __restrict__ dout, const double* __restrict__ y, const float* __restrict__ weights,
    const int32_t* __restrict__ row_of_slot, const int32_t* __restrict__ slot_of_row,
    const int32_t* __restrict__ total_rows, double* __restrict__ dy, float* __restrict__ dweights, int T_, int D,
    int K, int token_blocks, int row_capacity) {
  const int lane = threadIdx.x & 63;
  if (static_cast<int>(blockIdx.x) >= token_blocks) {
    const int r = (blockIdx.x - token_blocks) * 4 + (threadIdx.x >> 6);
    if (r >= row_capacity || r >= *total_rows || slot_of_row[r] >= 0) return;
    double* dst = dy + static_cast<int64_t>(r) * D;
    for (int i = lane; i < D; i += kWave) dst[i] = 0.0;
    return;
  }
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T_) return;
  const int64_t s0 = static_cast<int64_t>(t) * K;
  const double* g = dout + static_cast<int64_t>(t) * D;
  for (int k = 0; k < K; ++k) {
    const int r = row_of_slot[s0 + k];  // wave-uniform
    if (r < 0) {
      if (lane == 0 && dweights) dweights[s0 + k] = 0.0f;
      continue;
    }
    const double ww = static_cast<double>(weights[s0 + k]);
    const double* yr = y + static_cast<int64_t>(r) * D;
    double* dr = dy + static_cast<int64_t>(r) * D;
    double dot = 0.0;
    for (int i = lane; i < D; i += kWave) {
      const double gv = g[i];
      dot += yr[i] * gv;
      dr[i] = gv * ww;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) dot += __shfl_xor(dot, o, kWave);
    if (lane == 0 && dweights) dweights[s0 + k] = static_cast<float>(dot);
  }
}

}  // namespace
}  // namespace mi355

using namespace mi355;

extern "C" int mi355_combine_count_fwd(const void* y, int dtype, const float* weights, const int32_t* row_of_slot,
                                       const void* addend, void* out, int64_t T, int64_t D, int64_t K, int round_terms,
                                       const int32_t* counts, float* totals, int64_t E, void* stream) {
  MI355_REQUIRE(T >= 0 && D >= 1 && K >= 1 && K <= 64 && T < (1ll << 31) && D < (1ll << 31),
                "combine_fwd: bad shape (K must be <= 64)");
  if (T == 0 && !totals) return MI355_OK;
  MI355_REQUIRE(T == 0 || (weights && row_of_slot && out), "combine_fwd: null pointer");
  MI355_REQUIRE((!addend && !totals) || dtype != MI355_F64, "combine_fwd: no fp64 form with an addend or counts");
  MI355_REQUIRE(!totals || (counts && E >= 1 && E < (1ll << 31)), "combine_fwd: totals without counts");
  const int64_t tokens = std::max<int64_t>(1, (T + 3) / 4);  // groups of one workgroup's four (without any: for the counts)
  const int64_t kib = (D * (dtype == MI355_F32 ? 4 : 2) + 1023) / 1024;  // 64 lanes of 16 bytes
  const int64_t pieces = std::max<int64_t>(1, std::min<int64_t>(kib, 0xffffff / tokens));  // a launch: below 2^32 lanes
  auto launch = [&](auto kernel, auto* yp, auto* op) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tokens * pieces)), dim3(256), 0, as_stream(stream), yp, weights, row_of_slot,
                       static_cast<decltype(yp)>(addend), op, (int)T, (int)D, (int)K, round_terms, (int)pieces, counts,
                       totals, (int)E);
  };
  auto run = [&](auto* yp, auto* op) {
    using E = std::remove_pointer_t<decltype(op)>;
    launch(K <= 8 ? combine_fwd_kernel<E, true> : combine_fwd_kernel<E, false>, yp, op);
  };
  if (dtype == MI355_F32) {
    run(static_cast<const float*>(y), static_cast<float*>(out));
  } else if (dtype == MI355_BF16) {
    run(static_cast<const uint16_t*>(y), static_cast<uint16_t*>(out));
  } else if (dtype == MI355_F64) {
    hipLaunchKernelGGL(combine_fwd_f64_kernel, dim3((unsigned)tokens), dim3(256), 0, as_stream(stream), static_cast<const double*>(y),
                       weights, row_of_slot, static_cast<double*>(out), (int)T, (int)D, (int)K);
  } else
    return fail(MI355_EINVAL, "combine_fwd: unknown dtype %d", dtype);
  return check_launch("combine_fwd");
}

extern "C" int mi355_combine_add_fwd(const void* y, int dtype, const float* weights, const int32_t* row_of_slot,
                                     const void* addend, void* out, int64_t T, int64_t D, int64_t K, int round_terms,
                                     void* stream) {
  return mi355_combine_count_fwd(y, dtype, weights, row_of_slot, addend, out, T, D, K, round_terms, nullptr, nullptr, 0, stream);
}

extern "C" int mi355_combine_fwd(const void* y, int dtype, const float* weights,
                                 const int32_t* row_of_slot, void* out, int64_t T, int64_t D,
                                 int64_t K, int round_terms, void* stream) {
  return mi355_combine_add_fwd(y, dtype, weights, row_of_slot, nullptr, out, T, D, K, round_terms, stream);
}

extern "C" int mi355_combine_bwd(const void* dout, const void* y, int dtype, const float* weights,
                                 const int32_t* row_of_slot, const int32_t* slot_of_row,
                                 const int32_t* total_rows, void* dy, float* dweights, int64_t T,
                                 int64_t D, int64_t K, int64_t row_capacity, void* stream) {
  MI355_REQUIRE(T >= 0 && D >= 1 && K >= 1 && K <= 64 && T < (1ll << 31) && D < (1ll << 31) &&
                    row_capacity >= 0 && row_capacity < (1ll << 31),
                "combine_bwd: bad shape (K must be <= 64)");
  const int token_blocks = (int)((T + 3) / 4);
  const int pad_blocks = slot_of_row ? (int)((row_capacity + 3) / 4) : 0;
  if (token_blocks + pad_blocks == 0) return MI355_OK;
  MI355_REQUIRE(T == 0 || (dout && weights && row_of_slot && dy), "combine_bwd: null pointer");
  MI355_REQUIRE(!slot_of_row || total_rows, "combine_bwd: total_rows required with slot_of_row");
  const dim3 grid((unsigned)(token_blocks + pad_blocks));
  // dy larger than the 256 MiB memory-side cache is written with non-temporal stores (as the
  // row scatter of the forward permutation does)
  const int stream_stores = row_capacity * D * (dtype == MI355_F32 ? 4 : 2) > (256ll << 20);
  if (dtype == MI355_F32)
    hipLaunchKernelGGL(combine_bwd_kernel<float>, grid, dim3(256), 0, as_stream(stream),
                       static_cast<const float*>(dout), static_cast<const float*>(y), weights,
                       row_of_slot, slot_of_row, total_rows, static_cast<float*>(dy), dweights,
                       (int)T, (int)D, (int)K, token_blocks, (int)row_capacity, stream_stores);
  else if (dtype == MI355_BF16)
    hipLaunchKernelGGL(combine_bwd_kernel<uint16_t>, grid, dim3(256), 0, as_stream(stream),
                       static_cast<const uint16_t*>(dout), static_cast<const uint16_t*>(y), weights,
                       row_of_slot, slot_of_row, total_rows, static_cast<uint16_t*>(dy), dweights,
                       (int)T, (int)D, (int)K, token_blocks, (int)row_capacity, stream_stores);
  else if (dtype == MI355_F64)
    hipLaunchKernelGGL(combine_bwd_f64_kernel, grid, dim3(256), 0, as_stream(stream),
                       static_cast<const double*>(dout), static_cast<const double*>(y), weights, row_of_slot,
                       slot_of_row, total_rows, static_cast<double*>(dy), dweights, (int)T, (int)D, (int)K,
                       token_blocks, (int)row_capacity);
  else
    return fail(MI355_EINVAL, "combine_bwd: unknown dtype %d", dtype);
  return check_launch("combine_bwd");
}

// ---- the two small ends of the backward that folds the combine into the expert kernels --
namespace mi355 {
namespace {

__global__ __launch_bounds__(256) void row_scale_kernel(const float* __restrict__ weights,
                                                        const int32_t* __restrict__ slot_of_row,
                                                        float* __restrict__ row_scale, int rows, int slots) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= rows) return;
  const int slot = slot_of_row[r];
  row_scale[r] = (slot >= 0 && slot < slots) ? weights[slot] : 0.0f;
}

__global__ __launch_bounds__(256) void scores_bwd_kernel(const float* __restrict__ partial, int pieces,
                                                         const int32_t* __restrict__ row_of_slot,
                                                         float* __restrict__ dweights, int slots, int rows) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= slots) return;
  const int row = row_of_slot[i];
  float acc = 0.0f;
  if (row >= 0 && row < rows) {
    const float* src = partial + static_cast<int64_t>(row) * pieces;
    for (int s = 0; s < pieces; ++s) acc += src[s];  // fixed order: the same bits every run
  }
  dweights[i] = acc;
}

}  // namespace
}  // namespace mi355

extern "C" int mi355_combine_row_scale(const float* weights_TK, const int32_t* slot_of_row, float* row_scale,
                                       int64_t T, int64_t K, int64_t row_capacity, void* stream) {
  using namespace mi355;
  MI355_REQUIRE(T >= 0 && K >= 1 && T * K < (1ll << 31) && row_capacity >= 0 && row_capacity < (1ll << 31),
                "combine_row_scale: bad shape");
  if (row_capacity == 0) return MI355_OK;
  MI355_REQUIRE(slot_of_row && row_scale && (weights_TK || T == 0), "combine_row_scale: null pointer");
  hipLaunchKernelGGL(row_scale_kernel, dim3((unsigned)((row_capacity + 255) / 256)), dim3(256), 0,
                     as_stream(stream), weights_TK, slot_of_row, row_scale, (int)row_capacity, (int)(T * K));
  return check_launch("combine_row_scale");
}

extern "C" int mi355_combine_scores_bwd(const float* dot_partial, int64_t pieces, const int32_t* row_of_slot,
                                        float* dweights_TK, int64_t T, int64_t K, int64_t row_capacity,
                                        void* stream) {
  using namespace mi355;
  MI355_REQUIRE(T >= 0 && K >= 1 && T * K < (1ll << 31) && pieces >= 1 && pieces <= 4096 && row_capacity >= 0 &&
                    row_capacity < (1ll << 31),
                "combine_scores_bwd: bad shape");
  if (T == 0) return MI355_OK;
  MI355_REQUIRE(row_of_slot && dweights_TK && (dot_partial || row_capacity == 0), "combine_scores_bwd: null pointer");
  hipLaunchKernelGGL(scores_bwd_kernel, dim3((unsigned)((T * K + 255) / 256)), dim3(256), 0, as_stream(stream),
                     dot_partial, (int)pieces, row_of_slot, dweights_TK, (int)(T * K), (int)row_capacity);
  return check_launch("combine_scores_bwd");
}

