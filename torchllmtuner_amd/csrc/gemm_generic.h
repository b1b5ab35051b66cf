// Generic strided GEMM with fp32 MFMA accumulation (v_mfma_f32_32x32x2_f32).
//
// C(m,n) = sum_k A(m,k) * B(k,n) with arbitrary element strides on A and B, any
// mix of fp32 / bf16 storage, and three ways of slicing the problem:
//   DENSE   one problem, optional split-K into fp32 partials
//   ROWSEG  the M axis is a list of expert segments (tile list); B is picked per
//           expert (forward and data-gradient grouped GEMMs)
//   KSEG    one problem per expert whose K range is that expert's row segment
//           (weight-gradient grouped GEMMs)
// It carries the fp32 configuration, the router projections and every shape the
// bf16 MFMA kernels do not accept; it is not the bf16 hot path.
#pragma once

#include "common.h"

namespace mi355 {

enum GemmMode { GEMM_DENSE = 0, GEMM_ROWSEG = 1, GEMM_KSEG = 2 };

struct GemmArgs {
  const void* A;
  const void* B;
  void* C;
  const float* bias;  // per output column, fp32, may be null
  const void* addend; // DENSE, no split: C = round(result) + addend, in C's dtype and layout; may be null
  int64_t a_rs, a_cs; // A(m,k) = A[m*a_rs + k*a_cs]
  int64_t b_rs, b_cs; // B(k,n) = B[k*b_rs + n*b_cs]
  int64_t ldc;
  int64_t b_es, c_es; // expert strides (elements) for ROWSEG (B) and KSEG (C)
  int M, N, K;
  int mode;
  int accumulate;     // C += result (read-modify-write in C's dtype)
  int ksplit;         // DENSE only: >1 writes fp32 partials to C + z*M*ldc
  int tile_m;         // ROWSEG: rows per listed tile (multiple of 64)
  const int32_t* seg_offsets;
  const int32_t* seg_counts;
  const int32_t* tile_expert;
  const int32_t* tile_row0;
  const int32_t* num_tiles;
};

// a_dtype / b_dtype / c_dtype are MI355_F32 or MI355_BF16.
int launch_gemm(const GemmArgs& args, int a_dtype, int b_dtype, int c_dtype,
                dim3 grid, hipStream_t stream);

// Grid helpers.
dim3 gemm_grid_dense(int M, int N, int ksplit);
dim3 gemm_grid_rowseg(int64_t tile_capacity, int tile_m, int N);
dim3 gemm_grid_kseg(int M, int N, int El);

// out = sum_z partial[z] (+bias), partial: (ksplit, M, N) fp32 contiguous.
int launch_splitk_reduce(const float* partial, void* out, int out_dtype, int64_t MN,
                         int ksplit, hipStream_t stream);

// What a router's input gradient is added to (all null: nothing): `rows`, the experts' input gradients, summed over a token's K <= 16
// slots, and `addend`, each sum rounded.
struct RowSum {
  const void* addend = nullptr;
  const void* rows = nullptr;
  const int32_t* row_of_slot = nullptr;
  int64_t K = 0, row_capacity = 0;
};
// Router projections (router_gemm.hip).  Backward: three bf16 MFMAs per fp32 product, for bf16
// tokens, fp32 weights, D and E multiples of 64.
bool router_x3_ok(int x_dtype, int w_dtype, int64_t D, int64_t E);
int64_t router_x3_bwd_workspace(int64_t T, int64_t D, int64_t E);
// Backward for few experts, fp32 weights, D a multiple of four: both gradients in one launch (dx, dw: null = skip).
bool router_few_ok(int x_dtype, int w_dtype, int64_t D, int64_t E);
bool router_few_bwd_ok(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E);
int64_t router_few_bwd_workspace(int64_t T, int64_t D, int64_t E);
int router_few_bwd(const float* dlogits, const void* x, int x_dtype, const float* w, const RowSum& sum, void* dx, float* dw,
                   void* workspace, int64_t T, int64_t D, int64_t E, hipStream_t s);
// The same where the dW parts have run (`partial`, a slice of the tokens each) and the addend is the sum of the experts' rows.
int router_rows_bwd(const float* dlogits, int x_dtype, const float* w, const void* rows, const int32_t* row_of_slot,
                    int64_t row_capacity, int64_t K, const void* addend, void* dx, const float* partial, float* dw, int64_t T,
                    int64_t D, int64_t E, hipStream_t s);
// Forward: `splits` (T, E) partial sums of the contraction, to be added in order (with the bias,
// unless splits is 1: then it is added already and the one partial is the logits); 0 = no kernel
// of that file serves the case.  `pieces` is scratch of router_fwd_pieces_bytes.
int router_fwd_splits(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E);
int64_t router_fwd_pieces_bytes(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E);
int64_t router_fwd_kept_bytes(int x_dtype, int w_dtype, int64_t T, int64_t D, int64_t E);
int router_fwd_partial(const void* x, int x_dtype, const float* w, const float* bias, float* partial, void* pieces, void* keep,
                       int64_t T, int64_t D, int64_t E, hipStream_t s);
int router_logits_reduce(const float* partial, const float* bias, float* logits, int64_t T, int64_t E, int splits,
                         hipStream_t s);
int router_x3_bwd(const float* dlogits, const void* x, const float* w, const void* pieces, const RowSum& sum,
                  void* dx, float* dw, void* workspace, int64_t T, int64_t D, int64_t E, hipStream_t s);

}  // namespace mi355
