// bf16 MFMA tile helpers shared by the grouped expert GEMMs and the router projections:
// vector types, the two LDS operand layouts and their fragment reads, and a barrier that
// leaves global memory traffic in flight.
//
// LDS layouts (no padding, XOR swizzles; 16-byte chunks), BK = 64 contraction elements
// per K step:
//   KC  contraction axis contiguous in HBM: [row][64 k], chunk c of row r stored at
//       c ^ ((r >> 1) & 7); a fragment is one ds_read_b128 (measured conflict-free;
//       the key r & 7 costs a 2-way conflict).
//   KS  contraction axis strided in HBM: [k][cols], chunk c of row k stored at
//       c ^ ((k & 3) << 2) (16 chunks or more per row); a fragment is two ds_read_b64_tr_b16 (LDS transpose
//       reads: lane i of a 16-lane group supplies the address of row i/4, 8-byte
//       piece i%4, and receives column i of the four rows).
// v_mfma_f32_32x32x16_bf16 takes per lane 8 bf16 of each operand (row lane%32,
// k = 8*(lane/32)..+7) and yields 16 fp32 (column lane%32, rows 8*(i/4) + 4*(lane/32) + i%4).
#pragma once
#include "common.h"

namespace mi355 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

constexpr int BK = 64;

// KS swizzle key of LDS row k, in 16-byte chunks: a transpose read touches four
// consecutive k rows and 64 bytes of each per 32 lanes, and rows are a multiple of
// 256 bytes apart, so each row's four chunks are moved to their own quarter of the banks.
__device__ __forceinline__ int ks_key(int k) { return (k & 3) << 2; }

#define LDS_PTR(p) ((__attribute__((address_space(3))) s16x4*)(p))

// ---- fragment reads -----------------------------------------------------------------
__device__ __forceinline__ bf16x8 frag_kc(const uint16_t* tile, int row, int kk, int lane) {
  const int r = row + (lane & 31);
  const int c = kk * 2 + (lane >> 5);
  return *reinterpret_cast<const bf16x8*>(tile + r * BK + ((c ^ ((r >> 1) & 7)) << 3));
}

template <int COLS>
__device__ __forceinline__ bf16x8 frag_ks(const uint16_t* tile, int col, int kk, int lane) {
  const int g = lane >> 4, i = lane & 15;
  const int k = kk * 16 + 8 * (g >> 1) + (i >> 2);  // k & 3 == i >> 2 for both reads
  const int c = col + 16 * (g & 1) + 4 * (i & 3);
  const int off = (((c >> 3) ^ ks_key(k)) << 3) + (c & 7);
  const uint16_t* p = tile + k * COLS + off;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(p));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(p + 4 * COLS));
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

// ---- fragments for v_mfma_f32_16x16x32_bf16 -------------------------------------------
// Per lane 8 bf16 of each operand: row lane%16, k = 8*(lane/16)..+7 of a 32-wide K block;
// 4 fp32 of the result: column lane%16, rows 4*(lane/16) + i.  With random operand bits
// this shape sustains about 14 % more than 32x32x16 on MI355X (a quarter of the
// accumulator bytes per instruction for half the flops, and power is what limits both).
// KS key for the 16x16x32 reader: 32 lanes of a transpose read touch rows k..k+3 and
// k+8..k+11, 32 bytes of each, so the eight rows get an eighth of the banks each.
__device__ __forceinline__ int ks_key16(int k) { return ((k & 3) << 2) | (((k >> 3) & 1) << 1); }

// ---- requests straight into LDS ----------------------------------------------------------
typedef const __attribute__((address_space(3))) char* lds_cptr;

// Requests 16 (4) bytes a lane from base + voff + soff, straight into LDS: lane l's land at byte lds + 16 l (4 l).  Written
// out because the compiler drains the whole load counter in front of every LDS read once it knows of such a request; waited for by lds_wait.
// (base, soff and lds are wave-uniform; byte offsets up to 4 GiB; the wait states are for scalar registers that a vector instruction wrote just before)
__device__ __forceinline__ u32x4 lds_rsrc(uint64_t base, uint32_t bytes) {
  return u32x4{static_cast<uint32_t>(base), static_cast<uint32_t>(base >> 32), bytes, 0x00020000u};
}
template <bool STREAM = false, uint32_t BYTES = 0xffffffffu>  // with the non-temporal hint; from a buffer of so many bytes, zeros for what lies past its end
__device__ __forceinline__ void lds_load16(uint64_t base, uint32_t voff, uint32_t soff, uint32_t lds) {
  if constexpr (STREAM)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 ::"s"(lds), "v"(voff), "s"(lds_rsrc(base, BYTES)), "s"(soff) : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 ::"s"(lds), "v"(voff), "s"(lds_rsrc(base, BYTES)), "s"(soff) : "memory");
}
// the same from a buffer of `bytes` bytes; zeros for what lies past its end
__device__ __forceinline__ void lds_load16_within(uint64_t base, uint32_t bytes, uint32_t voff, uint32_t lds) {
  const u32x4 rsrc = {static_cast<uint32_t>(base), static_cast<uint32_t>(base >> 32), bytes, 0x00020000u};
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
               ::"s"(lds), "v"(voff), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void lds_load4_within(uint64_t base, uint32_t bytes, uint32_t voff, uint32_t lds) {
  const u32x4 rsrc = {static_cast<uint32_t>(base), static_cast<uint32_t>(base >> 32), bytes, 0x00020000u};
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, 0 offen lds"
               ::"s"(lds), "v"(voff), "s"(rsrc) : "memory");
}
__device__ __forceinline__ void lds_load4(uint64_t base, uint32_t voff, uint32_t soff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dword %1, %2, %3 offen lds"
               ::"s"(lds), "v"(voff), "s"(lds_rsrc(base, 0xffffffffu)), "s"(soff) : "memory");
}
// at most N of the wave's requests and stores are still under way
template <int N>
__device__ __forceinline__ void lds_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// the wave's LDS reads and writes are done, and at most N of its requests under way; then the workgroup's barrier
template <int N>
__device__ __forceinline__ void lds_sync() {
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (N < 63) lds_wait<N>();
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
// the same value, of which the compiler knows nothing: what is formed from it is formed there, not held in registers over a K loop
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}
// orders a wave's LDS writes and reads of its own region
__device__ __forceinline__ void wave_lds_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}
// LDS at a byte address (by way of the pointers' width on the host, where this is only compiled)
template <typename T>
__device__ __forceinline__ __attribute__((address_space(3))) T* lds_at(uint32_t at) {
  return (__attribute__((address_space(3))) T*)(static_cast<uintptr_t>(at));
}
__device__ __forceinline__ bf16x8 lds_read16(uint32_t at) { return *lds_at<const bf16x8>(at); }
__device__ __forceinline__ int lds_read_i32(uint32_t at) { return *lds_at<const int>(at); }
// Eight k of 16 columns from rows of PITCH bytes, as the 16x16x32 MFMA wants them.  Lane i of group g = lane / 16 asks for the 8-byte piece i % 4 of the
// 16 columns in row k = 8 g + i / 4 (chunk swizzled by ks_key16(k), the key of row k + 4 too) and receives column i of rows 8 g .. 8 g + 7.
template <uint32_t PITCH>
__device__ __forceinline__ bf16x8 lds_read_tr(uint32_t at) {
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_at<s16x4>(at));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(lds_at<s16x4>(at + 4 * PITCH));
  const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_bit_cast(bf16x8, v);
}

// Workgroup barrier that waits for this wave's own LDS operations only: global loads and
// stores stay in flight across it.
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

__device__ __forceinline__ uint32_t pack2(float a, float b) { return pack_bf16x2(a, b); }

}  // namespace mi355
