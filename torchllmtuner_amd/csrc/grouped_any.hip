// Grouped expert products of any width: fp32, and bf16 whose widths are not on the 64-column grid (or
// are below the 384 columns) of the kernels in grouped_bf16.hip.  Widths are multiples of four.
//
// One kernel template over the element type, the product and the tile: 256 lanes as 2 x 2 waves on a
// TM x TN output tile, each wave (TM/2) x (TN/2) in 32x32 accumulators (v_mfma_f32_32x32x16_bf16; fp32 on 32-row
// tiles v_mfma_f32_32x32x2_f32, on larger ones products of bf16 pieces, below), 128 bytes of the contraction per step,
// two LDS stages (of pieces one), the next step's operands held in registers.  Operands are fetched 16 bytes at a time whatever the width
// (buffer loads: dword alignment suffices for them, and what lies past a matrix reads as zero; the ends
// access whole fours of elements, so the matrices themselves start on 16-byte boundaries); the tail of
// the contraction is zeroed as it is parked.  LDS holds an operand as it lies in memory -- contraction
// contiguous [row][128 B + 16] or strided [k][cols], padded (fp32) or its chunks swizzled (bf16) so that fragment reads
// are free of bank conflicts -- and the fragment reads (b128, b32, or the transposing b64 for bf16)
// make up for the difference.
//   Products and their fused ends: gate and up in one pass with SwiGLU; down; dh with the SwiGLU
// backward; drows as one contraction over both halves; all three weight gradients in one launch.
//   What bounds them at the sizes they are for is latency and CUs without work: few tiles, short
// contractions.  Small tiles are used until the large ones fill the chip: 64 rows, and for fp32 32 x 32, where
// the four waves hold the same tile and split each step's contraction (their shares are added through LDS in
// wave order) and four steps are requested ahead.
//   512 tokens of 8 fp32 experts of 256 x 512, two each, gate/up + down and the backward experts 26 + 33 us; 200 tokens of 16 of
// 640 x 1024, two each, 51 + 83; 4096 of them, four each, 450 + 930; 1531 tokens of 16 bf16 experts of 320 x 232, 21 + 40 us.
#include <algorithm>
#include <type_traits>

#include "bf16_tiles.h"
#include "common.h"
#include "grouped_any.h"
#include "router_few.h"
#include "select_bwd.h"
#include "tile_list.h"

namespace mi355 {
namespace {

enum AnyMode { ANY_GATEUP, ANY_KC, ANY_DH, ANY_DX, ANY_KS, ANY_DW };

struct AnyDw {  // c[e] (M, N) = a[segment e]^T (rows, M) . b[segment e] (rows, N)
  const void *a, *b;
  void* c;
  int M, N, nt;  // nt: column tiles
  int through;   // FOLD: 1 a's rows through the row index, scaled; 2 b's rows through it
};

struct AnyArgs {
  const void *a0, *a1, *b0, *b1;  // rows; weights (El, ., .).  GATEUP: w1, w3; DX: dgate, dup and w1, w3
  void *c0, *c1, *c2;             // GATEUP gate, up, h; DH dgate, dup
  const void *gate, *up;          // DH
  int K, N, ldb;                  // contraction (of one half), output columns, row length of the weights
  int64_t rows, w_elems;          // rows of the buffers, elements of one expert's weights
  const int32_t *seg_offsets, *seg_counts;
  TileList list;
  int El, col_tiles;
  AnyDw dw[3];
  int num_dw;
  // FOLD: row r of the tokens' matrix (GATEUP a0, DH a0, a weight gradient's a or b) is its row src[r] of src_rows, of the
  // output gradient scaled by scale[r] (and rounded, as a copy of it would be)
  const int32_t* src;
  int src_rows;
  const float* scale;
};

// Which work a workgroup has.  Consecutive workgroups go to the eight XCDs in turn, each with an L2 of its own, and tiles that share rows or weights
// should share one.  So an XCD has a run of the row products' tiles (expert, pass of TM rows, columns), without the passes that a plan's 256-row tiles
// leave empty, and whole rows of a weight gradient's tiles, dealt in turn: those of an expert read the same strip of the first operand, and one that has most of
// the rows, whose contraction is the longest, is still spread over all of them (a run of whole experts per XCD: 4096 tokens of a skewed router of 16 x 640 x 1020 1564
// -> 1770 us, and nothing more elsewhere).  A training step, us, workgroups as they come / the row products' in runs / both: fp32, 225 tokens of 16 x 628 x 832, three each,
// 195 / 157 / 155; 400 of 16 x 640 x 1020, four each, 271 / 238 / 238; 4096 of them 1478 / 1414 / 1410; 2723 of 8 x 176 x 276, four each, 170 / 165 / 163; 1500 of 8 x 320 x
// 400, three each, 166 / 156 / 155; bf16, four each, 4096 of 32 x 472 x 364 252 / 211 / 202, of 8 x 400 x 300 211 / 190 / 178; 4000 of 4 x 480 x 428 231 / 215 / 203;
// 1000 of 32 x 480 x 432 142 / 131 / 128; of skewed routers 185 / 160 / 158, 1564 / 1526 / 1525, 274 / 242 / 230.

// the block-th tile of `total`; false: there is none
__device__ __forceinline__ bool any_run(int& block, int total) {
  const int xcd = block & 7, within = block >> 3, each = total >> 3, more = total & 7;
  if (within >= each + (xcd < more ? 1 : 0)) return false;
  block = xcd * each + min(xcd, more) + within;
  return true;
}

template <typename T> struct El;
template <> struct El<float> {
  static constexpr int KS_PAD = 8;   // words: rows k and k + 4 half the banks apart
  using V4 = f32x4;
};
template <> struct El<uint16_t> {
  static constexpr int KS_PAD = 0;   // (swizzled, below)
  using V4 = u32x2;
};

__device__ __forceinline__ f32x4 any_pack(float, float a, float b, float c, float d) { return {a, b, c, d}; }
__device__ __forceinline__ u32x2 any_pack(uint16_t, float a, float b, float c, float d) { return {pack2(a, b), pack2(c, d)}; }
// COUNT values of a row, on 8 bytes (bf16) or 16
template <typename T, int COUNT> struct Row;
template <> struct Row<float, 4> {
  static __device__ __forceinline__ void load(const float* p, float (&f)[4]) {
    const f32x4 v = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = v[i];
  }
  template <typename V> static __device__ __forceinline__ void store(float* p, const V& v) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
  }
};
template <int COUNT> struct Row<uint16_t, COUNT> {
  typedef uint32_t Words __attribute__((ext_vector_type(COUNT / 2), aligned(8)));
  static __device__ __forceinline__ void load(const uint16_t* p, float (&f)[COUNT]) {
    const Words v = *reinterpret_cast<const Words*>(p);
#pragma unroll
    for (int i = 0; i < COUNT; ++i) f[i] = __uint_as_float(i & 1 ? v[i >> 1] & 0xffff0000u : v[i >> 1] << 16);
  }
  template <typename V> static __device__ __forceinline__ void store(uint16_t* p, const V& v) {
    Words w;
#pragma unroll
    for (int i = 0; i < COUNT / 2; ++i) w[i] = pack2(v[2 * i], v[2 * i + 1]);
    *reinterpret_cast<Words*>(p) = w;
  }
};
template <typename T>
__device__ __forceinline__ float any_round(float v) {
  if constexpr (sizeof(T) == 2) return round_bf16(v);
  else return v;
}

// Buffer resource over [base, end) of a matrix, clipped to the 32-bit range of the offsets.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t any_rsrc(const void* base, int64_t bytes) {
  const int64_t clipped = bytes < 0 ? 0 : bytes < 0xfffffffcll ? bytes : 0xfffffffcll;
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(static_cast<uint32_t>(clipped)), 0x00020000);
}

// One operand's tile: ROWS rows (or columns) of the output, one 128-byte step of the contraction.
template <typename T, bool KS, int ROWS>
struct Operand {
  static constexpr int E = 16 / sizeof(T), BKE = 128 / sizeof(T);
  static constexpr int PITCH = KS ? ROWS + El<T>::KS_PAD : BKE + E;
  static constexpr int ELEMS = KS ? BKE * PITCH : ROWS * PITCH;
  static constexpr int CPR = KS ? ROWS / E : 8;  // chunks per stored row
  static constexpr int N = ROWS * 8 / 256;       // chunks per lane and step

  // bf16, strided: a transposing read touches 64 bytes of four consecutive k rows per 32 lanes, and each row gets a quarter of the
  // banks -- rows of 128 bytes lie on alternate halves already.  (Padding for it took half as much LDS again, and with it
  // two of five workgroups a CU.  A training step of 4096 tokens of 32 x 480 x 432, four each, 323 -> 315 us, of 4 x 440 x 432 273 -> 264.)
  static __device__ __forceinline__ int swizzle(int k) {
    if constexpr (KS && sizeof(T) == 2) return CPR >= 16 ? (k & 3) << 2 : (k >> 1 & 1) << 2;
    else return 0;
  }
  static __device__ __forceinline__ int at(int tid, int i) {
    const int q = tid + 256 * i;
    return (q / CPR) * PITCH + ((q % CPR) ^ swizzle(q / CPR)) * E;
  }
  // keep what lies inside the contraction (kv of BKE elements); a multiple of four
  static __device__ __forceinline__ u32x4 clip(const u32x4& v, int tid, int i, int kv) {
    const int q = tid + 256 * i;
    const int k = KS ? q / CPR : (q % CPR) * E;
    u32x4 r = v;
    const bool lo = k < kv, hi = KS || sizeof(T) == 4 ? lo : k + 4 < kv;
    r[0] = lo ? r[0] : 0; r[1] = lo ? r[1] : 0;
    r[2] = hi ? r[2] : 0; r[3] = hi ? r[3] : 0;
    return r;
  }
};

// Fragments of one 32-row block.  The weights' operand is the first of the MFMA, so that a lane holds four
// consecutive columns of one output row.
template <bool KS, int ROWS>
__device__ __forceinline__ bf16x8 any_frag(const uint16_t* tile, int row, int kk, int lane) {
  using O = Operand<uint16_t, KS, ROWS>;
  if constexpr (!KS) {
    return *reinterpret_cast<const bf16x8*>(tile + (row + (lane & 31)) * O::PITCH + kk * 16 + 8 * (lane >> 5));
  } else {
    const int g = lane >> 4, i = lane & 15;
    const int k = kk * 16 + 8 * (g >> 1) + (i >> 2), c = row + 16 * (g & 1) + 4 * (i & 3);  // (row k + 4 has row k's key)
    const uint16_t* p = tile + k * O::PITCH + (((c >> 3) ^ O::swizzle(k)) << 3) + (c & 7);
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(LDS_PTR(p + 4 * O::PITCH));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
}
// fp32: the four values of k = 8 kk + 4 (lane / 32) ..
template <bool KS, int ROWS>
__device__ __forceinline__ f32x4 any_frag(const float* tile, int row, int kk, int lane) {
  using O = Operand<float, KS, ROWS>;
  const int k = 8 * kk + 4 * (lane >> 5);
  if constexpr (!KS) return *reinterpret_cast<const f32x4*>(tile + (row + (lane & 31)) * O::PITCH + k);
  f32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = tile[(k + j) * O::PITCH + row + (lane & 31)];
  return v;
}

// fp32 on tiles of 64 rows and more, where the matrix cores were the bound (137 TFLOP/s a large product, these 100): an operand
// is parked as three bf16 pieces, each the nearest to what the ones before leave, 24 bits and their signs together, and a product is
// the six products of pieces whose weights are within 2^-16 of the first; what is left out is 2^-26 of it.  bf16 products are
// 16 times as fast.  The six of 16 k are added up, the smallest first, before they meet the sum, which so is rounded once for every
// 16 products: over steps of 64-4096 tokens of 64-640 x 96-1020 the rms error against fp64 is 0.30-0.95 of what fp32 products
// gave (2409 tokens of 8 x 360 x 648: dx 8.2e-7 -> 2.7e-7, dw2 6.7e-7 -> 2.3e-7; added to the sum one by one, 4-10 % faster, 0.8-1.4).
//   Split where it is parked, once a workgroup, not where each of the waves reads it (5.5 vector instructions an element); one
// stage, so that LDS (61 KB on 128-row tiles) holds two workgroups a CU and one splits while the other multiplies.  A training step,
// us, fp32 products / pieces on the same tiles: 4096 tokens of 16 x 640 x 1020 (four each) 2012 / 1538, 4096 of 4 (two each) 1053 / 864, 1000
// of 16 x 512 x 800 (three each) 322 / 262, 1500 of 8 x 320 x 400 (three each) 198 / 172.  Two, three and four steps requested ahead: large
// products 3-9 % slower, small ones the same.
//   Three pieces hold what fp32 does from 2^-110 on (bf16 ends at 2^-133) and as long as the first of them and their products stay
// finite: a value that is not finite, or rounds to infinity, has NaN for its second piece.  A tile one of whose operands' values has lost bits,
// or with a result that is not finite, is formed again by fp32 products, which say what it is.  Looking costs 0.7-1.5 % of
// those steps (us, without / with: 1550 / 1561, 870 / 879, 261 / 265, 173 / 175; by comparing every value with 2^-110 8 %).
template <bool KS, int ROWS>
struct Pieces {
  using O = Operand<float, KS, ROWS>;       // (the chunks of four that a lane fetches)
  static constexpr int PITCH = KS ? ROWS : 40;  // 80 bytes: 16 rows' b128 reads fall on 64 different banks
  static constexpr int ELEMS = (KS ? O::BKE : ROWS) * PITCH;
  static __device__ __forceinline__ int at(int tid, int i) {
    const int q = tid + 256 * i, r = q / O::CPR, c = q % O::CPR;
    if constexpr (!KS) return r * PITCH + c * 4;
    else return r * PITCH + (((c >> 1) ^ Operand<uint16_t, true, ROWS>::swizzle(r)) << 3) + (c & 1) * 4;
  }
  // lost: the third remainders' bits together; what bf16 does not hold of one is in its lower half
  static __device__ __forceinline__ void park(uint16_t* tile, int tid, int i, const u32x4& v, uint32_t& lost) {
    u32x2 hi, mid, lo;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float a = __uint_as_float(v[2 * j]), b = __uint_as_float(v[2 * j + 1]);
      hi[j] = pack_bf16x2(a, b);
      const float a1 = a - __uint_as_float(hi[j] << 16), b1 = b - __uint_as_float(hi[j] & 0xffff0000u);
      mid[j] = pack_bf16x2(a1, b1);
      const float a2 = a1 - __uint_as_float(mid[j] << 16), b2 = b1 - __uint_as_float(mid[j] & 0xffff0000u);
      lo[j] = pack_bf16x2(a2, b2);
      lost |= __float_as_uint(a2) | __float_as_uint(b2);
    }
    uint16_t* p = tile + at(tid, i);
    *reinterpret_cast<u32x2*>(p) = hi;
    *reinterpret_cast<u32x2*>(p + ELEMS) = mid;
    *reinterpret_cast<u32x2*>(p + 2 * ELEMS) = lo;
  }
  static __device__ __forceinline__ bf16x8 frag(const uint16_t* tile, int row, int kk, int lane) {
    if constexpr (!KS) return *reinterpret_cast<const bf16x8*>(tile + (row + (lane & 31)) * PITCH + kk * 16 + 8 * (lane >> 5));
    else return any_frag<true, ROWS>(tile, row, kk, lane);
  }
};
__device__ __forceinline__ f32x16 any_mfma(const bf16x8& b, const bf16x8& a, const f32x16& acc) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, acc, 0, 0, 0);
}
__device__ __forceinline__ f32x16 any_mfma(const f32x4& b, const f32x4& a, f32x16 acc) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j], a[j], acc, 0, 0, 0);
  return acc;
}

// a chunk of a row, scaled and rounded
__device__ __forceinline__ u32x4 any_scale(float, const u32x4& v, float f) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __float_as_uint(__uint_as_float(v[i]) * f);
  return r;
}
__device__ __forceinline__ u32x4 any_scale(uint16_t, const u32x4& v, float f) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = pack2(__uint_as_float(v[i] << 16) * f, __uint_as_float(v[i] & 0xffff0000u) * f);
  return r;
}

template <typename T, int TM> constexpr bool any_split() { return sizeof(T) == 4 && TM >= 64; }

// LDS of one instantiation: two stages; on 32-row tiles also the four waves' partial tiles
template <typename T, int MODE, int TM, int TN>
constexpr int any_lds() {
  constexpr bool B_KS = MODE == ANY_DH || MODE == ANY_DX || MODE == ANY_KS || MODE == ANY_DW;
  constexpr int stages = 2 * (Operand<T, MODE == ANY_DW, TM>::ELEMS + Operand<T, B_KS, TN>::ELEMS);
  constexpr int parts = TM == 32 ? 4 * 32 * TN * 4 / (int)sizeof(T) : 0;
  if (any_split<T, TM>()) {
    constexpr int pieces = 3 * (Pieces<MODE == ANY_DW, TM>::ELEMS + Pieces<B_KS, TN>::ELEMS) / 2;
    return stages / 2 > pieces ? stages / 2 : pieces;
  }
  return stages > parts ? stages : parts;
}

// FOLD: the tokens' rows are read through the plan's row index, and the output gradient's are scaled by the routing weight,
// where they are fetched: no copy of either in row order exists.  A weight gradient's contraction runs over the rows, so
// its indexes are requested as many steps before their rows as those are before their use.  What it saves is two launches and
// two passes over row-ordered copies; a training step of the block, us, copied / in place: 512 fp32 tokens of 8 x 256 x 512 132 / 126, 1531
// bf16 of 16 x 320 x 232 136 / 128, 4096 of 32 x 480 x 432 (four each) 358 / 324, 4096 fp32 of 16 x 640 x 1024 1999 / 1989.
template <typename T, int MODE, int TM, int TN, bool FOLD>
__device__ __forceinline__ void any_tile(const AnyArgs& p, int block, T* smem) {
  constexpr bool A_KS = MODE == ANY_DW, B_KS = MODE == ANY_DH || MODE == ANY_DX || MODE == ANY_KS || MODE == ANY_DW;
  using OA = Operand<T, A_KS, TM>;
  using OB = Operand<T, B_KS, TN>;
  // 32-row tiles: every wave holds the whole tile and takes a quarter of each step's contraction
  constexpr bool KSPLIT = TM == 32;
  constexpr int BKE = OA::BKE, MI = KSPLIT ? 1 : TM / 64, NJ = KSPLIT ? TN / 32 : TN / 64;
  constexpr int KK = 128 / sizeof(T) / (sizeof(T) == 2 ? 16 : 8);
  static_assert(KK == 4, "a step's fragments are dealt to four waves");
  constexpr int AHEAD = TM == 32 ? 4 : 1;  // steps requested ahead
  constexpr int STAGE = OA::ELEMS + OB::ELEMS;
  constexpr bool SPLIT = any_split<T, TM>();
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = KSPLIT ? 0 : (wave >> 1) * (TM / 2), wn = KSPLIT ? 0 : (wave & 1) * (TN / 2);

  // ---- which tile
  int m_valid, n0, N = p.N, M = 0, m0 = 0, K = p.K, k_rows = 0;
  int64_t row0 = 0;
  const T *A0, *A1 = nullptr, *B0, *B1 = nullptr;
  T *C0 = static_cast<T*>(p.c0);
  int lda = p.K, ldb = p.ldb;
  int64_t a_bytes, b_bytes;
  constexpr bool ROWS_FOLD = FOLD && (MODE == ANY_GATEUP || MODE == ANY_DH), K_FOLD = FOLD && MODE == ANY_DW;
  bool through_a = false, through_b = false;  // K_FOLD
  int64_t first_row = 0;
  if constexpr (MODE == ANY_DW) {
    const int xcd = block & 7;
    int d = 0, at = block >> 3, strip = 0, strips, before = 0;  // at: among the XCD's tiles; before: rows of tiles of the products before
    for (;; ++d) {
      if (d == p.num_dw) return;
      strips = (p.dw[d].M + TM - 1) / TM;
      const int first = (xcd - before) & 7, all = p.El * strips, mine = all > first ? (all - first + 7) >> 3 : 0, tiles = mine * p.dw[d].nt;
      if (at < tiles) {
        strip = first + 8 * (at / p.dw[d].nt);
        break;
      }
      at -= tiles;
      before += all;
    }
    const AnyDw& w = p.dw[d];
    const int e = strip / strips;
    M = w.M; N = w.N;
    m0 = (strip - e * strips) * TM;
    n0 = (at % w.nt) * TN;
    m_valid = min(TM, M - m0);
    k_rows = p.seg_counts[e];
    const int64_t first = p.seg_offsets[e];
    lda = M; ldb = N; K = k_rows;
    A0 = static_cast<const T*>(w.a) + first * M + m0;
    B0 = static_cast<const T*>(w.b) + first * N + n0;
    a_bytes = ((p.rows - first) * M - m0) * static_cast<int64_t>(sizeof(T));
    b_bytes = ((p.rows - first) * N - n0) * static_cast<int64_t>(sizeof(T));
    C0 = static_cast<T*>(w.c) + static_cast<int64_t>(e) * M * N;
    if constexpr (K_FOLD) {
      first_row = first;
      through_a = w.through == 1;
      through_b = w.through == 2;
      if (through_a) {
        A0 = static_cast<const T*>(w.a) + m0;
        a_bytes = (static_cast<int64_t>(p.src_rows) * M - m0) * static_cast<int64_t>(sizeof(T));
      }
      if (through_b) {
        B0 = static_cast<const T*>(w.b) + n0;
        b_bytes = (static_cast<int64_t>(p.src_rows) * N - n0) * static_cast<int64_t>(sizeof(T));
      }
    }
  } else {
    // Which expert, pass of TM rows and columns: every wave adds up the experts' passes itself, and their tiles, to see whether the list has them all.
    auto passes_of = [&](int count) { return (count + TM - 1) / TM; };
    auto count_of = [&](int b) { return b + lane < p.El ? p.seg_counts[b + lane] : 0; };
    const int count0 = count_of(0);
    int total = 0, unlisted = -p.list.size();
    for (int b = 0; b < p.El; b += 64) {
      const int c = b ? count_of(b) : count0;
      total += __builtin_amdgcn_readlane(wave_scan(passes_of(c)), 63);
      unlisted += __builtin_amdgcn_readlane(wave_scan(listed_tiles(c)), 63);
    }
    if (!any_run(block, total * p.col_tiles)) return;
    const int pass_of_all = block / p.col_tiles;
    int e = 0, cnt = 0, before = 0, run = 0;
    for (int b = 0; b < p.El; b += 64) {
      const int c = b ? count_of(b) : count0, to = run + wave_scan(passes_of(c));
      const unsigned long long past = __ballot(to > pass_of_all);
      if (past) {
        const int l = __ffsll(past) - 1;
        e = b + l;
        cnt = __builtin_amdgcn_readlane(c, l);
        before = __builtin_amdgcn_readlane(to, l) - passes_of(cnt);
        break;
      }
      run = __builtin_amdgcn_readlane(to, 63);
    }
    const int q = block - before * p.col_tiles;
    const int pass = q / p.col_tiles;
    const int seg0 = p.seg_offsets[e];
    int first = seg0 + pass * TM;
    m_valid = min(TM, cnt - pass * TM);
    if (unlisted != 0 && !listed_rows(p.list, e, seg0, cnt, first, m_valid)) return;
    row0 = first;
    n0 = (q - pass * p.col_tiles) * (MODE == ANY_GATEUP ? TN / 2 : TN);
    A0 = static_cast<const T*>(p.a0) + (ROWS_FOLD ? 0 : row0 * lda);
    a_bytes = (ROWS_FOLD ? p.src_rows : p.rows - row0) * lda * static_cast<int64_t>(sizeof(T));
    if (MODE == ANY_DX) A1 = static_cast<const T*>(p.a1) + row0 * lda;
    const int64_t w = e * p.w_elems + (B_KS ? n0 : static_cast<int64_t>(n0) * ldb);
    B0 = static_cast<const T*>(p.b0) + w;
    if (MODE == ANY_GATEUP || MODE == ANY_DX) B1 = static_cast<const T*>(p.b1) + w;
    b_bytes = (p.w_elems - (w - e * p.w_elems)) * static_cast<int64_t>(sizeof(T));
  }
  // ---- operand offsets (bytes): fixed per lane, plus the step's
  uint32_t offA[OA::N], offB[OB::N];
  float row_scale[MODE == ANY_DH && FOLD ? OA::N : 1];
  auto source = [&](int64_t row) { return static_cast<uint32_t>(min(max(p.src[row], 0), p.src_rows - 1)); };
#pragma unroll
  for (int i = 0; i < OA::N; ++i) {
    const int q = tid + 256 * i, r = q / OA::CPR, c = (q % OA::CPR) * OA::E;
    if constexpr (ROWS_FOLD) {
      const int64_t row = row0 + min(r, m_valid - 1);
      offA[i] = (source(row) * lda + c) * sizeof(T);
      if constexpr (MODE == ANY_DH) row_scale[i] = p.scale[row];
    } else {
      offA[i] = (A_KS ? static_cast<uint32_t>(r) * lda + c : static_cast<uint32_t>(min(r, m_valid - 1)) * lda + c) * sizeof(T);
    }
  }
  const int b_rows = (MODE == ANY_GATEUP ? TN / 2 : TN);  // KC: weight rows of the tile (of each of the two)
#pragma unroll
  for (int i = 0; i < OB::N; ++i) {
    const int q = tid + 256 * i, r = q / OB::CPR, c = (q % OB::CPR) * OB::E;
    offB[i] = (B_KS ? static_cast<uint32_t>(r) * ldb + c
                    : static_cast<uint32_t>(min(r % b_rows, N - 1 - n0)) * ldb + c) * sizeof(T);
  }
  const int half_steps = (K + BKE - 1) / BKE, steps = MODE == ANY_DX ? 2 * half_steps : half_steps;
  u32x4 ra[AHEAD][OA::N], rb[AHEAD][OB::N];
  const auto rsA0 = any_rsrc(A0, a_bytes), rsB0 = any_rsrc(B0, b_bytes);
  const auto rsA1 = MODE == ANY_DX ? any_rsrc(A1, a_bytes) : rsA0;
  const auto rsB1 = (MODE == ANY_GATEUP || MODE == ANY_DX) ? any_rsrc(B1, b_bytes) : rsB0;
  // K_FOLD: source rows of the steps ahead; scales of the steps held
  // (bf16, one step requested ahead: the indexes go two, so that a step's are older than the rows of the step before it
  // and waiting for them does not wait for those; fp32 steps are long enough without)
  constexpr int SRC = K_FOLD && sizeof(T) == 2 ? 2 : AHEAD;
  uint32_t srcA[K_FOLD ? SRC : 1][K_FOLD ? OA::N : 1], srcB[K_FOLD ? SRC : 1][K_FOLD ? OB::N : 1];
  float k_scale[K_FOLD ? AHEAD : 1][K_FOLD ? OA::N : 1];
  auto row_of = [&](int s, int chunk_row) -> int64_t { return first_row + min(s * BKE + chunk_row, K - 1); };
  auto request_sources = [&](int slot, int s) {
    if constexpr (K_FOLD) {
      if (through_a) {
#pragma unroll
        for (int i = 0; i < OA::N; ++i) srcA[slot][i] = p.src[row_of(s, (tid + 256 * i) / OA::CPR)];
      }
      if (through_b) {
#pragma unroll
        for (int i = 0; i < OB::N; ++i) srcB[slot][i] = p.src[row_of(s, (tid + 256 * i) / OB::CPR)];
      }
    }
  };
  auto fetch = [&](int slot, int s, int src) {  // src: the slot of its sources
    const bool second = MODE == ANY_DX && s >= half_steps;
    const uint32_t k = static_cast<uint32_t>(second ? s - half_steps : s) * BKE;
    const uint32_t ka = (A_KS ? k * lda : k) * sizeof(T), kb = (B_KS ? k * ldb : k) * sizeof(T);
    auto rsA = second ? rsA1 : rsA0, rsB = second ? rsB1 : rsB0, rsU = MODE == ANY_GATEUP ? rsB1 : rsB;
    if constexpr (KSPLIT) {
      // a step past the end reads as zero, without traffic, so that requests are unconditional and the
      // compiler counts them exactly
      const int64_t an = s < steps ? a_bytes : 0, bn = s < steps ? b_bytes : 0;
      rsA = any_rsrc(second ? A1 : A0, an);
      rsB = any_rsrc(second ? B1 : B0, bn);
      rsU = MODE == ANY_GATEUP ? any_rsrc(B1, bn) : rsB;
    }
    // (a source row is clamped where it is used, not where it is requested: that would wait for it)
    auto within = [&](uint32_t row) { return static_cast<uint32_t>(min(max(static_cast<int>(row), 0), p.src_rows - 1)); };
#pragma unroll
    for (int i = 0; i < OA::N; ++i) {
      uint32_t at = offA[i] + ka;
      if constexpr (K_FOLD)
        if (through_a) at = (within(srcA[src][i]) * lda + ((tid + 256 * i) % OA::CPR) * OA::E) * sizeof(T);
      ra[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(rsA, at, 0, 0);
      if constexpr (K_FOLD)
        if (through_a) k_scale[slot][i] = p.scale[row_of(s, (tid + 256 * i) / OA::CPR)];
    }
#pragma unroll
    for (int i = 0; i < OB::N; ++i) {
      uint32_t at = offB[i] + kb;
      if constexpr (K_FOLD)
        if (through_b) at = (within(srcB[src][i]) * ldb + ((tid + 256 * i) % OB::CPR) * OB::E) * sizeof(T);
      rb[slot][i] = __builtin_amdgcn_raw_buffer_load_b128(i >= OB::N / 2 ? rsU : rsB, at, 0, 0);
    }
    request_sources(src, s + SRC);
  };
  auto prepare = [&](int slot, int s) {  // what was requested, scaled and clipped
    const int kv = K - (MODE == ANY_DX && s >= half_steps ? s - half_steps : s) * BKE;
    if constexpr (FOLD && MODE == ANY_DH) {
#pragma unroll
      for (int i = 0; i < OA::N; ++i) ra[slot][i] = any_scale(T{}, ra[slot][i], row_scale[i]);
    }
    if constexpr (K_FOLD) {
      if (through_a) {
#pragma unroll
        for (int i = 0; i < OA::N; ++i) ra[slot][i] = any_scale(T{}, ra[slot][i], k_scale[slot][i]);
      }
    }
    if (kv < BKE) {  // the tail: whatever was read past the contraction must not meet anything
#pragma unroll
      for (int i = 0; i < OA::N; ++i) ra[slot][i] = OA::clip(ra[slot][i], tid, i, kv);
#pragma unroll
      for (int i = 0; i < OB::N; ++i) rb[slot][i] = OB::clip(rb[slot][i], tid, i, kv);
    }
  };
  auto park = [&](int slot, int s, int stage) {
    T* As = smem + stage * STAGE;
    T* Bs = As + OA::ELEMS;
    prepare(slot, s);
#pragma unroll
    for (int i = 0; i < OA::N; ++i) *reinterpret_cast<u32x4*>(As + OA::at(tid, i)) = ra[slot][i];
#pragma unroll
    for (int i = 0; i < OB::N; ++i) *reinterpret_cast<u32x4*>(Bs + OB::at(tid, i)) = rb[slot][i];
  };
  // column block j of the wave: GATEUP's first half of the blocks are gate columns, the second the same of up
  auto bcol = [&](int j) {
    if constexpr (MODE == ANY_GATEUP) return (j < NJ / 2 ? 0 : TN / 2) + (KSPLIT ? 0 : (wave & 1) * (TN / 4)) + (j % (NJ / 2)) * 32;
    else return wn + j * 32;
  };
  static_assert(MODE != ANY_GATEUP || NJ >= 2, "a wave of the gate/up product holds both of a column");

  f32x16 acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  auto multiply = [&](const T* As, const T* Bs, int kk) {
    decltype(any_frag<A_KS, TM>(As, 0, 0, 0)) af[MI];
#pragma unroll
    for (int i = 0; i < MI; ++i) af[i] = any_frag<A_KS, TM>(As, wm + i * 32, kk, lane);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const auto bf = any_frag<B_KS, TN>(Bs, bcol(j), kk, lane);
#pragma unroll
      for (int i = 0; i < MI; ++i) acc[i][j] = any_mfma(bf, af[i], acc[i][j]);
    }
  };
  if constexpr (SPLIT) {
    using PA = Pieces<A_KS, TM>;
    using PB = Pieces<B_KS, TN>;
    uint16_t* As = reinterpret_cast<uint16_t*>(smem);
    uint16_t* Bs = As + 3 * PA::ELEMS;
    uint32_t lost_a = 0, lost_b = 0;
    if (steps > 0) {
      request_sources(0, 0);
      fetch(0, 0, 0);
    }
    for (int s = 0; s < steps; ++s) {
      prepare(0, s);
      __syncthreads();
#pragma unroll
      for (int i = 0; i < OA::N; ++i) PA::park(As, tid, i, ra[0][i], lost_a);
#pragma unroll
      for (int i = 0; i < OB::N; ++i) PB::park(Bs, tid, i, rb[0][i], lost_b);
      if (s + 1 < steps) fetch(0, s + 1, 0);
      __syncthreads();
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        bf16x8 af[3][MI];
#pragma unroll
        for (int piece = 0; piece < 3; ++piece)
#pragma unroll
          for (int i = 0; i < MI; ++i) af[piece][i] = PA::frag(As + piece * PA::ELEMS, wm + i * 32, kk, lane);
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          bf16x8 bf[3];
#pragma unroll
          for (int piece = 0; piece < 3; ++piece) bf[piece] = PB::frag(Bs + piece * PB::ELEMS, bcol(j), kk, lane);
          f32x16 part[MI];
#pragma unroll
          for (int i = 0; i < MI; ++i) part[i] = f32x16{};
#pragma unroll
          for (int sum = 2; sum >= 0; --sum)
#pragma unroll
            for (int pb = 0; pb <= sum; ++pb)
#pragma unroll
              for (int i = 0; i < MI; ++i) part[i] = any_mfma(bf[pb], af[sum - pb][i], part[i]);
#pragma unroll
          for (int i = 0; i < MI; ++i) acc[i][j] += part[i];
        }
      }
    }
    // (not what was read past the ends of an operand that lies strided: a lane's columns of it are the same every step)
    if (A_KS && m0 + (tid % OA::CPR) * OA::E >= M) lost_a = 0;
    if (B_KS && n0 + (tid % OB::CPR) * OB::E >= N) lost_b = 0;
    bool again = ((lost_a | lost_b) & 0xffffu) != 0;
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int n = n0 + bcol(j) - (MODE == ANY_GATEUP && j >= NJ / 2 ? TN / 2 : 0) + q * 8 + 4 * (lane >> 5);
          bool finite = true;
#pragma unroll
          for (int v = 0; v < 4; ++v) finite &= fabsf(acc[i][j][q * 4 + v]) < INFINITY;
          again |= !finite && wm + i * 32 + (lane & 31) < m_valid && n < N;
        }
    if (__syncthreads_or(again)) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
      for (int s = 0; s < steps; ++s) {
        request_sources(0, s);
        fetch(0, s, 0);
        __syncthreads();
        park(0, s, 0);
        __syncthreads();
        const T* Af = smem;
#pragma unroll 1
        for (int kk = 0; kk < KK; ++kk) multiply(Af, Af + OA::ELEMS, kk);
      }
      __syncthreads();
    }
  } else if constexpr (!KSPLIT) {
    if (steps > 0) {
#pragma unroll
      for (int i = 0; i < SRC; ++i) request_sources(i, i);
      fetch(0, 0, 0);
      park(0, 0, 0);
      if (steps > 1) fetch(0, 1, SRC - 1);
    }
    __syncthreads();
    auto step = [&](int s, int src) {
      if (s + 1 < steps) park(0, s + 1, (s + 1) & 1);
      if (s + 2 < steps) fetch(0, s + 2, src);
      const T* As = smem + (s & 1) * STAGE;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) multiply(As, As + OA::ELEMS, kk);
      __syncthreads();
    };
    if constexpr (SRC == 1) {
      for (int s = 0; s < steps; ++s) step(s, 0);
    } else {
      for (int s = 0; s < steps; s += 2) {
        step(s, 0);
        if (s + 1 < steps) step(s + 1, 1);
      }
    }
  } else {
    if (steps > 0) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) request_sources(i, i);
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) fetch(i, i, i);
      park(0, 0, 0);
      fetch(0, AHEAD, 0);
      phase_barrier();
    }
    for (int s0 = 0; s0 < steps; s0 += AHEAD) {
#pragma unroll
      for (int i = 0; i < AHEAD; ++i) {
        const int s = s0 + i;
        if (s >= steps) goto done;
        if (s + 1 < steps) park((i + 1) % AHEAD, s + 1, (s + 1) & 1);
        fetch((i + 1) % AHEAD, s + 1 + AHEAD, (i + 1) % AHEAD);
        const T* As = smem + (s & 1) * STAGE;
        multiply(As, As + OA::ELEMS, wave);
        phase_barrier();
      }
    }
  done:
    // quad q of every column block goes to wave q, which adds the four waves' shares in their order
    f32x4* part = reinterpret_cast<f32x4*>(smem);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        part[((wave * NJ + j) * 4 + q) * 64 + lane] =
            f32x4{acc[0][j][q * 4], acc[0][j][q * 4 + 1], acc[0][j][q * 4 + 2], acc[0][j][q * 4 + 3]};
    phase_barrier();
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      f32x4 v = part[(j * 4 + wave) * 64 + lane];
#pragma unroll
      for (int w = 1; w < 4; ++w) v += part[((w * NJ + j) * 4 + wave) * 64 + lane];
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[0][j][r] = v[r];
    }
  }

  // ---- the fused ends, on N values of one output row from column n on
  auto finish = [&](int64_t at, auto count, const auto& v, const auto& u) {
    constexpr int COUNT = decltype(count)::value;
    using C = Row<T, COUNT>;
    if constexpr (MODE == ANY_GATEUP) {
      float h[COUNT];
#pragma unroll
      for (int r = 0; r < COUNT; ++r) h[r] = any_round<T>(v[r] / (1.0f + expf(-v[r]))) * u[r];
      C::store(C0 + at, v);
      C::store(static_cast<T*>(p.c1) + at, u);
      C::store(static_cast<T*>(p.c2) + at, h);
    } else if constexpr (MODE == ANY_DH) {
      float g[COUNT], up[COUNT], dg[COUNT], du[COUNT];
      C::load(static_cast<const T*>(p.gate) + at, g);
      C::load(static_cast<const T*>(p.up) + at, up);
#pragma unroll
      for (int r = 0; r < COUNT; ++r) {
        const float sig = 1.0f / (1.0f + expf(-g[r]));
        du[r] = v[r] * any_round<T>(g[r] * sig);
        dg[r] = any_round<T>(v[r] * up[r]) * (sig * (1.0f + g[r] * (1.0f - sig)));
      }
      C::store(C0 + at, dg);
      C::store(static_cast<T*>(p.c1) + at, du);
    } else {
      C::store(C0 + at, v);
    }
  };
  const int64_t c_row0 = MODE == ANY_DW ? m0 : row0;
  // the accumulators hold, per lane, output row lane & 31 of a block and four consecutive columns per q
  if constexpr (KSPLIT) {
    const int m = lane & 31;
#pragma unroll
    for (int j = 0; j < (MODE == ANY_GATEUP ? NJ / 2 : NJ); ++j) {
      const int n = n0 + wave * 8 + j * 32 + 4 * (lane >> 5);
      if (m >= m_valid || n >= N) continue;  // N is a multiple of four
      const f32x16 &c = acc[0][j], &cu = acc[0][MODE == ANY_GATEUP ? j + NJ / 2 : j];
      finish((c_row0 + m) * N + n, std::integral_constant<int, 4>{}, f32x4{c[0], c[1], c[2], c[3]}, f32x4{cu[0], cu[1], cu[2], cu[3]});
    }
  } else {
    // Through LDS, 32 rows at a time, so that a row's columns are read and written together, 16 bytes a lane: four columns of 32
    // rows an instruction were 32 lines for 256 bytes (bf16).  Experts' forward / backward, us, before and now: 16000 rows of 8 x 480 x
    // 432 70 / 163, 66 / 135; of 32 x 472 x 364 79 / 167, 75 / 148; 6000 of 16 x 440 x 360 34 / 69, 33 / 63; fp32, 16000 of 16 x
    // 640 x 1024 472 / 976, 463 / 958.
    constexpr int E = OA::E, NB = MODE == ANY_GATEUP ? NJ / 2 : NJ, W = 32 * NB, CH = W / E, P = W + E;
    constexpr int TILES = MODE == ANY_GATEUP ? 2 : 1;
    static_assert(4 * TILES * 32 * P <= any_lds<T, MODE, TM, TN>(), "the waves' tiles fit");
    T* st = smem + wave * (TILES * 32 * P);
    const int c0 = n0 + (MODE == ANY_GATEUP ? (wave & 1) * (TN / 4) : wn);
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      if (wm + i * 32 >= m_valid) break;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const f32x16& c = acc[i][j];
          *reinterpret_cast<typename El<T>::V4*>(st + ((j / NB) * 32 + (lane & 31)) * P + (j % NB) * 32 + q * 8 + 4 * (lane >> 5)) =
              any_pack(T{}, c[q * 4], c[q * 4 + 1], c[q * 4 + 2], c[q * 4 + 3]);
        }
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): the wave's own writes have landed
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int it = 0; it < CH / 2; ++it) {
        const int idx = it * 64 + lane, m = idx / CH, c = (idx % CH) * E;
        const int row = wm + i * 32 + m, n = c0 + c;
        if (row < m_valid && n < N) {
          float v[E], u[E];
          Row<T, E>::load(st + m * P + c, v);
          if constexpr (MODE == ANY_GATEUP) Row<T, E>::load(st + (32 + m) * P + c, u);
          const int64_t at = (c_row0 + row) * N + n;
          if (E == 4 || n + E <= N) finish(at, std::integral_constant<int, E>{}, v, u);
          else finish(at, std::integral_constant<int, 4>{}, v, u);  // (N is a multiple of four)
        }
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);
      __builtin_amdgcn_wave_barrier();
    }
  }
}

// (two workgroups a CU said to the compiler: at most 256 registers, and products then go to ordinary ones -- from the others every
// partial sum had to be copied before it could be added)
template <typename T, int MODE, int TM, int TN, bool FOLD>
__global__ __launch_bounds__(256, 2) void any_kernel(AnyArgs p) {
  __shared__ __attribute__((aligned(16))) T smem[any_lds<T, MODE, TM, TN>()];
  any_tile<T, MODE, TM, TN, FOLD>(p, blockIdx.x, smem);
}

// What runs beside the experts' products in workgroups past theirs: the router gate's weight gradient, or the selection's backward.
template <typename T>
__device__ __forceinline__ void beside_part(const GateDw& job, int part, float* lds) { gate_dw_part<T>(job, part, lds); }
template <typename T>
__device__ __forceinline__ void beside_part(const SelectBwd& job, int part, float* lds) { select_bwd_part<1, T>(job, part, lds); }
int64_t beside_parts(const GateDw& job) { return gate_dw_parts(job); }
int64_t beside_parts(const SelectBwd& job) { return select_bwd_parts(job); }

// The experts' dH and one of those.  The selection's backward and dH read the output gradient and what the forward left, neither the other's result, and
// neither fills the chip; the gate's weight gradient, which reads what the selection's left, then runs beside the input and weight gradients of the experts
// (any_dx_dw_kernel), or, where those are launches of their own, here behind it.  With the gate's input gradient taking the sum over a
// token's rows along, and the slices' sum beside it, a backward has three launches, or four, instead of seven.  The selection's backward as a launch of its own in
// front / beside dH, a training step's GPU time and a whole step on a box where the host is what it waits for, us: 512 fp32 tokens of two of 8 x 256 x 512 84 / 80, 130 / 125; 1531 bf16 of
// four of 16 x 320 x 232 92 / 86, 130 / 125; 105 of two of 16 x 464 x 168 63 / 59, 132 / 126; 3310 of two of 8 x 352 x 360 118 / 114, 130 / 125.
template <typename T, int TM, int TN, typename Job>
__global__ __launch_bounds__(256, 2) void any_dh_beside_kernel(AnyArgs p, Job job, int blocks) {
  constexpr int A = any_lds<T, ANY_DH, TM, TN>(), B = kGateDwLds * 4 / sizeof(T);
  static_assert(kGateDwLds >= 4 * 2 * kSelectBesideE, "either job's LDS");
  __shared__ __attribute__((aligned(16))) T smem[A > B ? A : B];
  const int block = blockIdx.x;
  if (block < blocks) any_tile<T, ANY_DH, TM, TN, true>(p, block, smem);
  else beside_part<T>(job, block - blocks, reinterpret_cast<float*>(smem));
}

// The input gradient and the weight gradients of a backward pass read the same buffers and write different
// ones: with few tiles each they share a launch (at 512 fp32 tokens of 8 experts 26 + 16 us one after the
// other).  The longer contraction starts first.  With a fold the gate's weight gradient may come last.
template <typename T, int TX, int TW, bool FOLD>
__global__ __launch_bounds__(256, 2) void any_dx_dw_kernel(AnyArgs dx, AnyArgs dw, int dx_blocks, int dw_blocks, int dw_first, GateDw gate) {
  constexpr int A = any_lds<T, ANY_DX, TX, TX>(), B = any_lds<T, ANY_DW, TW, TW>(), C = FOLD ? kGateDwLds * 4 / sizeof(T) : 0;
  __shared__ __attribute__((aligned(16))) T smem[A > B ? (A > C ? A : C) : (B > C ? B : C)];
  if constexpr (FOLD) {
    if (static_cast<int>(blockIdx.x) >= dx_blocks + dw_blocks) {
      gate_dw_part<T>(gate, blockIdx.x - dx_blocks - dw_blocks, reinterpret_cast<float*>(smem));
      return;
    }
  }
  const int block = static_cast<int>(blockIdx.x) - (dw_first ? dw_blocks : 0);  // of dx
  if (block >= 0 && block < dx_blocks) any_tile<T, ANY_DX, TX, TX, false>(dx, block, smem);
  else any_tile<T, ANY_DW, TW, TW, FOLD>(dw, dw_first ? blockIdx.x : block - dx_blocks, smem);
}

template <int MODE, int TM, int TN>
int launch_any(const AnyArgs& p, int dtype, int64_t blocks, hipStream_t s, const char* what, const GateDw* gate = nullptr,
               const SelectBwd* select = nullptr) {
  if (blocks <= 0) return MI355_OK;
  if (dtype != MI355_F32 && TM == 32) return fail(MI355_EUNSUP, "%s: 32-row tiles are for fp32", what);
  if constexpr (MODE == ANY_DH) {
    auto beside = [&](const auto& job) {
      using Job = std::decay_t<decltype(job)>;
      const dim3 grid((unsigned)(blocks + beside_parts(job))), lanes(256);
      if (dtype == MI355_F32) {
        hipLaunchKernelGGL((any_dh_beside_kernel<float, TM, TN, Job>), grid, lanes, 0, s, p, job, (int)blocks);
      } else if constexpr (TM != 32) {
        hipLaunchKernelGGL((any_dh_beside_kernel<uint16_t, TM, TN, Job>), grid, lanes, 0, s, p, job, (int)blocks);
      }
      return check_launch(what);
    };
    if (select) return beside(*select);
    if (gate) return beside(*gate);
  }
  auto run = [&](auto fold) {
    constexpr bool FOLD = decltype(fold)::value;
    const dim3 grid((unsigned)blocks), lanes(256);
    if (dtype == MI355_F32) hipLaunchKernelGGL((any_kernel<float, MODE, TM, TN, FOLD>), grid, lanes, 0, s, p);
    else if constexpr (TM != 32) hipLaunchKernelGGL((any_kernel<uint16_t, MODE, TM, TN, FOLD>), grid, lanes, 0, s, p);
  };
  if constexpr (MODE == ANY_GATEUP || MODE == ANY_DH || MODE == ANY_DW) {
    if (p.src) run(std::true_type{});
    else run(std::false_type{});
  } else {
    run(std::false_type{});
  }
  return check_launch(what);
}

// passes of t rows that the experts have, at most
int64_t any_passes(const AnyArgs& p, int64_t t) { return p.rows / t + std::min<int64_t>(p.El, p.rows); }

// Large tiles (128 x 128) once they give two workgroups for every CU, for bf16 already where they give every second CU one: its
// steps are mostly loads and LDS, which a large tile has half as many of (the forward, us, 64 / 128: 141 tiles, 2000 rows of 32 x
// 300 x 300, 18.3 / 19.0; 156, 4000 of 8 x 480 x 432, 30.7 / 26.4; 186, 6000 of 16 x 440 x 360, 41.7 / 34.6; 252, 4000 of 32 x
// 480 x 432, 40.0 / 33.5).  Not so dH, whose end has as much to do (4000 of 8 x 480 x 432: the backward 52 / 56), and not the input
// gradient where the weight gradients share its launch, which is worth more (8000 of 4 x 480 x 432: 86 / 94): two a CU.  fp32 products
// run on 32 x 32 tiles where 64-row ones leave CUs without work or, with few rows per expert, are mostly padding.  Experts' forward
// / backward in us, 64 against 32:
//   few tiles: 119 (75 rows per expert, 320 x 400) 29 / 40 against 21 / 27, 135 (375, 256 x 300) 26 / 35 against 23 / 31, 152 (250,
//     512 x 512) 40 / 49 against 34 / 45, 250 (750, 256 x 300) 30 / 42 against 37 / 46, 312 (250, 256 x 512) 34 / 48 against 35 / 47;
//   16 experts of 640 x 1024: 25 rows each 73 / 124 against 50 / 84, 50 rows 75 / 128 against 67 / 118, 75 rows 77 / 138 against
//     81 / 138, 250 rows 145 / 279 against 189 / 338.
// The lines for pieces (64 rows per expert; the weight gradients' 160 and 448 tiles and 400 rows, below) against those fp32 products had
// (160; 256 and 512 tiles, no rows), a training step, us, theirs / these: 200 tokens of 16 x 640 x 1020, two each, 185 / 162, 400, four each, 310 / 282,
// 600 of 16 x 512 x 800, four each, 283 / 243, 1000 of 8 x 640 x 640, two each, 229 / 205; from 2000 tokens of 16 x 640 x 1020 on the same.
// bf16 steps are shorter and gain nothing (14 / 17 against 14 / 18, slower with more tiles).
int row_tile(const AnyArgs& p, int dtype, int64_t El, int64_t cols, int bf16_large) {
  auto tiles = [&](int64_t t) { return any_passes(p, t) * ((cols + t - 1) / t); };
  if (dtype == MI355_F32 && (p.rows <= 64 * El || tiles(64) < 200)) return 32;
  return tiles(128) >= (dtype == MI355_F32 ? 512 : bf16_large) ? 128 : 64;
}

template <int MODE>
int launch_rows(AnyArgs& p, int dtype, int64_t El, int64_t cols, hipStream_t s, const char* what,
                const GateDw* gate = nullptr, const SelectBwd* select = nullptr) {
  constexpr bool GU = MODE == ANY_GATEUP;
  const int t = row_tile(p, dtype, El, cols, MODE == ANY_DH ? 512 : 150), width = GU && t == 128 ? 64 : t;
  p.col_tiles = (int)((cols + width - 1) / width);
  const int64_t blocks = any_passes(p, t) * p.col_tiles;
  MI355_REQUIRE(blocks < (1ll << 30), "%s: too many tiles", what);
  if (t == 128) return launch_any<MODE, 128, 128>(p, dtype, blocks, s, what, gate, select);
  return t == 64 ? launch_any<MODE, 64, GU ? 128 : 64>(p, dtype, blocks, s, what, gate, select)
                 : launch_any<MODE, 32, GU ? 64 : 32>(p, dtype, blocks, s, what, gate, select);
}

// the weight gradients' tiles, and each one's columns of them
int64_t dw_tiles(AnyArgs& p, int64_t El, int tile) {
  int64_t tiles = 0;
  for (int d = 0; d < p.num_dw; ++d) {
    AnyDw& w = p.dw[d];
    w.nt = (w.N + tile - 1) / tile;
    tiles += El * ((w.M + tile - 1) / tile) * w.nt;
  }
  return tiles;
}
// the workgroups of those: of each product a whole round of rows of tiles over the XCDs
int64_t dw_blocks(const AnyArgs& p, int tile) {
  int64_t blocks = 0;
  for (int d = 0; d < p.num_dw; ++d) blocks += (p.El * ((p.dw[d].M + tile - 1) / tile) + 7) / 8 * 8 * static_cast<int64_t>(p.dw[d].nt);
  return blocks;
}

}  // namespace

// (a matrix of rows and an expert's weights within the 32-bit range of the operand offsets; matrices that
// start anywhere else than an allocation would go to the strided kernels, which load element by element)
bool any_path_ok(int dtype, int64_t D, int64_t F, int64_t R, std::initializer_list<const void*> matrices) {
  return aligned16(matrices) && (dtype == MI355_F32 || dtype == MI355_BF16) && D % 4 == 0 && F % 4 == 0 &&
         std::max(R * std::max(D, F), D * F) * (dtype == MI355_F32 ? 4 : 2) < (int64_t{1} << 32) - 4;
}

static AnyArgs any_args(const AnySeg& g, int64_t rows, const AnyFold* f = nullptr) {
  AnyArgs p{};
  p.El = (int)g.El;
  if (f) {
    p.src = f->token_of_row; p.src_rows = (int)f->tokens; p.scale = f->row_scale;
  }
  p.rows = rows;
  p.seg_offsets = g.seg_offsets; p.seg_counts = g.seg_counts;
  p.list = {g.tile_expert, g.tile_row0, g.num_tiles, (int)std::min<int64_t>(g.tile_capacity, INT32_MAX)};
  return p;
}

int any_gateup(const AnySeg& g, int dtype, const void* rows, const void* w1, const void* w3, void* gate, void* up, void* h,
               int64_t D, int64_t F, int64_t R, const AnyFold* f, hipStream_t s) {
  AnyArgs p = any_args(g, R, f);
  p.a0 = rows; p.b0 = w1; p.b1 = w3; p.c0 = gate; p.c1 = up; p.c2 = h;
  p.K = (int)D; p.N = (int)F; p.ldb = (int)D; p.w_elems = D * F;
  return launch_rows<ANY_GATEUP>(p, dtype, g.El, F, s, "grouped gate/up");
}

int any_linear(const AnySeg& g, int dtype, const void* x, const void* w, void* y, int64_t I, int64_t O, int64_t R,
               hipStream_t s) {
  AnyArgs p = any_args(g, R);
  p.a0 = x; p.b0 = w; p.c0 = y;
  p.K = (int)I; p.N = (int)O; p.ldb = (int)I; p.w_elems = I * O;
  return launch_rows<ANY_KC>(p, dtype, g.El, O, s, "grouped linear");
}

int any_linear_dx(const AnySeg& g, int dtype, const void* dy, const void* w, void* dx, int64_t I, int64_t O, int64_t R,
                  hipStream_t s) {
  AnyArgs p = any_args(g, R);
  p.a0 = dy; p.b0 = w; p.c0 = dx;
  p.K = (int)O; p.N = (int)I; p.ldb = (int)I; p.w_elems = I * O;
  return launch_rows<ANY_KS>(p, dtype, g.El, I, s, "grouped linear dx");
}

int any_dh(const AnySeg& g, int dtype, const void* dy, const void* w2, const void* gate, const void* up, void* dgate,
           void* dup, int64_t D, int64_t F, int64_t R, const AnyFold* f, const AnyGate* router, const AnySelect* select,
           hipStream_t s) {
  AnyArgs p = any_args(g, R, f);
  p.a0 = dy; p.b0 = w2; p.c0 = dgate; p.c1 = dup; p.gate = gate; p.up = up;
  p.K = (int)D; p.N = (int)F; p.ldb = (int)F; p.w_elems = D * F;
  GateDw job{};
  SelectBwd sel{};
  if (router) job = gate_dw_job(router->dlogits, router->x, router->partial, f->tokens, D, router->E);
  if (select)
    sel = {select->logits, select->ids, nullptr, nullptr, DotPieces{}, DotRows{select->dout, select->y, select->row_of_slot, (int)D, (int)R},
           BalanceGrad{select->aux_f, select->aux_scale, select->padding}, select->dlogits, (int)f->tokens, (int)select->E,
           (int)select->K, select->score_func, select->route_norm, select->route_scale, MI355_SELECT_TOPK};
  return launch_rows<ANY_DH>(p, dtype, g.El, F, s, "grouped dh", router ? &job : nullptr, select ? &sel : nullptr);
}

namespace {
// How a backward pass is launched: the weight gradients' tile, the input gradient's, and whether they share a launch.
struct BackwardPlan {
  bool dw_large, dw_small, one;
  int t;
};
BackwardPlan backward_plan(const AnyArgs& p, AnyArgs& w, int dtype, int64_t El, int64_t D, const void* drows, int count, int64_t R) {
  // Weight gradients on 128 x 128 tiles once these fill the chip; fp32 ones where their contraction is long enough to be what
  // takes the time (us, the backward, 64 / 128: 250 rows an expert 279 / 290, 500 497 / 482, 1000 950 / 895).  fp32 on 32 x 32 tiles while
  // there are few (us, 64 / 32: 48 tiles 32 / 24, 96 28 / 22, 240 35 / 38).
  const bool f32 = dtype == MI355_F32;
  // bf16 ones also where the input gradient is large enough for a launch of its own (16000 rows of 8 x 480 x 432, 384 tiles: 183 / 162;
  // a step of 4000 tokens of 4 x 480 x 428, four each, 192 tiles: 264 / 277).
  // ... but with 64 x 64 tiles input and weight gradients share a launch and the selection's backward runs beside dH, which is worth more where 128 x 128
  // ones cover a quarter more than those, and where all of it is small.  A step of bf16, us, large tiles / one launch of small ones, by R D F in 10^9 and what large tiles cover over
  // small ones: 4096 tokens of 8 x 400 x 300, four each (2.0, 1.37) 172.7 / 158.2; 8192 of it, three each (2.9) 239.8 / 223.3; 3000 of 32 x 400 x 300 (1.4) 148.9 / 141.8; 4096 of
  // 16 x 440 x 400 (2.9, 1.31) 214.6 / 199.9; of 32 x 320 x 300, three each (1.2, 1.44) 138.0 / 126.8; 2500 of 16 x 480 x 400 (1.9, 1.14) 154.5 / 145.2; 4096 of 32 x it, two each
  // (1.6) 157.9 / 154.4; 3000 of 16 x 480 x 360 (2.1, 1.0) 153.5 / 152.0; 4096 of 32 x 472 x 364 (2.8, 1.0) 197.4 / 208.4; of 32 x 480 x 432 (3.4, 1.14) 223.3 / 227.4; 8192 of 16 x
  // it (6.8) 346 / 363; 16000 of 16 x 320 x 232 (4.8, 1.2) 339 / 338.
  auto covered = [&](int64_t t) { return (w.dw[0].M + t - 1) / t * t * ((w.dw[0].N + t - 1) / t * t); };
  const bool together = !f32 && drows && count &&
                        (4 * covered(128) >= 5 * covered(64) || R * w.dw[0].M * w.dw[0].N <= int64_t{2400} << 20);
  const bool alone = !f32 && drows && row_tile(p, dtype, El, D, 512) == 128;
  const bool dw_large = !together && count && dw_tiles(w, El, 128) >= (f32 ? 448 : alone ? 300 : 512) && !(f32 && R < 400 * El);
  const int64_t tiles = dw_tiles(w, El, dw_large ? 128 : 64);
  const bool dw_small = f32 && tiles < 160;
  if (dw_small) dw_tiles(w, El, 32);
  const int t = together ? 64 : row_tile(p, dtype, El, D, count && !dw_large ? 512 : 150);
  return {dw_large, dw_small, drows && count && !dw_large && t < 128, t};
}

void set_grads(AnyArgs& w, const AnyGrad* grads, int count) {
  for (int i = 0; i < count; ++i)
    w.dw[i] = {grads[i].a, grads[i].b, grads[i].c, (int)grads[i].M, (int)grads[i].N, 0, grads[i].through};
  w.num_dw = count;
}
}  // namespace

bool any_backward_is_one_launch(const AnySeg& g, int dtype, const void* drows, int64_t D, const AnyGrad* grads, int count, int64_t R) {
  const AnyArgs p = any_args(g, R);
  AnyArgs w = any_args(g, R);
  set_grads(w, grads, count);
  return backward_plan(p, w, dtype, g.El, D, drows, count, R).one;
}

int any_backward(const AnySeg& g, int dtype, const void* dgate, const void* dup, const void* w1, const void* w3, void* drows,
                 int64_t D, int64_t F, const AnyGrad* grads, int count, int64_t R, const AnyFold* f, const AnyGate* router,
                 hipStream_t s) {
  AnyArgs p = any_args(g, R);
  p.a0 = dgate; p.a1 = dup; p.b0 = w1; p.b1 = w3; p.c0 = drows;
  p.K = (int)F; p.N = (int)D; p.ldb = (int)D; p.w_elems = D * F;
  AnyArgs w = any_args(g, R, f);
  set_grads(w, grads, count);
  const BackwardPlan plan = backward_plan(p, w, dtype, g.El, D, drows, count, R);
  const int64_t tiles = dw_blocks(w, plan.dw_small ? 32 : plan.dw_large ? 128 : 64);
  const bool dw_large = plan.dw_large, dw_small = plan.dw_small, one = plan.one;
  const int t = plan.t;
  MI355_REQUIRE(tiles < (1ll << 30), "grouped weight gradients: too many tiles");
  MI355_REQUIRE(!router || (one && f), "grouped backward: nothing to form the gate's gradient beside");
  if (one) {
    p.col_tiles = (int)((D + t - 1) / t);
    const int64_t dx_blocks = any_passes(p, t) * p.col_tiles;
    MI355_REQUIRE(dx_blocks < (1ll << 30), "grouped drows: too many tiles");
    GateDw gate{};
    if (router) gate = gate_dw_job(router->dlogits, router->x, router->partial, f->tokens, D, router->E);
    const dim3 grid((unsigned)(dx_blocks + tiles + (router ? gate_dw_parts(gate) : 0)));
    const int dw_first = R / g.El > 2 * F;
    auto run = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, p, w, (int)dx_blocks, (int)tiles, dw_first, gate);
    };
    auto choose = [&](auto fold) {
      constexpr bool FOLD = decltype(fold)::value;
      if (dtype == MI355_BF16) run(any_dx_dw_kernel<uint16_t, 64, 64, FOLD>);
      else if (dw_small) run(t == 64 ? any_dx_dw_kernel<float, 64, 32, FOLD> : any_dx_dw_kernel<float, 32, 32, FOLD>);
      else run(t == 64 ? any_dx_dw_kernel<float, 64, 64, FOLD> : any_dx_dw_kernel<float, 32, 64, FOLD>);
    };
    if (f) choose(std::true_type{});
    else choose(std::false_type{});
    return check_launch("grouped drows and weight gradients");
  }
  if (drows)
    if (int rc = launch_rows<ANY_DX>(p, dtype, g.El, D, s, "grouped drows")) return rc;
  if (!count) return MI355_OK;
  if (dw_small) return launch_any<ANY_DW, 32, 32>(w, dtype, tiles, s, "grouped weight gradients");
  return dw_large ? launch_any<ANY_DW, 128, 128>(w, dtype, tiles, s, "grouped weight gradients")
                  : launch_any<ANY_DW, 64, 64>(w, dtype, tiles, s, "grouped weight gradients");
}

}  // namespace mi355
