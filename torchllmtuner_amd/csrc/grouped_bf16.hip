// Grouped SwiGLU expert GEMMs in bf16 on the gfx950 matrix cores.
//
// Products (no transpose is ever materialised):
//   gate/up  rows . w1^T, rows . w3^T   A KC, B KC   fused SiLU*up epilogue
//   down     h . w2^T                   A KC, B KC
//   dh       dy . w2                    A KC, B KS   fused SwiGLU backward epilogue
//   drows    dgate . w1 + dup . w3      A KC, B KS   (one accumulator, K = 2F)
//   dw*      a_e^T . b_e                A KS, B KS   K = the expert's rows
//
// Shape of the kernels.  256x256 output tiles for the row-tiled products and the weight
// gradients alike, eight waves per workgroup as 4 (rows) x 2 (columns), two per SIMD, each
// wave a 64x128 accumulator tile; one workgroup per CU, two 64 KiB LDS stages of operand
// tiles.  Row tiles come from the permutation plan's tile list (up to 256 rows of one expert each).
//
// K loop of the row-tiled products.  Operands go from memory straight into LDS (1 KiB a wave and instruction,
// the swizzle applied to the address each lane asks for), so no register holds them on the way: 64
// of a wave's 256 registers hold two sets of fragments instead, and the next quarter's fragments are
// read under this quarter's MFMAs.  A K step of 64 is four quarters of 16 MFMAs and two barriers: behind the first, where the rows and half of the
// weights have been read, their part of the stage is requested for the K step after the next; behind the second, the other half.  Every request has
// one and a half K steps to arrive.  Requests and reads go out between the 16-row blocks of MFMAs: in bursts
// behind the barriers they cost 7 % (all eight waves issue them at once while the matrix cores run dry).  The requests
// run on into the next tile, whose first two K steps land while this one's results are written through 4 KiB a wave of LDS of their own.
// A tile's 16-row blocks are dealt to the wave rows in turn and the loop exists for 0 to 4 blocks a wave, so
// that a tile that is not full costs what its rows cost and no branch stands between MFMAs (a branch per block: 3-5 % of a full tile).
//
// What that measured, us, operands parked in LDS through registers / straight into LDS: 128 experts of 2048 x 768, 8192 tokens of eight each: gate/up
// 487 / 433, down 250 / 226, dH 309 / 289, dRows 443 / 392; one dense segment of 4096 rows of 7168 x 2048 198 / 172, 109 / 98, 130 / 107, 209 / 185 (gate
// and up not kept: 1.38 PFLOP/s), 300 rows of it 129 / 90, 41 / 31, 92 / 64, 80 / 60; 32 experts of 7168 x 2048, 128 rows each 385 / 366,
// 217 / 204, 203 / 195, 399 / 387 (there the weights' way from memory counts), nine rows each 317 / 314, 169 / 168, 164 / 159, 317 / 334: the one
// that lost, a read of the weights at 5.6 TB/s.  The same bits.
//
// What is left.  With operands of random bits the card's power management holds the core clock near 1.5-1.9 GHz
// (a register-resident MFMA loop sustains 1.45-2.2 PFLOP/s by operand values instead of the 2.5 of the data sheet); with constant operands the same
// launches take 10-20 % less.  Without requests the loop takes 20-35 % less, without barriers 1-3 %.  Around the loop:
//   * persistent workgroups: block b serves XCD b % 8 and walks that XCD's contiguous
//     run of tiles with stride gridDim/8, so the tiles in flight on an XCD are
//     neighbours that share an expert's weights in its L2, and no workgroup launch sits
//     between two tiles;
//   * tile metadata looked up two tiles ahead;
//   * hardware bf16 conversion and transcendental-unit sigmoid in the epilogues (they
//     were VALU bound).
//
// The weight gradients' loop is the same, with both operands' contraction strided: what a barrier frees is the first or the last 32 k of both.
// Rows past the segment lie past the end of the buffer that a request names, which makes them zeros.  A gathered operand's row indices are requested a K step before
// its rows, into the wave's own LDS.  The contraction is the rows, two to eight K steps of an expert where the load is balanced, so requests run over tile ends into
// as many as two tiles, and a tile's stores may still be under way in the next one's first step: their number is known, and waits count them.
// What bounds them: 128 experts of 2048 x 768, 512 rows each: 248 / 222 us, 241 / 218, 241 / 217 (0.93 PFLOP/s; operands parked through registers / straight into
// LDS), a tile 18 us, 13 of them K steps; 16384 tokens of a skewed router 477 / 437, 468 / 425; 32 of 7168 x 2048, 128 rows each 231 / 209, 228 / 206 (the
// results, written at 4.6 TB/s); one dense segment of 4096 rows 116 / 102, 120 / 105; 12 or fewer rows an expert of 2048 x 768 75 / 77 (written at 5.2 TB/s).
// Beside the MFMAs the loop has 48 reads and 140 other instructions a wave and K step, and they count: with addresses formed from scratch at each request (100
// more) it took 8-10 % longer, with the row indices in scalar registers 3 %.
// A gathered row's address without a branch for rows past the segment and with a 24-bit product (30 fewer), and a result's as one addition: dW2 of the first 210 / 203,
// dW1 and dW3 409 / 402, of 250 rows each 108 / 105, 203 / 198, of the skewed router 364 / 359, 685 / 671; of 32 of 7168 x 2048, 128 rows 170 / 166.
//
// Instructions count in the row tiles too.  A result's address used to be formed from scratch, with a division, a 64-bit product and a branch for rows past the
// last (about 35 vector instructions a store, 24 stores a tile of gate/up, 3 us of its 8 us epilogue); now the tile's rows are a buffer that ends behind the
// last of them and an address is one addition.  A request of weights used to branch on whether it carries the non-temporal hint; now the loop exists with
// and without it (a K step's 104 scalar and 41 vector instructions are 62 and 4).  Rows past the last of a tile were read as copies of it; now they are zeros that nothing is read
// for, but of dH.  The three, us, before / with them: 128 experts of 2048 x 768, 512 rows each by Poisson draws gate/up 475 / 435, dRows 412 / 391, down 229 / 221; 16384
// tokens of a skewed router 801 / 765, 772 / 731, 418 / 407; 64 of 1024 x 512, 281 rows 66 / 63, 56 / 53; one dense segment of 4096 rows of 7168 x 2048 178 / 172, 203 / 189, 99 / 97, dH
// (the first two) 114 / 105.  Most of it is the first's: the present code with a branch at each request instead of the second has gate/up, dRows and dH of the 512 rows in 415 / 393 / 299
// instead of 404 / 383 / 299, of 700 dense rows 130 / 79 / 85 instead of 121 / 75 / 79, of 520 rows of the 64 experts 86 / 75 / 91 instead of 85 / 74 / 91; with copies instead of the third 405 / 385,
// 121 / 76, 85 / 73 (369 instead of 364 in gate/up of 200 rows of 32 of 7168 x 2048).
//
// MFMA of both: v_mfma_f32_16x16x32_bf16.  Per lane 8 bf16 of each operand (row lane%16,
// k = 8*(lane/16)..+7), 4 fp32 of the result (column lane%16, rows 4*(lane/16) + i).
// With random operand bits this shape sustains about 14 % more than 32x32x16 on this
// card (2.17 against 1.90 PFLOP/s register-resident, +7 % in a whole K loop).  The weight tile is passed as the FIRST operand
// and the activation tile as the second, so a lane ends up with four CONSECUTIVE
// output columns of one output row: epilogues pack them and go through LDS to
// write 16-byte, fully coalesced rows.
//
// The LDS layouts (KC / KS) and fragment reads are in bf16_tiles.h.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

#include "bf16_tiles.h"
#include "common.h"
#include "tile_list.h"

namespace mi355 {
namespace {

constexpr int NT = 512;  // threads per workgroup

// 1 / (1 + e^-x) on the transcendental unit (v_exp_f32, v_rcp_f32: about 1 ulp each; every
// use is rounded to bf16 right after)
__device__ __forceinline__ float fast_sigmoid(float x) {
  return __builtin_amdgcn_rcpf(1.0f + __expf(-x));
}

// int32 data that no kernel of this file writes (the plan's arrays), for uniform lookups
typedef const int32_t __attribute__((address_space(4))) * const_i32;

// LDS of the row-tiled kernels, in bytes: two stages of operands (A tile, B tile), 4 KiB a wave for its results
constexpr uint32_t A_BYTES = 32768, STAGE_BYTES = 65536;
constexpr uint32_t kNoRow = 0xffffff80u;  // no row of a matrix of whole 128-byte lines below 4 GiB begins there
constexpr int R_LDS_BYTES = 2 * STAGE_BYTES + 8 * 4096;

// n / d for 0 <= n < 2^31 and a divisor that the host knows: a product instead of the thirty instructions of a division, of which a tile's lookups had five.
// (mul = ceil(2^shift / d) with shift = 31 + ceil(log2 d) is below 2^32 and n * (mul * d - 2^shift) below 2^shift.)
struct Divisor {
  uint32_t mul, shift;
};
inline Divisor divisor(int64_t d) {
  uint32_t log = 0;
  while ((int64_t{1} << log) < d) ++log;
  return {static_cast<uint32_t>(((uint64_t{1} << (31 + log)) + d - 1) / d), 31 + log};
}
__device__ __forceinline__ int quotient(int n, Divisor d) {
  return static_cast<int>((static_cast<uint64_t>(static_cast<uint32_t>(n)) * d.mul) >> d.shift);
}
__device__ __forceinline__ int third(int n) { return static_cast<int>(__umulhi(static_cast<uint32_t>(n), 0x55555556u)); }

// RM_DLIN: the product of RM_DH (rows . w[e], the weight's contraction axis strided) with a plain epilogue:
// the input gradient of one grouped linear map
enum RowMode { RM_GATEUP = 0, RM_DOWN = 1, RM_DH = 2, RM_DX = 3, RM_DLIN = 4 };

struct RowArgs {
  const uint16_t* a0;  // GATEUP rows | DOWN h | DH dy | DX dgate
  const uint16_t* a1;  // DX dup
  const uint16_t* b0;  // GATEUP w1 | DOWN w2 | DH w2 | DX w1
  const uint16_t* b1;  // GATEUP w3 | DX w3
  uint16_t* o0;        // GATEUP gate | DOWN y | DH dgate | DX drows
  uint16_t* o1;        // GATEUP up   | DH dup
  uint16_t* o2;        // GATEUP h
  const uint16_t* gate;  // DH
  const uint16_t* up;    // DH
  const int32_t* a_src;  // GATEUP, DH: row -> row of a0 to read (token gather), or null
  int a_rows;            // rows of a0 when a_src is given: gathered indices are clamped to [0, a_rows)
  // DH with a_src (the combine's backward folded in): a0 is the layer's output gradient (T, D),
  // row r stands for row_scale[r] * a0[a_src[r]]; o2 receives row_scale * h and dot_partial
  // [row][dot_slots] the pieces of <unscaled dh row, h row>, one per 128 output columns
  const float* row_scale;
  float* dot_partial;
  int dot_slots;
  const int32_t* seg_offsets;
  const int32_t* seg_counts;
  const int32_t* tile_expert;
  const int32_t* tile_row0;
  const int32_t* num_tiles;
  int D, F;
  int n_tiles;
  Divisor by_n_tiles, by_steps;  // n_tiles; K steps
  int stream;  // weights of experts with one row tile are read with the non-temporal hint
  int short_tiles;  // tiles of up to 128 rows may take the place of the listed ones
  int El;
};

// Rows of a short tile, and whether short tiles (`total`, `n_tiles` of them across) take the place of the 256-row ones (`whole` of all experts' rows, `listed` in the list) on
// `blocks` workgroups.  Not where the list leaves tiles out, which the counts know nothing of: short tiles searched the list for their rows and read the weights of all experts.
// Half and a quarter of 128 experts of 2048 x 768 listed, 60 rows each, us, short tiles / the list's: gate/up 141 / 84, 138 / 42, down 80 / 45, 78 / 24; of 32 of 7168 x 2048 dRows
// 322 / 165, 323 / 76.
constexpr int kShortTile = 128;
__host__ __device__ inline bool short_tiles_serve(int total, int whole, int listed, int n_tiles, int blocks) {
  auto rounds = [&](int n) { return (n * n_tiles + blocks - 1) / blocks; };
  return listed == whole && total * 4 <= whole * 5 && rounds(total) <= rounds(whole);
}

// The tiles of up to 128 rows that the experts' rows make (at most 256 experts), found by every wave from the counts.
struct ShortTiles {
  int to[4];  // lane l, b: tiles of the experts up to and with 64 b + l
  int total = 0, whole = 0;  // tiles; those of 256 rows
  __device__ __forceinline__ void find(const RowArgs& p) {
    const int lane = threadIdx.x & 63;
    int count[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) count[b] = 64 * b + lane < p.El ? p.seg_counts[64 * b + lane] : 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      to[b] = total + wave_scan((count[b] + kShortTile - 1) / kShortTile);
      total = __builtin_amdgcn_readlane(to[b], 63);
      whole += __builtin_amdgcn_readlane(wave_scan(listed_tiles(count[b])), 63);
    }
  }
  // the expert of tile t and the tiles of those before it
  __device__ __forceinline__ int expert(int t, int& before) const {
    int e = 0;
#pragma unroll
    for (int b = 3; b >= 0; --b) {
      const unsigned long long past = __ballot(to[b] > t);
      if (past) e = 64 * b + __ffsll(past) - 1;
    }
    const int l = (e - 1) & 63, b = (e - 1) >> 6;
    before = e == 0 ? 0 : __builtin_amdgcn_readlane(b < 2 ? (b == 0 ? to[0] : to[1]) : (b == 2 ? to[2] : to[3]), l);
    return e;
  }
};

// Row-tiled kernel: 256 rows of one expert x 64 NJ output columns, 8 waves as 4 (rows) x 2 (columns), each wave
// 64 rows -- the 16-row blocks w, w + 4, w + 8, w + 12 for wave row w -- x 32 NJ.  GATEUP's columns are half gate and half
// up columns of the same f range, so a wave holds gate and up of the same 16 NJ f.

typedef __amdgpu_buffer_rsrc_t RowsOut;

struct TileMeta {
  int e, row0, valid, n0, nt;
  int k_start;  // the contraction's first K step; it goes on from step 0 after the last
  bool stream;  // no other tile reads the weights
};

// sum over each group of 16 (8) consecutive lanes, left in all of them (DPP row operations)
template <int LANES = 16>
__device__ __forceinline__ float row16_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));   // quad_perm [1,0,3,2]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));   // quad_perm [2,3,0,1]
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xf, 0xf, false));  // row_half_mirror
  if constexpr (LANES == 16)
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x140, 0xf, 0xf, false));  // row_mirror
  return v;
}

// SAVE_GU (GATEUP only): also write gate and up, which the backward reads; a forward-only caller
// leaves them out -- a third of the kernel's output bytes and of its epilogue's LDS traffic.
//
// TURN (weights with the contraction contiguous): a tile's contraction starts at a K step of its own, by expert and
// column tile, and goes on from step 0 after the last.  Workgroups run in step, and with the same start all of
// them read the same 128 bytes of weight rows that lie a row length apart: rows of 2048 elements, 4 KiB, then meet few memory
// channels at a time.  The column tile counts only where the output is a whole number of tiles: a last tile
// that would overhang computes some of its neighbour's columns again and must give the same bits, so both add up in
// the same order.  An expert's row tiles and, where there are several, its column tiles stay in step: they share operands in L2.
template <int MODE, int NJ, bool GATHER, bool SAVE_GU, bool TURN, int MB>
__device__ __forceinline__ void row_tiles(const RowArgs& p, const ShortTiles& tiles) {
  constexpr int WM = 4, WN = 2;            // waves along the rows and along the columns
  constexpr int TBM = 16 * MB * WM;        // rows of the tile
  constexpr bool SHORT = MB == 2;
  constexpr uint32_t A_BYTES = TBM * 128u, STAGE_BYTES = A_BYTES + 32768u;
  constexpr int BNT = 32 * NJ * WN;        // output columns of the tile (WN waves x NJ x 32)
  constexpr int NA = TBM / 64;             // 1 KiB pieces of the A tile a wave requests per K step
  constexpr int NB = BNT / 64;             // the same for B
  constexpr bool DH_LIKE = (MODE == RM_DH || MODE == RM_DLIN);  // same operands, different epilogue
  constexpr bool B_KS = (DH_LIKE || MODE == RM_DX);
  // Pieces of B requested behind barrier X and behind barrier Y: the columns that a wave's first half of MFMAs reads and the others; with the
  // contraction strided its first and its last 32 k (whole rows of the tile, 512 bytes: 256-byte halves of all 64 k, requested apart, cost 4-8 % where the product
  // is a read of the weights).  Narrow down tiles: a piece holds both halves of a wave's columns.
  constexpr int NBX = MODE == RM_DOWN && NJ == 2 ? 0 : NB / 2, NBY = NB - NBX;
  constexpr int VM = NBX ? NA + NB : NA;   // requests younger than those a barrier of the loop waits for
  constexpr int VM_EPI = SHORT ? NA + NB : NBX ? NBY : 0;    // ... than those that the next tile's first K step needs
  static_assert(!GATHER || MODE == RM_GATEUP || MODE == RM_DH, "only gate/up and dH gather their rows");
  static_assert(!SHORT || MODE != RM_DH, "dH's epilogue counts the requests of two stages");
  static_assert(!TURN || !B_KS, "only contractions that are contiguous in memory are turned");
  static_assert(!(GATHER && MODE == RM_DH) || NJ == 4 || NJ == 2, "the fused dH epilogue reduces over 16 lanes per row, or 8 and a second wave");
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_cptr)smem));

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave / WN, wn = wave % WN;
  const int D = p.D, F = p.F;
  const int Kdim = (MODE == RM_GATEUP || DH_LIKE) ? D : (MODE == RM_DOWN ? F : 2 * F);
  const int lda = (MODE == RM_GATEUP || DH_LIKE) ? D : F;
  const int Ncols = (MODE == RM_GATEUP || DH_LIKE) ? F : D;  // output width
  const int64_t wsz = static_cast<int64_t>(D) * F;
  const int ksteps = Kdim / BK;

  // Persistent workgroups: block b serves XCD b % 8 and walks that XCD's contiguous run
  // of the tile list with stride gridDim/8, the order in which the hardware dispatcher
  // would have started one-tile blocks.  Tile metadata is looked up two tiles ahead.
  const int total = (SHORT ? tiles.total : *p.num_tiles) * p.n_tiles;
  const int chunk = (total + 7) >> 3;
  const int stride = gridDim.x >> 3;
  const int pid_base = (blockIdx.x & 7) * chunk;
  int within = blockIdx.x >> 3;
  if (within >= chunk || pid_base + within >= total) return;
  auto exists = [&](int w) { return w < chunk && pid_base + w < total; };
  auto load_meta = [&](int w) -> TileMeta {
    const int pid = pid_base + w;
    // scalar loads (constant address space): as vector loads these lookups would share the
    // counter of the operand stream and of the epilogue stores, and waiting for one of them
    // would wait for all of those
    const int t = quotient(pid, p.by_n_tiles);  // some tile of the expert this work item belongs to
    TileMeta m;
    [[maybe_unused]] int before = 0;
    m.e = SHORT ? tiles.expert(t, before) : ((const_i32)p.tile_expert)[t];
    const int cnt_e = ((const_i32)p.seg_counts)[m.e], off_e = ((const_i32)p.seg_offsets)[m.e];
    const int nrt = max((cnt_e + TBM - 1) / TBM, 1);  // row tiles of the expert
    const bool few = nrt <= 3;
    // (even_tile_rows, up to three tiles without a division)
    const int h = nrt == 1 ? TBM : few ? ((nrt == 2 ? (cnt_e + 1) >> 1 : third(cnt_e + 2)) + 15) & ~15 : even_tile_rows(cnt_e, TBM);
    // Within an expert the work items run column-tile-major over groups of three row tiles:
    // the row tiles of one column tile are neighbours, so the weight tile they share -- the
    // larger operand: an expert's weights are several times its rows -- is in L2 when the next
    // one asks for it, and a row tile's column tiles are still at most 3 x n_tiles work items
    // apart, inside what an XCD has in flight.  Row-tile-major throughout (neighbours share
    // the row tile only) left a quarter of the weight tiles to be fetched twice;
    // column-tile-major throughout fetches the rows of an expert with many row tiles once per
    // column tile.
    constexpr int G = 3;
    int t0 = before;  // the expert's first tile
    if constexpr (!SHORT) {
      const int above = ((const_i32)p.tile_row0)[t] - off_e;
      t0 = t - (few ? (above >= h) + (above >= 2 * h) : above / h);
    }
    const int q = pid - t0 * p.n_tiles;
    const int blk = few ? 0 : quotient(q, p.by_n_tiles) / G;
    const int qb = q - blk * (G * p.n_tiles);
    const int g = min(G, nrt - blk * G);  // row tiles of this group (>= 1)
    const int nt = g == 1 ? qb : g == 2 ? qb >> 1 : third(qb), rt = blk * G + (qb - nt * g);
    m.row0 = off_e + rt * h;
    m.valid = min(h, cnt_e - rt * h);
    // a last tile that would overhang starts early instead and recomputes a few columns
    // of its neighbour (same values), so no column is ever clamped
    constexpr int W = (MODE == RM_GATEUP ? BNT / 2 : BNT);
    m.n0 = min(nt * W, Ncols - W);
    m.nt = nt;
    m.stream = p.stream && nrt == 1;
    m.k_start = 0;
    if constexpr (TURN) {
      m.k_start = 5 * m.e + (cnt_e <= 256 && Ncols % W == 0 ? 3 * nt : 0);
      m.k_start -= quotient(m.k_start, p.by_steps) * ksteps;
    }
    return m;
  };

  // ---- operand requests: 1 KiB a wave and instruction, straight into LDS --------------------
  const int ldb = B_KS ? Ncols : (MODE == RM_GATEUP ? D : F);
  const int kc_row = 8 * wave + (lane >> 3);
  const int kc_chunk = (lane & 7) ^ ((kc_row >> 1) & 7);
  uint32_t voffB;
  if constexpr (!B_KS) {
    voffB = static_cast<uint32_t>(kc_row * ldb + kc_chunk * 8) * 2u;
  } else {
    constexpr int CPR = BNT / 8;  // 16-byte chunks per k row
    const int k = (64 / CPR) * wave + lane / CPR, cc = (lane % CPR) ^ ks_key16(k);
    voffB = static_cast<uint32_t>(k * ldb + cc * 8) * 2u;
  }
  // state of the tile whose operands are being requested
  uint64_t gA0, gA1, gB0, gB1;  // A rows (k = 0), DX: second half of the contraction (dup); the B tile's origin in both weight stacks
  uint32_t voffA[NA];
  int k_start = 0, fk = 0;
  auto setup = [&](const TileMeta& m, const int (&asrc)[NA]) {
    const int64_t arow = GATHER ? 0 : static_cast<int64_t>(m.row0) * lda;
    gA0 = reinterpret_cast<uint64_t>(p.a0 + arow);
    gA1 = (MODE == RM_DX) ? reinterpret_cast<uint64_t>(p.a1 + arow) : gA0;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int src = GATHER ? min(max(asrc[i], 0), p.a_rows - 1) : asrc[i];
      voffA[i] = (static_cast<uint32_t>(src) * static_cast<uint32_t>(lda) + static_cast<uint32_t>(kc_chunk * 8)) * 2u;
      // (dH's stay copies: as zeros 79.3 us instead of 78.7 for 700 dense rows of 7168 x 2048, 34.1 instead of 33.7 for 2000 of 2048 x 2048, nothing between 60 and 520 rows an expert)
      if (MODE != RM_DH && kc_row + 64 * i >= m.valid) voffA[i] = kNoRow;
    }
    // KC: the tile's first weight row is n0; KS: its first column is n0
    const int64_t borg = m.e * wsz + (B_KS ? static_cast<int64_t>(m.n0) : static_cast<int64_t>(m.n0) * ldb);
    gB0 = reinterpret_cast<uint64_t>(p.b0 + borg);
    gB1 = (MODE == RM_GATEUP || MODE == RM_DX) ? reinterpret_cast<uint64_t>(p.b1 + borg) : gB0;
    k_start = m.k_start;
    fk = 0;
  };
  // rows past the tile's last: past the end of the buffer that a request names, which makes them zeros and reads nothing; dH: the last row again
  auto tile_row = [&](const TileMeta& m, int i) { return max(min(kc_row + 64 * i, m.valid - 1), 0); };
  auto kofs = [&]() {
    if constexpr (!TURN) return fk * BK;
    const int ks = fk + k_start;
    return (ks < ksteps ? ks : ks - ksteps) * BK;
  };
  uint32_t fst = 0;  // LDS stage (byte offset) the requests go to
  [[maybe_unused]] uint32_t rst = 0;  // ... and, of three, the one that is read
  const uint32_t wdst = lds0 + wave * 1024u;
  auto req_a = [&](int i) {
    int k0 = kofs();
    uint64_t g = gA0;
    if constexpr (MODE == RM_DX) {
      if (k0 >= F) { k0 -= F; g = gA1; }
    }
    lds_load16<false, kNoRow>(g, voffA[i], k0 * 2, fst + wdst + i * 8192u);
  };
  auto req_b = [&](int i, auto stream) {
    int k0 = kofs();
    uint64_t g = gB0;
    uint32_t so;
    if constexpr (MODE == RM_GATEUP) {
      // rows 0..BNT/2 of the tile come from w1, the rest from w3, same f range
      if (i >= NB / 2) g = gB1;
      so = (64 * (i % (NB / 2)) * ldb + k0) * 2;
    } else if constexpr (MODE == RM_DOWN) {
      so = (64 * i * ldb + k0) * 2;
    } else {
      if constexpr (MODE == RM_DX) {
        if (k0 >= F) { k0 -= F; g = gB1; }
      }
      so = (k0 + i * (BK / NB)) * ldb * 2;
    }
    const uint32_t dst = fst + wdst + A_BYTES + i * 8192u;
    if (stream) lds_load16<true>(g, voffB, so, dst);
    else lds_load16(g, voffB, so, dst);
  };
  // the pieces of B in the order of the halves
  auto b_piece = [](int h, int j) { return MODE == RM_DOWN && NBX ? h + 2 * j : h * NBX + j; };
  auto req_x = [&](int i, auto stream) {
    if (i < NA) req_a(i);
    else req_b(b_piece(0, i - NA), stream);
  };
  auto req_y = [&](int j, auto stream) { req_b(b_piece(1, j), stream); };
  auto next_stage = [](uint32_t& st) {
    if constexpr (SHORT) st = st == 2 * STAGE_BYTES ? 0 : st + STAGE_BYTES;
    else st ^= STAGE_BYTES;
  };
  auto issue = [&](const TileMeta& cur) {
#pragma unroll
    for (int i = 0; i < NA + NBX; ++i) req_x(i, cur.stream);
#pragma unroll
    for (int j = 0; j < NBY; ++j) req_y(j, cur.stream);
    next_stage(fst);
    ++fk;
  };

  // ---- fragment reads ------------------------------------------------------------------------
  const int l15 = lane & 15, l4 = lane >> 4;
  const uint32_t cpos = static_cast<uint32_t>((l4 ^ (l15 >> 1)) * 16);  // k 0..31; k 32..63: ^ 64
  uint32_t ra = lds0 + (16 * wr + l15) * 128u + cpos;
  uint32_t rb[B_KS ? 4 : 1];
  if constexpr (!B_KS) {
    rb[0] = lds0 + A_BYTES + (wn * (MODE == RM_GATEUP ? 16 * NJ : 32 * NJ) + l15) * 128u + cpos;
  } else {
    const int k = 8 * l4 + (l15 >> 2);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int c = wn * 4 * NJ + b * 2 + ((l15 & 3) >> 1);
      rb[b] = lds0 + A_BYTES + k * (BNT * 2u) + (c ^ ks_key16(k)) * 16u + (l15 & 1) * 8u;
    }
  }
  auto rd_a = [&](bf16x8 (&f)[4], int kk, int mi) { f[mi] = lds_read16((kk ? ra ^ 64u : ra) + mi * 8192u); };
  auto rd_b = [&](bf16x8 (&f)[NJ], int kk, int hb, int b) {
    if constexpr (!B_KS) {
      const uint32_t base = kk ? rb[0] ^ 64u : rb[0];
      f[b] = lds_read16(base + (MODE == RM_GATEUP ? hb * (BNT / 2) * 128u + b * 2048u : (hb * NJ + b) * 2048u));
    } else {
      f[b] = lds_read_tr<BNT * 2>((NJ == 4 ? rb[b] ^ (hb * 128u) : rb[(hb * NJ + b) & 3]) + kk * 32u * (BNT * 2u));
    }
  };

  constexpr int NJ2 = 2 * NJ;
  f32x4 acc[MB][NJ2];

  TileMeta cur = load_meta(within);
  // the wave's own 4 KiB for its results: of a third stage's, the one that the next tile's first step will request
  uint32_t epi = 2 * STAGE_BYTES + wave * 4096u;
  const uint32_t idx_at = SHORT ? 3 * STAGE_BYTES + wave * 256u : epi;  // ... 256 bytes for the next tile's row indices
  {
    int asrc[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int r = tile_row(cur, i);
      asrc[i] = GATHER ? p.a_src[cur.row0 + r] : r;
    }
    setup(cur, asrc);
    issue(cur);
    issue(cur);
  }
  // (looked up with the first operands under way, not in front of them)
  TileMeta nxt = load_meta(exists(within + stride) ? within + stride : within);
  lds_sync<VM_EPI>();

  for (;;) {
  const bool more = exists(within + stride);
  const int row0 = cur.row0, valid = cur.valid, n0 = cur.n0, ntile = cur.nt;
  if constexpr (GATHER) {
    // the next tile's row indices into the wave's own LDS: lane 8 i + r has that of row r of its i-th piece
    const int ol = opaque(lane), r = max(min(8 * wave + (ol & 7) + 64 * ((ol >> 3) & 3), nxt.valid - 1), 0);
    lds_load4(reinterpret_cast<uint64_t>(p.a_src + nxt.row0), r * 4u, 0, lds0 + idx_at);
  }

#pragma unroll
  for (int mi = 0; mi < MB; ++mi)
#pragma unroll
    for (int nj = 0; nj < NJ2; ++nj)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[mi][nj][i] = 0.0f;

  // The tile's 16-row blocks are dealt to the four wave rows in turn, so that a tile that is not full keeps all waves
  // equally busy; the K loop is instantiated for the number of blocks a wave has.
  const int act = min(max(((valid + 15) >> 4) - wr + 3, 0) >> 2, MB);
  auto next_tile = [&]() {
    if (more) {
      int asrc[NA];
#pragma unroll
      for (int i = 0; i < NA; ++i)
        asrc[i] = GATHER ? lds_read_i32(lds0 + idx_at + (8 * i + (opaque(lane) >> 3)) * 4) : tile_row(nxt, i);
      setup(nxt, asrc);
    } else {
      fk = 0;
    }
  };
  [[maybe_unused]] auto k_loop = [&](auto act_t, auto stream) {
    constexpr int ACT = decltype(act_t)::value;
    // A quarter of a K step's MFMAs; what else the quarter holds -- requests of the K step after the next, fragment reads of the
    // next quarter -- goes out between its 16-row blocks, where the matrix core is busy with the block before.
    auto mm = [&](const bf16x8 (&af)[4], const bf16x8 (&bf)[NJ], int hb, auto between) {
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        __builtin_amdgcn_sched_barrier(0);
        between(mi);
        __builtin_amdgcn_sched_barrier(0);
        if (mi < ACT) {
#pragma unroll
          for (int b = 0; b < NJ; ++b)
            acc[mi][hb * NJ + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[b], af[mi], acc[mi][hb * NJ + b], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    bf16x8 a0[4], a1[4], b0[NJ], b1[NJ];
#pragma unroll
    for (int i = 0; i < ACT; ++i) rd_a(a0, 0, i);
#pragma unroll
    for (int b = 0; b < NJ; ++b) rd_b(b0, 0, 0, b);
    for (int ks = 0; ks < ksteps; ++ks) {
      if (ks == ksteps - 2) next_tile();
      // contraction contiguous: first columns k 0-31, k 32-63, last columns likewise; strided: k 0-31 first and last columns, k 32-63 likewise
      mm(a0, b0, 0, [&](int q) {
        if (q < ACT) rd_a(a1, 1, q);
        if (q < NJ) rd_b(b1, B_KS ? 0 : 1, B_KS ? 1 : 0, q);
      });
      if (NBX > 0 && ks > 0) lds_wait<VM>();
      lds_sync<63>();
      mm(B_KS ? a0 : a1, b1, B_KS ? 1 : 0, [&](int q) {
        if (q == 0) return;
        req_x(q - 1, stream);
#pragma unroll
        for (int b = (q - 1) * 2; b < q * 2 && b < NJ; ++b) rd_b(b0, B_KS ? 1 : 0, B_KS ? 0 : 1, b);
      });
      mm(B_KS ? a1 : a0, b0, B_KS ? 0 : 1, [&](int q) {
        if (q + 3 < NA + NBX) req_x(q + 3, stream);
#pragma unroll
        for (int b = q * 2; b < q * 2 + 2 && b < NJ; ++b) rd_b(b1, 1, 1, b);
      });
      if (ks > 0) lds_wait<VM>();
      lds_sync<63>();
      ra ^= STAGE_BYTES;
#pragma unroll
      for (int b = 0; b < (B_KS ? 4 : 1); ++b) rb[b] ^= STAGE_BYTES;
      mm(a1, b1, 1, [&](int q) {
        if (q == 0) return;
        if (q - 1 < NBY) req_y(q - 1, stream);
#pragma unroll
        for (int i = (q - 1) * 2; i < q * 2 && i < 4; ++i) {
          if (i < ACT) rd_a(a0, 0, i);
          if (i < NJ) rd_b(b0, 0, 0, i);
        }
      });
      fst ^= STAGE_BYTES;
      ++fk;
    }
  };
  [[maybe_unused]] auto k_loop_short = [&](auto act_t, auto stream) {
    constexpr int ACT = decltype(act_t)::value;
    // Half a K step's MFMAs: 32 k of the tile's columns, requests and the other half's fragment reads between its groups of four.
    auto mm = [&](const bf16x8 (&af)[2], const bf16x8 (&bf)[NJ2], auto between) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        __builtin_amdgcn_sched_barrier(0);
        between(q);
        __builtin_amdgcn_sched_barrier(0);
        if ((q & 1) < ACT) {
#pragma unroll
          for (int b = 0; b < NJ; ++b)
            acc[q & 1][(q >> 1) * NJ + b] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[(q >> 1) * NJ + b], af[q & 1], acc[q & 1][(q >> 1) * NJ + b], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    bf16x8 a0[2], a1[2], b0[NJ2], b1[NJ2];
    auto read = [&](bf16x8 (&a)[2], bf16x8 (&b)[NJ2], int kk, int q) {
      if (q < ACT) a[q] = lds_read16((kk ? ra ^ 64u : ra) + rst + q * 8192u);
#pragma unroll
      for (int j = 2 * q; j < 2 * q + 2; ++j) {
        if constexpr (!B_KS) {
          const uint32_t base = (kk ? rb[0] ^ 64u : rb[0]) + rst;
          b[j] = lds_read16(base + (MODE == RM_GATEUP ? (j / NJ) * (BNT / 2) * 128u + (j % NJ) * 2048u : j * 2048u));
        } else {
          b[j] = lds_read_tr<BNT * 2>((rb[j % NJ] ^ ((j / NJ) * 128u)) + rst + kk * 32u * (BNT * 2u));
        }
      }
    };
    auto request = [&](int i) { i < NA + NBX ? req_x(i, stream) : req_y(i - NA - NBX, stream); };
    auto step = [&](int ks, auto first_t) {
      constexpr bool FIRST = decltype(first_t)::value;
      if (ks == ksteps - 2) next_tile();
      if constexpr (!FIRST) lds_wait<NA + NB>();
      lds_sync<63>();
      auto between = [&](int q) {
        read(a0, b0, 0, q);
        if (q > 0) request(q - 1);
      };
      if constexpr (FIRST) {
#pragma unroll
        for (int q = 0; q < 4; ++q) between(q);
      } else {
        mm(a1, b1, between);
      }
      mm(a0, b0, [&](int q) {
        read(a1, b1, 1, q);
        if (q < 3) request(q + 3);
      });
      next_stage(fst);
      next_stage(rst);
      ++fk;
    };
    step(0, std::true_type{});
    for (int ks = 1; ks < ksteps; ++ks) step(ks, std::false_type{});
    mm(a1, b1, [](int) {});
  };
  // (the hint is the tile's own, also for what its loop requests of the next tile; a branch at each request instead: top of this file)
  auto with_blocks = [&](auto stream) {
    if constexpr (SHORT) {
      switch (act) {
        case 0: k_loop_short(std::integral_constant<int, 0>{}, stream); break;
        case 1: k_loop_short(std::integral_constant<int, 1>{}, stream); break;
        default: k_loop_short(std::integral_constant<int, 2>{}, stream);
      }
    } else {
      switch (act) {
        case 0: k_loop(std::integral_constant<int, 0>{}, stream); break;
        case 1: k_loop(std::integral_constant<int, 1>{}, stream); break;
        case 2: k_loop(std::integral_constant<int, 2>{}, stream); break;
        case 3: k_loop(std::integral_constant<int, 3>{}, stream); break;
        default: k_loop(std::integral_constant<int, 4>{}, stream);
      }
    }
  };
  if (cur.stream) with_blocks(std::true_type{});
  else with_blocks(std::false_type{});
  if constexpr (SHORT) {
    lds_sync<63>();  // all waves have read the stage that the results go through
    epi = fst + wave * 4096u;
  }

  // the tile after the next: looked up here, where the next one's operands are waited for in any case, used one tile later
  TileMeta nxt2;
  auto look_up = [&]() { nxt2 = load_meta(exists(within + 2 * stride) ? within + 2 * stride : within); };
  if constexpr (MODE != RM_DH) look_up();

  // ---- epilogue: 16 rows at a time through the wave's own LDS, 16-byte coalesced rows ----
  // acc[mi][nj][i]: output row = wm + mi*16 + (lane&15); output column within the nj-th
  // 16-column tile = 4*(lane>>4) + i.
  const uint32_t el = opaque(lane);
  constexpr int CH = 4 * NJ;  // 16-byte chunks per row of the wave's sub-tile
  auto key = [](uint32_t m) { return CH == 16 ? m : m >> 1; };
  auto put = [&](int nj, u32x2 pk) {
    const uint32_t c = nj * 2 + ((el >> 4) >> 1);
    *reinterpret_cast<u32x2*>(reinterpret_cast<char*>(smem) + epi + (el & 15) * (CH * 16) + ((c ^ key((el & 15))) * 16) + ((el >> 4) & 1) * 8) = pk;
  };
  auto get = [&](uint32_t m, uint32_t c) {
    return *reinterpret_cast<const u32x4*>(reinterpret_cast<const char*>(smem) + epi + m * (CH * 16) + ((c ^ key(m)) * 16));
  };
  // The tile's rows of a matrix with rows of `pitch` bytes, as a buffer that ends behind the last of them: what a lane of the last 16-row block stores past them
  // is dropped and what it loads is zero, so that every access is unconditional and one addition forms its address.
  auto rows_of = [&](const auto* base, uint32_t pitch) {
    const char* first = reinterpret_cast<const char*>(base) + static_cast<int64_t>(row0) * pitch;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(first), 0, valid * pitch, 0x00020000);
  };
  auto store16 = [&](RowsOut to, uint32_t offset, u32x4 v) { __builtin_amdgcn_raw_buffer_store_b128(v, to, offset, 0, 0); };
  if constexpr (MODE == RM_GATEUP) {
    // 16 rows of gate and up side by side (16 NJ columns each), then of h in the same place
    constexpr int WC = 16 * NJ, CPT = WC / 8;  // columns and chunks of one of them
    const uint32_t pitch = F * 2u, at = (wr * 16 + el / CPT) * pitch + (n0 + wn * WC) * 2u + el % CPT * 16u;
    [[maybe_unused]] const RowsOut o0 = rows_of(p.o0, pitch), o1 = rows_of(p.o1, pitch);
    const RowsOut o2 = rows_of(p.o2, pitch);
    lds_wait<VM_EPI>();
#pragma unroll
    for (int mi = 0; mi < MB; ++mi) {
      if (mi >= act) continue;
#pragma unroll
      for (int part = SAVE_GU ? 0 : 1; part < 2; ++part) {
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          u32x2 g, u, h;
#pragma unroll
          for (int r = 0; r < 2; ++r) {
            float g0 = acc[mi][j][2 * r], g1 = acc[mi][j][2 * r + 1], u0 = acc[mi][j + NJ][2 * r], u1 = acc[mi][j + NJ][2 * r + 1];
            g[r] = round_bf16x2(g0, g1);
            u[r] = round_bf16x2(u0, u1);
            float s0 = g0 * fast_sigmoid(g0), s1 = g1 * fast_sigmoid(g1);
            round_bf16x2(s0, s1);
            h[r] = pack2(s0 * u0, s1 * u1);
          }
          if (part == 0) {
            put(j, g);
            put(NJ + j, u);
          } else {
            put(j, h);
          }
        }
        wave_lds_sync();
        // rows of one matrix, 64 / CPT an instruction
#pragma unroll
        for (int t = 0; t < (part == 0 ? 2 : 1); ++t)
#pragma unroll
          for (int it = 0; it < CPT / 4; ++it) {
            const uint32_t m = it * (64 / CPT) + el / CPT, c = el % CPT;
            store16(part == 1 ? o2 : t == 0 ? o0 : o1, at + (mi * 64 + it * (64 / CPT)) * pitch, get(m, t * CPT + c));
          }
        wave_lds_sync();
      }
    }
  } else if (act > 0) {
    const int c0 = n0 + wn * (32 * NJ);
    // 64 rows x CH chunks, CH per lane; a row's bytes go out contiguously; tiles never overhang in the columns.
    constexpr int IPB = CH / 4;  // 16-byte pieces a lane has of a block of 16 rows, 64 / CH rows apart
    const uint32_t pitch = Ncols * 2u, lrow = el / CH, lc = el % CH, at = (wr * 16 + lrow) * pitch + c0 * 2u + lc * 16u;
    auto offset_at = [&](int mi, int u) { return at + (mi * 64 + u * (64 / CH)) * pitch; };
    const RowsOut o0 = rows_of(p.o0, pitch);
    auto stage = [&](int mi) {
#pragma unroll
      for (int nj = 0; nj < NJ2; ++nj)
        put(nj, u32x2{pack2(acc[mi][nj][0], acc[mi][nj][1]), pack2(acc[mi][nj][2], acc[mi][nj][3])});
      wave_lds_sync();
    };
    if constexpr (MODE == RM_DH) {
      // SwiGLU backward on 8 consecutive f: dgate = dh*up*silu'(gate), dup = dh*silu(gate).
      // gate and up of the next 16 rows are requested before the current ones are stored:
      // a load issued behind a store cannot complete before it.
      // With the combine's backward folded in (FUSE), the staged value is the unscaled dh row:
      // its product with the row's h (recomputed from gate and up) summed over f is the
      // gradient of the row's routing score, reduced here over the 16 lanes that share a row
      // and written once per row and 128-column slot; dh itself is then scaled by the score,
      // and score * h goes out as the operand of the dW2 product.
      constexpr bool FUSE = GATHER;
      constexpr int G = IPB;
      [[maybe_unused]] float* dots = reinterpret_cast<float*>(reinterpret_cast<char*>(smem) + epi + 2048);
      u32x4 gq[G], uq[G];
      float sq = 1.0f;  // lane l: the score of the block's row l % 16
      const RowsOut o1 = rows_of(p.o1, pitch), in_gate = rows_of(p.gate, pitch), in_up = rows_of(p.up, pitch);
      [[maybe_unused]] const RowsOut o2 = FUSE ? rows_of(p.o2, pitch) : o0, scale = FUSE ? rows_of(p.row_scale, 4) : o0,
                                     slots = FUSE ? rows_of(p.dot_partial, p.dot_slots * 4u) : o0;
      auto request = [&](int mi, u32x4 (&g)[G], u32x4 (&u)[G], float& sc) {
#pragma unroll
        for (int i = 0; i < G; ++i) {
          const uint32_t o = offset_at(mi, i);
          g[i] = __builtin_amdgcn_raw_buffer_load_b128(in_gate, o, 0, 0);
          u[i] = __builtin_amdgcn_raw_buffer_load_b128(in_up, o, 0, 0);
        }
        if constexpr (FUSE) sc = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(scale, (mi * 64 + wr * 16 + (el & 15)) * 4u, 0, 0));
      };
      request(0, gq, uq, sq);
      look_up();
      lds_wait<2 * G>();  // (2 G requests and more are younger than the next tile's operands)
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        if (mi >= act) break;
        u32x4 gn[G], un[G];
        float sn;
        // (the last block again past it: every load is unconditional)
        if (mi < 3) request(min(mi + 1, act - 1), gn, un, sn);
        stage(mi);
#pragma unroll
        for (int u = 0; u < G; ++u) {
          const uint32_t m = u * (64 / CH) + lrow;
          const u32x4 v = get(m, lc);
          const u32x4 gv = gq[u], uv = uq[u];
          const float sc = FUSE ? __shfl(sq, m) : 1.0f;
          float dot = 0.0f;
          u32x4 dg, du, hs;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            float dh[2], uu[2], sl[2], slope[2], ds[2];
#pragma unroll
            for (int hlf = 0; hlf < 2; ++hlf) {
              dh[hlf] = __uint_as_float(hlf ? (v[w] & 0xffff0000u) : (v[w] << 16));
              const float g = __uint_as_float(hlf ? (gv[w] & 0xffff0000u) : (gv[w] << 16));
              uu[hlf] = __uint_as_float(hlf ? (uv[w] & 0xffff0000u) : (uv[w] << 16));
              const float sig = fast_sigmoid(g);
              sl[hlf] = g * sig;
              slope[hlf] = sig * (1.0f + g * (1.0f - sig));
            }
            round_bf16x2(sl[0], sl[1]);
            if constexpr (FUSE) {
              float hv[2] = {sl[0] * uu[0], sl[1] * uu[1]};
              round_bf16x2(hv[0], hv[1]);  // h as the forward stored it
#pragma unroll
              for (int hlf = 0; hlf < 2; ++hlf) {
                dot += dh[hlf] * hv[hlf];
                dh[hlf] *= sc;
              }
              hs[w] = pack2(sc * hv[0], sc * hv[1]);
            }
            ds[0] = dh[0] * uu[0], ds[1] = dh[1] * uu[1];
            round_bf16x2(ds[0], ds[1]);
            dg[w] = pack2(ds[0] * slope[0], ds[1] * slope[1]);
            du[w] = pack2(dh[0] * sl[0], dh[1] * sl[1]);
          }
          const uint32_t o = offset_at(mi, u);
          store16(o0, o, dg);
          store16(o1, o, du);
          if constexpr (FUSE) {
            store16(o2, o, hs);
            // columns below the tile's nominal start belong to its neighbour (a last tile
            // that would overhang starts early): they must not be counted twice
            if (c0 + static_cast<int>(lc) * 8 < ntile * BNT) dot = 0.0f;
            const float total = row16_sum<CH>(dot);
            // all 16 lanes of the row store the same value to the same address (unconditional,
            // like every other access of this epilogue); of a narrow tile, whose 128 columns are two waves', to LDS
            if constexpr (NJ == 4)
              __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(total), slots, ((mi * 64 + wr * 16 + m) * p.dot_slots + ntile * WN + wn) * 4u, 0, 0);
            else dots[mi * 16 + m] = total;
          }
        }
        wave_lds_sync();
        if (mi < 3) {
#pragma unroll
          for (int u = 0; u < G; ++u) {
            gq[u] = gn[u];
            uq[u] = un[u];
          }
          if constexpr (FUSE) sq = sn;
        }
      }
    } else {
      lds_wait<VM_EPI>();
#pragma unroll
      for (int mi = 0; mi < MB; ++mi) {
        if (mi < act) {
          stage(mi);
#pragma unroll
          for (int u = 0; u < IPB; ++u) store16(o0, offset_at(mi, u), get(u * (64 / CH) + lrow, lc));
        }
        wave_lds_sync();
      }
    }
  } else {
    if constexpr (MODE == RM_DH) look_up();
    lds_wait<VM_EPI>();
  }
  if constexpr (MODE == RM_DH && GATHER && NJ == 2) {
    // a narrow tile's slot: both waves' sums; the slots past the last tile's, which a wide tile would have filled, are zero
    lds_sync<63>();
    const int m = static_cast<int>((el >> 4) * 64 + wr * 16 + (el & 15));  // of the tile
    if (wn == 0 && m < valid) {
      const float* dots = reinterpret_cast<const float*>(reinterpret_cast<const char*>(smem) + epi + 2048);
      const float* other = dots + 1024;
      float* slot = p.dot_partial + static_cast<int64_t>(row0 + m) * p.dot_slots;
      slot[ntile] = dots[el] + other[el];
      if (ntile == p.n_tiles - 1)
        for (int i = p.n_tiles; i < p.dot_slots; ++i) slot[i] = 0.0f;
    }
  }
  if (!more) break;
  within += stride;
  cur = nxt;
  nxt = nxt2;
  }
  lds_wait<0>();
}

// Short tiles, of up to 128 rows with three stages of operands, where most experts have no more rows, so that the product is a read of their weights: a step's
// requests then go out two whole steps ahead and behind one barrier.  A plain read in this pattern has 6.1 TB/s with two stages of 32 KiB and 7.0 with three; with
// the rows and their results beside it, us, 256-row tiles / these, of Poisson loads from memory: 128 experts of 2048 x 768, 40 rows each gate/up 146 / 142, down
// 82 / 79; 62 rows 147 / 144, 87 / 83; 100 rows 152 / 149, 92 / 89; 32 of 7168 x 2048, 60 rows 311 / 303, 176 / 173, 347 / 341; 100
// rows 323 / 316, 182 / 178, 361 / 360; 60 of 1728 x 960, 60 and 100 rows gate/up 83 / 80, 88 / 85, down 45 / 44, 48 / 47, dRows 80 / 77, 85 / 82.  The same bits.
//   Not where the tiles are more by a quarter, or need a round of workgroups more (115 rows of the first, one expert in nine above 128: gate/up 156 / 182, dRows
// 155 / 171); not where the weights stay in the memory-side cache (64 experts of 1024 x 512, 100 rows: dRows 31 / 37); not dH, whose epilogue's loads
// wait for what has been requested before them: 160 / 163; not dRows where weight rows lie a multiple of 4 KiB apart (20 rows of the first 130 / 134, 62 rows 146 / 146).  A forward
// of 1000 tokens of the first, eight each, 257 / 252.
//   Uneven loads: of 430 products (128 of 2048 x 768 and 1344 x 704, 64 of 2048 x 1408, 60 of 1728 x 960 and 1920 x 704, 32 of 7168 x 2048; 25 to 110 rows an expert drawn evenly, by Zipf's
// laws of 0.3 to 1.2, all from a half, a quarter or 16 of the experts, and 30 or 60 rows each beside one to six experts of 300 to 2000) that choose these, three take 1 % to 1.5 % longer than
// on 256-row tiles (32 of 7168 x 2048, 60 rows beside one of 2000, gate/up 396 / 402), the median 4.5 % less and the best 15 %.
template <int MODE, int NJ, bool GATHER, bool SAVE_GU = true, bool TURN = false>
__global__ __launch_bounds__(NT, 2) void row_tiled_kernel(RowArgs p) {
  ShortTiles tiles;
  if constexpr (NJ == 4 && (MODE == RM_GATEUP || MODE == RM_DOWN || MODE == RM_DX)) {
    if (p.short_tiles) {
      tiles.find(p);
      if (short_tiles_serve(tiles.total, tiles.whole, *(const_i32)p.num_tiles, p.n_tiles, static_cast<int>(gridDim.x))) {
        row_tiles<MODE, NJ, GATHER, SAVE_GU, TURN, 2>(p, tiles);
        return;
      }
    }
  }
  row_tiles<MODE, NJ, GATHER, SAVE_GU, TURN, 4>(p, tiles);
}

// ---- weight gradients: C[e](M,N) = sum_{r in segment e} A[r][m] * B[r][n] ----------
// 256 x 256 output tile, 8 waves as 4 (m) x 2 (n), each wave 64 x 128; both operands KS.
constexpr int WBM = 256, WBN = 256;

struct WgradArgs {
  const uint16_t* a;  // (rows, M) row-major
  const uint16_t* b;  // (rows, N) row-major
  uint16_t* c;        // (El, M, N)
  const int32_t* a_src;  // row -> row of a to read, or null (GATHER_A)
  const int32_t* b_src;  // row -> row of b to read (token gather), or null
  int src_rows;          // rows of the gathered operand: indices are clamped to [0, src_rows)
  const int32_t* seg_offsets;
  const int32_t* seg_counts;  // (2 El): row counts, then the local experts by descending count
  int El;
  int M, N;
  int m_tiles, n_tiles;
  Divisor by_tiles, by_n_tiles;  // m_tiles * n_tiles; n_tiles
  int total;  // El * m_tiles * n_tiles
  const uint16_t* a1;  // null, or the first operand of another product with the same b, and its result
  uint16_t* c1;
};

template <bool GATHER, bool GATHER_A = false>
__global__ __launch_bounds__(NT, 2) void wgrad_kernel(WgradArgs p) {
  constexpr int PITCH = 512;  // bytes of an operand's k row in LDS
  constexpr bool INDEXED = GATHER || GATHER_A;
  constexpr int VM = 8;       // requests younger than those a barrier of the loop waits for: two groups of four
  constexpr int VMY = VM + INDEXED;  // ... and, at the second barrier, the row indices
  constexpr int STORES = 16;  // of a tile's results, a lane
  extern __shared__ __attribute__((aligned(16))) uint16_t smem[];
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_cptr)smem));
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wave >> 1, wn = wave & 1;
  const int M = p.M, N = p.N;
  const int per_e = p.m_tiles * p.n_tiles;
  const int pair = p.c1 != nullptr ? 1 : 0;  // two products of the same b: their tiles in turn

  // Persistent workgroups.  A tile's cost is its expert's row count (the contraction
  // length), which a skewed router spreads over two orders of magnitude, so tiles are not
  // walked in expert order: experts are taken by descending row count (the plan's order,
  // second half of seg_counts) and dealt to the eight XCDs a round at a time, and the CUs of an
  // XCD deal that XCD's tiles round-robin among themselves -- the longest contractions
  // start first and in parallel, and an expert's tiles still share one L2.
  const int El = p.El;
  const int xcd = blockIdx.x & 7;
  // The plan arrays are read-only here and every lookup is workgroup-uniform: read through
  // the constant address space they are scalar loads.  As vector loads (what the compiler
  // makes of them inside this loop) each lookup would share the counter of the operand
  // stream and of the epilogue stores, and waiting for it would wait for all of those.
  const const_i32 order = (const_i32)(p.seg_counts + El);
  const const_i32 seg_offsets = (const_i32)p.seg_offsets;
  const const_i32 seg_counts = (const_i32)p.seg_counts;
  // Whole experts are dealt in rounds of eight, each round in the opposite direction of the
  // one before (so no XCD always gets the larger expert of its round); the El % 8 smallest
  // experts left over are cut into eight equal contiguous runs of tiles instead.
  const int n_full = (El >> 3) * per_e;
  const int pool = (El & 7) * per_e;
  const int p0 = static_cast<int>(static_cast<int64_t>(pool) * xcd >> 3);
  const int p1 = static_cast<int>(static_cast<int64_t>(pool) * (xcd + 1) >> 3);
  const int n_x = (n_full + (p1 - p0)) << pair;  // tiles of this XCD
  const int stride = gridDim.x >> 3;
  int within = blockIdx.x >> 3;
  if (within >= n_x) return;
  auto exists = [&](int w) { return w < n_x; };
  struct Tile {
    int e, seg0, cnt, m0, n0, second;
  };
  // this XCD's w-th tile (w clamped to an existing tile): the rank of its expert, and its tile in the expert
  auto place = [&](int w, int& rank) -> int {
    w = (exists(w) ? w : within) >> pair;
    const bool full = w < n_full;
    const int u = full ? w : p0 + (w - n_full), r = quotient(u, p.by_tiles);
    rank = full ? r * 8 + ((r & 1) ? 7 - xcd : xcd) : (El & ~7) + r;
    return u - r * per_e;
  };
  // (clamped: an order array the caller never filled must not turn into a wild address)
  auto expert_at = [&](int w) -> int {
    int rank;
    place(w, rank);
    return min(max(order[rank], 0), El - 1);
  };
  // a last tile that would overhang starts early instead (M, N >= 256) and recomputes a few
  // rows or columns of its neighbour -- the same values -- so every tile is whole
  auto tile_at = [&](int w, int e) -> Tile {
    int rank;
    const int t = place(w, rank), m = quotient(t, p.by_n_tiles);
    return {e, seg_offsets[e], seg_counts[e], min(m * WBM, M - WBM), min((t - m * p.n_tiles) * WBN, N - WBN), (exists(w) ? w : within) & pair};
  };
  // (field by field: a choice between the structures would leave them in memory)
  auto either = [](bool c, Tile a, Tile b) -> Tile {
    return {c ? a.e : b.e, c ? a.seg0 : b.seg0, c ? a.cnt : b.cnt, c ? a.m0 : b.m0, c ? a.n0 : b.n0, c ? a.second : b.second};
  };
  Tile t0 = tile_at(within, expert_at(within));

  // ---- operand requests: two k rows of 256 columns a wave and instruction, straight into LDS ----
  const int krow = 2 * wave + (lane >> 5);
  const uint32_t cc16 = static_cast<uint32_t>((lane & 31) ^ ks_key16(krow)) * 16u;
  const uint32_t voffA = GATHER_A ? cc16 : static_cast<uint32_t>(krow * M) * 2u + cc16;
  const uint32_t voffB = GATHER ? cc16 : static_cast<uint32_t>(krow * N) * 2u + cc16;
  const uint32_t wdst = lds0 + wave * 1024u;
  uint32_t fst = 0;  // LDS stage (byte offset) the requests go to
  // State of the K step whose operands are being requested, kept up by additions (scalar arithmetic between the MFMAs is what this loop has least room
  // for): how many tiles ahead, rows of the segment from this step on, operand addresses and bytes to the segment's end
  int ahead = 0, left;
  uint64_t gA, gB;
  uint32_t bytesA, bytesB;
  [[maybe_unused]] uint32_t voffG[4];  // where the lane's pieces of the gathered operand lie
  // The same for its row indices, which are requested a K step earlier still: all 64 of a step into one of four 256-byte places of the wave's own LDS, which its results
  // go through too: what has been requested is in registers by then
  [[maybe_unused]] int i_ahead = 0, i_left = 0;
  [[maybe_unused]] uint64_t ix = 0;
  [[maybe_unused]] uint32_t i_to = 0, i_from = 0;
  const uint32_t epi = 2 * STAGE_BYTES + wave * 4096u;
  const uint32_t ldA = static_cast<uint32_t>(M) * 2u, ldB = static_cast<uint32_t>(N) * 2u;  // bytes
  // bytes of the gathered operand; an offset past them for rows past the segment (whole 128-byte lines below 4 GiB: no operand has it, nor has one from a later column on)
  const uint64_t src_bytes = static_cast<uint64_t>(p.src_rows) * (GATHER ? ldB : ldA);
  constexpr uint32_t kNowhere = 0xffffff80u;
  int fm0, fn0;
  auto set_bytes = [&]() {
    // (a step of 64 rows ends before the next row's first column)
    const uint32_t rows = static_cast<uint32_t>(min(max(left, 0), BK));
    if constexpr (!GATHER_A) bytesA = rows ? rows * ldA - fm0 * 2u : 0u;
    if constexpr (!GATHER) bytesB = rows ? rows * ldB - fn0 * 2u : 0u;
  };
  auto request_indices = [&]() {
    if constexpr (INDEXED) {
      lds_load4_within(ix, static_cast<uint32_t>(max(i_left, 0)) * 4u, opaque(lane) * 4u, lds0 + epi + i_to);
      i_to = (i_to + 256) & 1023;
    }
  };
  auto indices_of = [&](Tile t) {
    if constexpr (INDEXED) {
      i_left = t.cnt;
      ix = reinterpret_cast<uint64_t>((GATHER ? p.b_src : p.a_src) + t.seg0);
    }
  };
  auto to_tile = [&](Tile t) {
    left = t.cnt;
    fm0 = t.m0;
    fn0 = t.n0;
    gA = reinterpret_cast<uint64_t>((t.second ? p.a1 : p.a) + (GATHER_A ? 0 : static_cast<int64_t>(t.seg0) * M) + t.m0);
    gB = reinterpret_cast<uint64_t>(p.b + (GATHER ? 0 : static_cast<int64_t>(t.seg0) * N) + t.n0);
    if constexpr (GATHER_A) bytesA = static_cast<uint32_t>(src_bytes - t.m0 * 2u);
    if constexpr (GATHER) bytesB = static_cast<uint32_t>(src_bytes - t.n0 * 2u);
  };
  auto read_indices = [&]() {
    if constexpr (INDEXED) {
      const uint32_t at = lds0 + epi + i_from + (2 * wave + (opaque(lane) >> 5)) * 4u;
#pragma unroll
      for (int i = 0; i < 4; ++i) voffG[i] = lds_read_i32(at + 64 * i);
      i_from = (i_from + 256) & 1023;
    }
  };
  auto take_row = [&](int i) {
    if constexpr (INDEXED) {
      // (rows and bytes of a row of a matrix below 4 GiB of 768 bytes a row or more both have 24 bits)
      const int r = min(max(static_cast<int>(voffG[i]), 0), p.src_rows - 1);
      const uint32_t at = __umul24(static_cast<uint32_t>(r), GATHER ? ldB : ldA) + cc16;
      voffG[i] = krow < left - 16 * i ? at : kNowhere;
    }
  };
  auto req = [&](bool is_a, int i) {
    const uint32_t dst = fst + wdst + (is_a ? 0u : A_BYTES) + i * 8192u;
    const uint32_t voff = (is_a ? GATHER_A : GATHER) ? voffG[i] : opaque(is_a ? voffA : voffB) + 16u * i * (is_a ? ldA : ldB);
    lds_load16_within(is_a ? gA : gB, is_a ? bytesA : bytesB, voff, dst);
  };
  // pieces 0 and 1 of both operands hold a K step's first 32 k, 2 and 3 the others
  auto req_q = [&](int half, int j) { req(j < 2, 2 * half + (j & 1)); };
  // The tiles after the first, the expert of the one after those.  Requests run two K steps ahead, their row indices three: of as many tiles
  // where each has one K step.  (Looked up once the first tile's operands are on their way, where it has enough steps.)
  Tile t1 = t0, t2 = t0, t3 = t0;
  auto next_step = [&]() {
    fst ^= STAGE_BYTES;
    left -= BK;
    if (left > 0) {
      if constexpr (!GATHER_A) gA += BK * static_cast<uint64_t>(ldA);
      if constexpr (!GATHER) gB += BK * static_cast<uint64_t>(ldB);
    } else {
      ++ahead;
      to_tile(either(ahead == 1, t1, either(ahead == 2, t2, t3)));
    }
    set_bytes();
  };
  auto next_indices = [&]() {
    if constexpr (INDEXED) {
      i_left -= BK;
      if (i_left > 0) {
        ix += BK * 4;
      } else {
        ++i_ahead;
        indices_of(either(i_ahead == 1, t1, either(i_ahead == 2, t2, t3)));
      }
      request_indices();
    }
  };
  auto req_all = [&]() {
    if constexpr (INDEXED) {
      read_indices();
#pragma unroll
      for (int i = 0; i < 4; ++i) take_row(i);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) req_q(j >> 2, j & 3);
    next_step();
  };
  to_tile(t0);
  indices_of(t0);
  set_bytes();
  request_indices();
  const bool early = t0.cnt > 2 * BK;
  if (early) {
    next_indices();
    if constexpr (INDEXED) lds_wait<0>();
    req_all();
    req_all();
  }
  t1 = tile_at(within + stride, expert_at(within + stride));
  t2 = tile_at(within + 2 * stride, expert_at(within + 2 * stride));
  t3 = tile_at(within + 3 * stride, expert_at(within + 3 * stride));
  int e4 = expert_at(within + 4 * stride);
  if (!early) {
    next_indices();
    if constexpr (INDEXED) lds_wait<0>();
    req_all();
    req_all();
  }
  next_indices();

  // ---- fragment reads ------------------------------------------------------------------------
  const int l15 = lane & 15, l4 = lane >> 4;
  uint32_t ra[4], rb[4];
  {
    const int k = 8 * l4 + (l15 >> 2);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int x = b * 2 + ((l15 & 3) >> 1);
      ra[b] = lds0 + k * PITCH + ((wr * 8 + x) ^ ks_key16(k)) * 16u + (l15 & 1) * 8u;
      rb[b] = lds0 + A_BYTES + k * PITCH + ((wn * 16 + x) ^ ks_key16(k)) * 16u + (l15 & 1) * 8u;
    }
  }
  auto rd_a = [&](bf16x8 (&fr)[4], int kk, int mi) { fr[mi] = lds_read_tr<PITCH>(ra[mi] + kk * 32u * PITCH); };
  auto rd_b = [&](bf16x8 (&fr)[4], int kk, int hb, int b) { fr[b] = lds_read_tr<PITCH>((rb[b] ^ (hb * 128u)) + kk * 32u * PITCH); };

  lds_sync<INDEXED ? 0 : 4>();
  read_indices();
  bool first = true;
  for (;;) {
    const bool more = exists(within + stride);
    f32x4 acc[4][8];
    // a quarter of a K step's MFMAs, requests and fragment reads between its blocks, as in the row-tiled kernel
    // (ZERO: to nothing, not to the sum so far -- 128 registers set to zero are half a microsecond a tile)
    auto mm = [&](auto zero_t, const bf16x8 (&af)[4], const bf16x8 (&bf)[4], int hb, auto between) {
      constexpr bool ZERO = decltype(zero_t)::value;
#pragma unroll
      for (int mi = 0; mi < 4; ++mi) {
        __builtin_amdgcn_sched_barrier(0);
        between(mi);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int b = 0; b < 4; ++b)
          acc[mi][hb * 4 + b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[b], af[mi], ZERO ? f32x4{0, 0, 0, 0} : acc[mi][hb * 4 + b], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    bf16x8 a0[4], a1[4], b0[4], b1[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rd_a(a0, 0, i);
      rd_b(b0, 0, 0, i);
    }
    const int ksteps = max((t0.cnt + BK - 1) / BK, 1);  // (no rows: one step of zeros)
    auto kstep = [&](int ks, auto first_t) {
      constexpr bool FIRST = decltype(first_t)::value;
      using F_ = std::false_type;
      mm(first_t, a0, b0, 0, [&](int q) {
        rd_b(b1, 0, 1, q);
        if (q == 3 && INDEXED && !FIRST) {
          lds_wait<VM>();
          read_indices();
        }
      });
      // (the last tile's stores may still be under way in the first step and, up to its first barrier, the second)
      if constexpr (FIRST) {
        if (!first) lds_wait<VM + STORES>();
      } else {
        if (INDEXED || ks > 1 || first) lds_wait<VM>();
        else lds_wait<VM + STORES>();
      }
      lds_sync<63>();
      mm(first_t, a0, b1, 1, [&](int q) {
        rd_a(a1, 1, q);
        rd_b(b0, 1, 0, q);
        if (q == 0) return;
        take_row(q - 1);
        if (q == 1) next_indices();
        if (q == 3) take_row(3);
        req_q(0, q - 1);
      });
      mm(F_{}, a1, b0, 0, [&](int q) {
        rd_b(b1, 1, 1, q);
        if (q == 0) req_q(0, 3);
      });
      if constexpr (!FIRST) lds_wait<VMY>();
      else if (!first) lds_wait<VM + STORES>();
      lds_sync<63>();
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        ra[b] ^= STAGE_BYTES;
        rb[b] ^= STAGE_BYTES;
      }
      mm(F_{}, a1, b1, 1, [&](int q) {
        if (q == 0) return;
        rd_a(a0, 0, q - 1);
        rd_b(b0, 0, 0, q - 1);
        req_q(1, q - 1);
        if (q < 3) return;
        rd_a(a0, 0, 3);
        rd_b(b0, 0, 0, 3);
        req_q(1, 3);
        next_step();
      });
    };
    kstep(0, std::true_type{});
    for (int ks = 1; ks < ksteps; ++ks) kstep(ks, std::false_type{});

    // the tile's results, 16 rows at a time through the wave's own LDS
    const uint32_t el = opaque(lane);
    char* own = reinterpret_cast<char*>(smem) + epi;
    uint16_t* C = (t0.second ? p.c1 : p.c) + static_cast<int64_t>(t0.e) * M * N + static_cast<int64_t>(t0.m0 + wr * 64) * N + t0.n0 + wn * 128;
    const RowsOut results = __builtin_amdgcn_make_buffer_rsrc(C, 0, 0xffffffffu, 0x00020000);
    const uint32_t at = (el >> 4) * ldB + (el & 15) * 16u;
    if constexpr (INDEXED) {
      lds_wait<VM>();
      read_indices();
    }
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) {
#pragma unroll
      for (int nj = 0; nj < 8; ++nj) {
        const uint32_t m = el & 15, c = nj * 2 + (el >> 5);
        const u32x2 pk = {pack2(acc[mi][nj][0], acc[mi][nj][1]), pack2(acc[mi][nj][2], acc[mi][nj][3])};
        *reinterpret_cast<u32x2*>(own + m * 256 + ((c ^ m) * 16) + ((el >> 4) & 1) * 8) = pk;
      }
      wave_lds_sync();
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const uint32_t m = u * 4 + (el >> 4), c = el & 15;
        // (non-temporal: a weight gradient is several times the size of L2 and is read next by the
        // optimizer; written through the cache as ordinary stores, an expert's 30-60 MB of results push
        // its own operands out of L2 between two of its tiles -- with few rows per expert, where the
        // product is bound by these writes, the gathered rows were fetched from memory several times over)
        constexpr int kNonTemporal = 2;
        __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4*>(own + m * 256 + ((c ^ m) * 16)), results,
                                               at + (mi * 16 + u * 4) * ldB, 0, kNonTemporal);
      }
      wave_lds_sync();
    }
    if (!more) break;
    first = false;
    within += stride;
    t0 = t1;
    t1 = t2;
    t2 = t3;
    t3 = tile_at(within + 3 * stride, e4);
    e4 = expert_at(within + 4 * stride);
    --ahead;
    --i_ahead;
  }
  lds_wait<0>();
}

template <typename K>
int set_lds(K kernel, int bytes) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  return e == hipSuccess ? MI355_OK : fail(MI355_ELAUNCH, "hipFuncSetAttribute: %s", hipGetErrorString(e));
}

}  // namespace

// The MFMA path needs whole 64-wide K steps, 16-byte aligned rows, and outputs at least
// one tile wide (a last tile that would overhang is shifted back, never clamped).
int bf16_row_tile_m() { return 256; }

// ... and one expert's weight matrix below 2 GiB: operand loads address a tile with 32-bit byte offsets.
bool bf16_fast_path_ok(int64_t D, int64_t F) {
  return D % 64 == 0 && F % 64 == 0 && D >= 384 && F >= 384 && D * F < (1ll << 30);
}

enum { STAGE_GATEUP = 1, STAGE_DOWN = 2, STAGE_DH = 4, STAGE_DX = 8, STAGE_DW2 = 16, STAGE_DW1 = 32, STAGE_DW3 = 64, STAGE_BESIDE = 128 };

static unsigned round8(int64_t v) { return static_cast<unsigned>((v + 7) / 8 * 8); }

// One workgroup per CU (a workgroup takes the whole LDS), rounded to whole XCD rounds.
static unsigned resident_blocks() {
  static unsigned n = 0;
  if (n == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 8)
      cus = 256;
    n = static_cast<unsigned>(cus / 8 * 8);
  }
  return n;
}


// Pieces of `height` rows that a segment has, of a number of rows around the mean like the sum of independent draws.
static double pieces(double mean, double sd, int height) {
  if (sd == 0.0) return std::ceil(mean / height);
  double n = 1.0;
  for (int j = height; j < mean + 5.0 * sd; j += height) n += 0.5 * std::erfc((j + 0.5 - mean) / (sd * std::sqrt(2.0)));
  return n;
}

// Whether a product of El experts runs on 128-column tiles (`narrow_n` of them across) instead of 256-column ones (`wide_n`): where their rounds of
// workgroups, seven tenths as long, take less time.  The number of row tiles is that of loads spread like independent draws around the mean
// (experts of 256 rows on average have one tile and a half each); one expert's share of a wider router counts rows it does not get, which errs
// towards wide tiles.  A narrow tile's time over a wide one's, launch included, where both are one round: 0.60-0.73 mostly full, 0.68-0.83 partly; three rounds over two
// 0.85-0.92, four over two 1.02-1.3.  Of 450 products (gate/up, down, dH, dRows of 4 to 48 experts of 640 x 448 to 2048 x 768, 40 to 500 rows each) 269
// run on narrow tiles, two of them up to 17 % slower than on wide ones, the others up to 40 % faster, and 29 of the rest would gain.  (A rule of halves and three eighths of
// one round of evenly filled tiles had chosen 14 that lose and left 60.)
// One dense segment: the input gradient alone (the dH of 4096 rows x 2048 columns is 16 x 8 tiles).  It runs beside other products, and
// narrow gate/up and down tiles take CUs those would have had (one rank's share, 1000 tokens: 595 / 638).
static bool narrow(int mode, int64_t El, int64_t wide_n, int64_t narrow_n, int64_t tile_capacity) {
  const int64_t cus = resident_blocks();
  if (El == 1) return (mode == RM_DH || mode == RM_DLIN) && tile_capacity * wide_n * 4 <= cus * 3;
  const int64_t spare = std::max<int64_t>(tile_capacity - El - 1, 0);  // 256 rows each
  if (spare * wide_n > 4 * cus) return false;
  const double mean = (static_cast<double>(spare) + 0.5) * 256.0 / static_cast<double>(El), tiles = pieces(mean, std::sqrt(mean), 256);
  auto rounds = [&](int64_t n) { return std::ceil((tiles * static_cast<double>(El * n) - 0.5) / static_cast<double>(cus)); };
  return rounds(narrow_n) * 0.7 < rounds(wide_n);
}

// Whether experts with one row tile -- whose weights no other tile reads -- have them read with the non-temporal hint: where the three weight stacks do
// not stay in the 256 MB of memory-side cache from one product to the next, putting them there costs more than it can give back.  us, as ever / with the hint:
//   one product, 128 experts of 2048 x 768, 1000 tokens of eight: gate/up 165 / 150 (5.4 TB/s), down 93 / 86, dH 107 / 95, dRows 153 / 147; 32 of 7168 x
//   2048, nine rows each: 312 / 276 (6.8 TB/s), 170 / 149, 161 / 141, 336 / 299, 128 rows each 363 / 337, 203 / 184, 194 / 169, 387 / 369
//   block forward, then a training step, 24 / 80 / 180 rows an expert, time with the hint over without, by the stacks' size: 16 experts of 1024 x 512 (48 MiB) 1.08
//   1.07 1.08, 1.0-1.03; 16 of 2048 x 1024 (192) 1.11 1.12 1.12, 1.10 1.08 1.05; 60 of 1280 x 640 (281) 1.01 1.06 1.03, 1.04 1.01 0.99; 32 of 1792 x
//   1024 (336) 0.91 0.95 1.02, 1.0 1.01 1.01; 60 of 2048 x 512 (360) 0.92 0.95 0.99, 0.92 0.94 0.97; 128 of 1024 x 512 (384) 0.90 0.98 1.01, 0.96 0.92 0.92;
//   128 of 1024 x 1024 (768) 0.90 0.97 0.96, 0.94 0.84 0.93
// With two row tiles or more an expert, which share the weights in L2, the hint costs 2-8 % (8192 tokens of the first block, 16384 of a skewed router).
static bool streamed(int64_t El, int64_t D, int64_t F) { return El * D * F * 6 > (int64_t{320} << 20); }

// Whether a row product on wide tiles may choose short ones by the counts (of which the kernel's waves add up 256): where the weights come from memory.  dRows' weights are read
// in rows of the output's width, which the two stages wait less for where they lie a multiple of 4 KiB apart.
static bool short_tiles_may(int mode, int64_t El, int64_t D, int64_t F) {
  return streamed(El, D, F) && El > 1 && El <= 256 && !(mode == RM_DX && D % 2048 == 0);
}

// Workgroups of a gate/up product that runs beside the launches of a router (a shared expert's): a workgroup takes a CU whole until its list of tiles
// ends, so a product that holds every CU makes each of them wait (rank and plan, 12 and 11 us alone, took 195 and 63), and the routed experts, often a
// read of their weights, start when it has ended instead of running beside it.  An eighth of the CUs is enough to prevent that.  Block forward, us, all CUs / seven eighths /
// three quarters: one rank's share of 7168 x 256 experts x 2048 at 3600 tokens (240 tiles) 847 / 840 / 842, 4096 996 / 893 / 886, 4500 1044 / 1021 / 1030,
// 5500 (352) 1022 / 994 / 992; 64 experts of 2048 x 1408 and a shared one of twice that at 2600 tokens (242) 463 / 433 / 447; 32 of 1024 x 512, 8192 tokens
// 218 / 211 / 209.  Past one and a half rounds of workgroups, where the product is long beside the router: 7000 tokens of the share 1416 / 1439 on
// one box, 1401 / 1406 on another, 8192 1504 / 1529, 1482 / 1490, 5600 and 16384 of the second block 795 / 781 and 2000 / 2033.  The down projection starts behind the router: on fewer CUs nothing more, at some sizes 1-2 % slower.
static unsigned beside_router_blocks(int64_t tiles) {
  const unsigned n = resident_blocks();
  return n >= 64 && tiles * 2 <= 3 * static_cast<int64_t>(n) ? n / 64 * 56 : n;
}

// width: output columns; gate/up tiles hold both halves of their column range.  Tiles are
// 256 or 128 wide (a 192-wide KS tile would not hold the swizzle: 24 chunks per row are not a multiple
// of the 16 the key permutes); an overhanging last tile shifts back.
template <int MODE, bool GATHER = false, bool SAVE_GU = true, bool TURN = false>
static int launch_row(RowArgs& a, int64_t width, int64_t El, int64_t tile_capacity, hipStream_t s, const char* what,
                      bool beside = false) {
  constexpr int div = MODE == RM_GATEUP ? 2 : 1;
  a.stream = streamed(El, a.D, a.F);
  a.by_steps = divisor((MODE == RM_DOWN ? a.F : MODE == RM_DX ? 2 * static_cast<int64_t>(a.F) : a.D) / BK);
  a.El = (int)El;
  a.short_tiles = short_tiles_may(MODE, El, a.D, a.F);
  a.n_tiles = (int)((width + 256 / div - 1) / (256 / div));
  const int64_t narrow_n = (width + 128 / div - 1) / (128 / div);
  if (narrow(MODE, El, a.n_tiles, narrow_n, tile_capacity)) {
    a.n_tiles = (int)narrow_n;
    static PerDeviceOnce narrow_configured;
    if (narrow_configured.needed()) {
      if (int rc = set_lds(row_tiled_kernel<MODE, 2, GATHER, SAVE_GU, TURN>, R_LDS_BYTES)) return rc;
      narrow_configured.done();
    }
    a.by_n_tiles = divisor(a.n_tiles);
    const unsigned blocks = std::min(round8(tile_capacity * a.n_tiles), resident_blocks());
    hipLaunchKernelGGL((row_tiled_kernel<MODE, 2, GATHER, SAVE_GU, TURN>), dim3(blocks), dim3(NT), R_LDS_BYTES, s, a);
    return check_launch(what);
  }
  static PerDeviceOnce configured;  // one per kernel instantiation
  if (configured.needed()) {
    if (int rc = set_lds(row_tiled_kernel<MODE, 4, GATHER, SAVE_GU, TURN>, R_LDS_BYTES)) return rc;
    configured.done();
  }
  a.by_n_tiles = divisor(a.n_tiles);
  const unsigned blocks = std::min(round8(tile_capacity * a.n_tiles), beside ? beside_router_blocks(tile_capacity * a.n_tiles) : resident_blocks());
  hipLaunchKernelGGL((row_tiled_kernel<MODE, 4, GATHER, SAVE_GU, TURN>), dim3(blocks), dim3(NT), R_LDS_BYTES, s, a);
  return check_launch(what);
}

// grouped_few.hip
int few_rows_fwd(int stage, const void* a, const int32_t* a_src, int64_t a_rows, const void* b0, const void* b1,
                 void* gate, void* up, void* out, const int32_t* seg_offsets, const int32_t* seg_counts,
                 const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* num_tiles, int64_t tiles, int64_t K,
                 int64_t N, bool stream, hipStream_t s);

// grouped_short.hip
int short_rows_fwd(int stage, bool tall, const void* a, const int32_t* a_src, int64_t a_rows, const void* b0, const void* b1,
                   void* gate, void* up, void* out, const int32_t* seg_offsets, const int32_t* seg_counts, const int32_t* tile_expert,
                   const int32_t* tile_row0, const int32_t* num_tiles, int64_t tile_capacity, int64_t El, int64_t K, int64_t N,
                   int64_t row_capacity, bool stream, bool turn, hipStream_t s);

// Up to eight rows per expert, or 64 rows in all (`rows`: as many as there may be; one rank's share of the experts may draw every token's).
// A 16-row pass over an expert's weights costs the same for one row as for sixteen and a second pass
// reads them again, from L2 at best.  Block forward of 128 experts of 2048 x 768, these kernels / the row tiles, us: 16 tokens (1 row on average) 133 / 147, 33 183 /
// 200, 64 202 / 210, 100 (6) 205 / 216, 128 (8) 216 / 215; 32 of 256 experts of 7168 x 2048, 16 tokens 186 / 230, 32 245 / 254.  One dense
// segment of 7168 x 2048 alone, gate/up and down, 60 rows 41 + 16 / 79 + 26, 128 rows 79 + 25 / 93 + 30; but beside the routed experts of that share, whose CUs it takes
// then, 128 rows 422 / 401.  Beyond, 64-row passes (grouped_short.hip).
//   Not by what a share's rows are on average: 16 rows a pass read the weights again for each of many (its products, us, these / 64-row passes / row tiles: 100 tokens of eight,
// drawn evenly from the 256 experts 372 / 386 / 408, all from these 32 870 / 430 / 442, from 16 of them 812 / 230 / 228; 40 tokens 229 / 260 / 315, 422 / 413 / 427, 413 / 214 / 217).
static bool few_rows(int64_t El, int64_t rows, int64_t R, int64_t D, int64_t F) {
  return rows <= std::max<int64_t>(8 * El, 64) && R * std::max(D, F) * 2 < (int64_t{1} << 32);
}

// Rows of a pass of grouped_short.hip, 0 for the row tiles (block forward, us, row tiles / 64 / 128 rows a pass).
//   Up to 45 rows an expert 64, as long as a token is one row of an expert and there are no more than 64 (every pass is the only reader of its weights), or the products are
// small; 128 for up to 128 tokens.  Beyond, the host does not know the load, and where a few experts have all rows, or a share all tokens, the passes are
// short of matrix-core time.  The products alone, weights from memory, us, 64 / 128 / row tiles, of loads drawn evenly, by Zipf's law, from a quarter of the experts (a share: from the rank's
// own 32), from 16, from eight: 32 of 256 of 7168 x 2048, 64 tokens 384 / 390 / 405, 261 / 271 / 315, 420 / 420 / 433, 218 / 222 / 219, 117 / 120 / 156; 100 tokens 386 / 391 / 408,
// 306 / 312 / 355, 430 / 433 / 442, 230 / 235 / 228, 177 / 139 / 163; 128 tokens 408 / 409 / 424, 326 / 327 / 362, 442 / 446 / 449, 301 / 249 / 235, 189 / 148 / 168; 256 tokens 412 / 412 /
// 427, 394 / 432 / 422, 607 / 497 / 475, 425 / 418 / 253, 292 / 250 / 210.  128 of 2048 x 768, 300 tokens (2400 rows, 3.8 * 10^9 of rows D F) 192 / 194 / 198, 196 / 206 / 230, 79 / 68 / 68, 63 / 60 / 62,
// 43 / 52 / 54; 400 tokens 198 / 200 / 204, 206 / 209 / 211, 81 / 76 / 71, 70 / 67 / 68, 56 / 56 / 63; 600 tokens 211 / 215 / 215, 230 / 225 / 250, 108 / 113 / 78, 90 / 97 / 66, 79 / 72 / 67.
//   The share's whole forward, us, row tiles from 33 tokens on / these, evenly, from its 32, from 16, from eight: 40 tokens 396 / 386, 462 / 446, 252 / 246, 188 / 144; 64 tokens 390 / 339, 472 /
// 456, 258 / 256, 194 / 153; 128 tokens 458 / 443, 489 / 481, 270 / 280, 205 / 181 (16 rows a pass up to 102 tokens, then 64: 40 tokens 351, 454, 448, 354; 100 tokens 429, 905, 818, 793; 400 tokens, where these
// and the row tiles are the same 483, 552, 341, 309: 467, 716, 573, 502).
//   As many where all passes are at most two workgroups a CU, and 256-row tiles would leave most CUs without one: 16 experts of 512 x 384, four each, 90 to 300
// rows an expert 35-41 / 31-36 / 35-39; 16 of 1024 x 512, 90 to 220 rows 44-50 / 39-44 / 45-48, 300 51 / 53 / 54, 400 56 / 64 / 56; 32 of it, 90 rows 55 / 53 /
// 52, 130 58 / 64 / 67; one dense segment of 7168 x 2048, 129 rows 132 / 78 / 118, 512 177 / 83 / 119, 1000 179 / 115 / 126, 1400 182 / 164 / 164, 2000
// 187 / 238 / 185; of 2048 x 1408, 129 to 1400 rows 60-83 / 41-46 / 53-57.
//   128 up to 90 rows where the passes are more and the weights stay in the memory-side cache: 64 of 1024 x 512, 60 / 75 / 90 rows
// 75 / 76 / 71, 77 / 81 / 74 (80 rows), 79 / 85 / 79; 64 of 640 x 704, 90 rows 80 / 79 / 75; 32 of 1280 x 640 71 / 68 / 72, 73 / 75 / 74, 75 / 77 / 78.  (16 of 2048 x 1024 are
// just two workgroups a CU and stay with 64: drawn evenly 74 / 78 / 66, 75 / 77 / 68, 76 / 77 / 70, but the products alone by Zipf's law 54 / 55 / 69, 58 / 55 / 71, 84 / 58 / 68.)  Weights from memory
// arrive as fast through row tiles then (60 of 1728 x 960, 60 rows 150 / 162 / 151; 128 of 2048 x 768 261 / 300 / 267).
// (These times are of row tiles whose addresses were formed from scratch, top of this file.  With the present ones gate/up and down alone, even loads, passes / row tiles: 64 of
// 1024 x 512, 45 rows (64-row passes) 48 / 46, 60 rows 50 / 47, 85 rows 55 / 48; 20 rows 42 / 43; 128 of 2048 x 768, 12 rows 191 / 194, by Zipf's law 200 / 219; 32 of 7168 x 2048, 20
// and 45 rows 444 / 439, 480 / 464.  The lines stand for the uneven loads, which have not been timed again above 12 rows.)
//   A dense segment beside other products leaves them more CUs in passes of 128, up to 256 rows (one rank's share of 7168 x 2048 with a shared expert of 2048, 100 / 128 / 150 / 256 / 300 /
// 350 / 400 tokens 378 / 385 / 372, 386 / 398 / 384, 420 / 428 / 420, 426 / 441 / 427, 418 / 432 / 423, 424 / 447 / 431, 438 / 462 / 461; 64 experts of 2048 x 1408 with one of 2816, 100 / 200 / 300 / 400 213 /
// 209 / 208, 219 / 216 / 219, 224 / 231 / 236, 233 / 237 / 245; 16 of 64 of 4096 x 1024 with one of 1024, 100 / 300 143 / 126 / 138, 149 / 129 / 144).
static int short_rows(int64_t El, int64_t rows, int64_t tokens, int64_t D, int64_t F, bool beside) {
  if (El > 256 || rows < 1) return 0;  // (what a wave there adds up)
  if (El == 1 && beside) return rows <= 256 ? 128 : 0;
  const double mean = static_cast<double>(rows) / static_cast<double>(El), sd = El == 1 ? 0.0 : std::sqrt(mean);
  if (El > 1 && mean <= 45.0) {
    if (tokens <= 64 || rows * D * F <= 4'000'000'000) return 64;
    if (tokens <= 128) return 128;
  }
  const int64_t groups = std::max((F + 63) / 64, (D + 127) / 128);
  if (pieces(mean, sd, 64) * static_cast<double>(El * groups) <= 2.0 * resident_blocks()) return 64;
  return El > 1 && mean <= 90.0 && !streamed(El, D, F) ? 128 : 0;
}

// Turned contractions: where weight rows lie a multiple of 4 KiB apart (2048 elements) and most experts have one row
// tile, so that the product is a read of the weights.  Block forward, 128 experts of 2048 x 768, eight a token, us, as ever / turned:
// 150 tokens 278 / 243, 300 269 / 248, 600 303 / 263, 1000 279-306 / 271, 2000 340 / 313, 3000 (187 rows) 378 / 365, 4000 (250) 474 / 476,
// 8192 766 / 779; 64 experts of 2048 x 2048, 700 tokens of six 355 / 329, 4096 x 1024 366 / 336; rows of 1024, 1536 and 7168 elements
// the same within 1 %.  The fp32 sums are the same products in another order, so a bf16 result may round the other way: across 200 rows
// an expert (and 8, grouped_few.hip) a token's bits depend on how many come with it (1000 tokens of that block: 3e-4 of the output, at most a bf16 step).
static bool turned(int64_t El, int64_t R, int64_t K) { return El > 1 && R <= 200 * El && K * 2 % 4096 == 0; }

// Rows that a pass of the forward's kernels has: 16, 64, 128 or 256.  tokens: 0 where the rows are read in place.
static int pass_rows(int64_t El, int64_t D, int64_t F, int64_t row_capacity, int64_t rows_expected, int64_t tokens, bool beside) {
  if (few_rows(El, rows_expected, row_capacity, D, F)) return 16;
  const int pass = short_rows(El, rows_expected, tokens > 0 ? tokens : rows_expected, D, F, beside);
  return pass ? pass : 256;
}

int bf16_fwd_kernels(int64_t El, int64_t D, int64_t F, int64_t row_capacity, int64_t rows_expected, int64_t tokens, int64_t tile_capacity) {
  const int pass = pass_rows(El, D, F, row_capacity, rows_expected, tokens, false);
  auto across = [](int64_t width, int64_t tile) { return (width + tile - 1) / tile; };
  const bool tiles = pass == 256, turn = pass > 16;
  return pass | (tiles && narrow(RM_GATEUP, El, across(F, 128), across(F, 64), tile_capacity) ? MI355_FWD_NARROW_GATEUP : 0) |
         (tiles && narrow(RM_DOWN, El, across(D, 256), across(D, 128), tile_capacity) ? MI355_FWD_NARROW_DOWN : 0) |
         (turn && (tokens > 0 || !tiles) && turned(El, row_capacity, D) ? MI355_FWD_TURNED_GATEUP : 0) |
         (turn && turned(El, row_capacity, F) ? MI355_FWD_TURNED_DOWN : 0);
}

// Work items on short tiles that a product of these counts makes (0: it walks the list's tiles); stage: one of gate/up, down, dRows.
int64_t bf16_short_tiles(int stage, int64_t El, int64_t D, int64_t F, int64_t row_capacity, int64_t tokens, int64_t tile_capacity,
                         const int32_t* counts, int64_t listed) {
  const int mode = stage == STAGE_GATEUP ? RM_GATEUP : stage == STAGE_DOWN ? RM_DOWN : RM_DX;
  const int64_t width = mode == RM_GATEUP ? F : D, tile = mode == RM_GATEUP ? 128 : 256, across = (width + tile - 1) / tile;
  if (!short_tiles_may(mode, El, D, F) || narrow(mode, El, across, (2 * width + tile - 1) / tile, tile_capacity) ||
      (mode != RM_DX && pass_rows(El, D, F, row_capacity, row_capacity, tokens, false) != 256))
    return 0;
  int total = 0, whole = 0;
  for (int64_t e = 0; e < El; ++e) {
    total += (counts[e] + kShortTile - 1) / kShortTile;
    whole += (counts[e] + kListTile - 1) / kListTile;
  }
  const unsigned blocks = std::min(round8(tile_capacity * across), resident_blocks());
  return short_tiles_serve(total, whole, (int)listed, (int)across, (int)blocks) ? total * across : 0;
}

int bf16_grouped_fwd(const void* rows, const int32_t* token_of_row, int64_t num_tokens, const void* w1,
                     const void* w3, const void* w2, const int32_t* seg_offsets, const int32_t* seg_counts,
                     const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* num_tiles,
                     int64_t tile_capacity, void* gate, void* up, void* h, void* y, int64_t El, int64_t D,
                     int64_t F, int64_t row_capacity, int64_t rows_expected, int stages, hipStream_t s) {
  const bool stream = streamed(std::min(El, row_capacity), D, F);  // (of the experts that can have rows)
  const int pass = pass_rows(El, D, F, row_capacity, rows_expected, token_of_row ? num_tokens : 0, stages & STAGE_BESIDE);
  if (pass == 16) {
    const int64_t tiles = std::min(tile_capacity, std::min(El, row_capacity) + row_capacity / 256);
    if (stages & STAGE_GATEUP)
      if (int rc = few_rows_fwd(1, rows, token_of_row, num_tokens, w1, w3, gate, up, h, seg_offsets, seg_counts,
                                tile_expert, tile_row0, num_tiles, tiles, D, F, stream, s))
        return rc;
    if (stages & STAGE_DOWN)
      return few_rows_fwd(2, h, nullptr, 0, w2, w2, nullptr, nullptr, y, seg_offsets, seg_counts, tile_expert, tile_row0,
                          num_tiles, tiles, F, D, stream, s);
    return MI355_OK;
  }
  if (pass < 256) {
    if (stages & STAGE_GATEUP)
      if (int rc = short_rows_fwd(1, pass > 64, rows, token_of_row, num_tokens, w1, w3, gate, up, h, seg_offsets, seg_counts,
                                  tile_expert, tile_row0, num_tiles, tile_capacity, El, D, F, row_capacity, stream,
                                  turned(El, row_capacity, D), s))
        return rc;
    if (stages & STAGE_DOWN)
      return short_rows_fwd(2, pass > 64, h, nullptr, 0, w2, w2, nullptr, nullptr, y, seg_offsets, seg_counts, tile_expert, tile_row0,
                            num_tiles, tile_capacity, El, F, D, row_capacity, stream, turned(El, row_capacity, F), s);
    return MI355_OK;
  }
  const bool beside = stages & STAGE_BESIDE;
  RowArgs a{};
  a.seg_offsets = seg_offsets; a.seg_counts = seg_counts; a.tile_expert = tile_expert;
  a.tile_row0 = tile_row0; a.num_tiles = num_tiles; a.D = (int)D; a.F = (int)F;
  if (stages & STAGE_GATEUP) {
    a.a0 = (const uint16_t*)rows; a.a_src = token_of_row; a.a_rows = (int)num_tokens;
    a.b0 = (const uint16_t*)w1; a.b1 = (const uint16_t*)w3;
    a.o0 = (uint16_t*)gate; a.o1 = (uint16_t*)up; a.o2 = (uint16_t*)h;
    // gate == up == null: a forward-only caller; the kernel then writes h alone
    const bool save = gate != nullptr;
    int rc;
    if (token_of_row && turned(El, row_capacity, D))
      rc = save ? launch_row<RM_GATEUP, true, true, true>(a, F, El, tile_capacity, s, "grouped gate/up", beside)
                : launch_row<RM_GATEUP, true, false, true>(a, F, El, tile_capacity, s, "grouped gate/up (h only)", beside);
    else if (token_of_row)
      rc = save ? launch_row<RM_GATEUP, true>(a, F, El, tile_capacity, s, "grouped gate/up", beside)
                : launch_row<RM_GATEUP, true, false>(a, F, El, tile_capacity, s, "grouped gate/up (h only)", beside);
    else
      rc = save ? launch_row<RM_GATEUP>(a, F, El, tile_capacity, s, "grouped gate/up", beside)
                : launch_row<RM_GATEUP, false, false>(a, F, El, tile_capacity, s, "grouped gate/up (h only)", beside);
    if (rc) return rc;
  }
  if (stages & STAGE_DOWN) {
    RowArgs b = a;
    b.a_src = nullptr;
    b.a0 = (const uint16_t*)h; b.b0 = (const uint16_t*)w2; b.o0 = (uint16_t*)y;
    if (int rc = turned(El, row_capacity, F) ? launch_row<RM_DOWN, false, true, true>(b, D, El, tile_capacity, s, "grouped down")
                      : launch_row<RM_DOWN>(b, D, El, tile_capacity, s, "grouped down"))
      return rc;
  }
  return MI355_OK;
}

// dx = dy . w[e] over the listed segments: dy (rows, O), w (El, O, I), dx (rows, I)
int bf16_grouped_linear_dx(const void* dy, const void* w, const int32_t* seg_offsets, const int32_t* seg_counts,
                           const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* num_tiles,
                           int64_t tile_capacity, void* dx, int64_t El, int64_t O, int64_t I, hipStream_t s) {
  RowArgs a{};
  a.seg_offsets = seg_offsets; a.seg_counts = seg_counts; a.tile_expert = tile_expert;
  a.tile_row0 = tile_row0; a.num_tiles = num_tiles; a.D = (int)O; a.F = (int)I;
  a.a0 = (const uint16_t*)dy; a.b0 = (const uint16_t*)w; a.o0 = (uint16_t*)dx;
  return launch_row<RM_DLIN>(a, I, El, tile_capacity, s, "grouped linear dx");
}

int bf16_fused_dot_slots(int64_t F) {
  // one partial per 128 output columns of the dH tile (two waves across its 256 columns)
  return (int)((F + 255) / 256) * 2;
}

// row_scale != null: the combine's backward is folded in.  dy is then the layer's output
// gradient (T, D), read through token_of_row and scaled by row_scale; `h` is written (it
// receives row_scale * h, the operand of dW2) and dot_partial gets the score-gradient pieces.
int bf16_grouped_bwd(const void* dy, const void* rows, const int32_t* token_of_row, int64_t num_tokens,
                     const void* w1, const void* w3, const void* w2, const void* gate, const void* up,
                     const void* h, const float* row_scale, float* dot_partial,
                     const int32_t* seg_offsets, const int32_t* seg_counts,
                     const int32_t* tile_expert, const int32_t* tile_row0, const int32_t* num_tiles,
                     int64_t tile_capacity, void* dgate, void* dup, void* drows, void* dw1,
                     void* dw3, void* dw2, int64_t El, int64_t D, int64_t F, int stages,
                     hipStream_t s) {
  RowArgs a{};
  a.seg_offsets = seg_offsets; a.seg_counts = seg_counts; a.tile_expert = tile_expert;
  a.tile_row0 = tile_row0; a.num_tiles = num_tiles; a.D = (int)D; a.F = (int)F;
  if (stages & STAGE_DH) {
    a.a0 = (const uint16_t*)dy; a.b0 = (const uint16_t*)w2;
    a.gate = (const uint16_t*)gate; a.up = (const uint16_t*)up;
    a.o0 = (uint16_t*)dgate; a.o1 = (uint16_t*)dup;
    if (row_scale) {
      a.a_src = token_of_row; a.a_rows = (int)num_tokens; a.row_scale = row_scale; a.dot_partial = dot_partial;
      a.o2 = (uint16_t*)const_cast<void*>(h);
      a.dot_slots = bf16_fused_dot_slots(F);
      if (int rc = launch_row<RM_DH, true>(a, F, El, tile_capacity, s, "grouped dh + combine")) return rc;
      a.a_src = nullptr;
    } else {
      if (int rc = launch_row<RM_DH>(a, F, El, tile_capacity, s, "grouped dh")) return rc;
    }
  }
  if (drows && (stages & STAGE_DX)) {
    RowArgs b = a;
    b.a0 = (const uint16_t*)dgate; b.a1 = (const uint16_t*)dup;
    b.b0 = (const uint16_t*)w1; b.b1 = (const uint16_t*)w3; b.o0 = (uint16_t*)drows;
    if (int rc = launch_row<RM_DX>(b, D, El, tile_capacity, s, "grouped drows")) return rc;
  }
  static PerDeviceOnce wconfigured;
  if (wconfigured.needed()) {
    if (int rc = set_lds(wgrad_kernel<false>, R_LDS_BYTES)) return rc;
    if (int rc = set_lds(wgrad_kernel<true>, R_LDS_BYTES)) return rc;
    if (int rc = set_lds(wgrad_kernel<false, true>, R_LDS_BYTES)) return rc;
    wconfigured.done();
  }
  auto wgrad = [&](const void* A, const void* B, const int32_t* b_src, void* C, int64_t M, int64_t N, const char* what,
                   const int32_t* a_src = nullptr, const void* A1 = nullptr, void* C1 = nullptr) {
    WgradArgs w{};
    w.a = (const uint16_t*)A; w.b = (const uint16_t*)B; w.c = (uint16_t*)C; w.b_src = b_src; w.a_src = a_src;
    w.src_rows = (int)num_tokens;
    w.seg_offsets = seg_offsets; w.seg_counts = seg_counts; w.El = (int)El; w.M = (int)M; w.N = (int)N;
    w.m_tiles = (int)((M + WBM - 1) / WBM); w.n_tiles = (int)((N + WBN - 1) / WBN);
    w.total = (int)(El * w.m_tiles * w.n_tiles);
    w.by_tiles = divisor(w.m_tiles * w.n_tiles);
    w.by_n_tiles = divisor(w.n_tiles);
    w.a1 = (const uint16_t*)A1; w.c1 = (uint16_t*)C1;
    const dim3 grid(std::min(round8((int64_t)w.total * (C1 ? 2 : 1)), resident_blocks()));
    if (a_src)
      hipLaunchKernelGGL((wgrad_kernel<false, true>), grid, dim3(NT), R_LDS_BYTES, s, w);
    else if (b_src)
      hipLaunchKernelGGL(wgrad_kernel<true>, grid, dim3(NT), R_LDS_BYTES, s, w);
    else
      hipLaunchKernelGGL(wgrad_kernel<false>, grid, dim3(NT), R_LDS_BYTES, s, w);
    return check_launch(what);
  };
  // folded combine: dW2 = (gathered output gradient)^T . (row_scale * h)
  if (dw2 && (stages & STAGE_DW2))
    if (int rc = wgrad(dy, h, nullptr, dw2, D, F, "grouped dw2", row_scale ? token_of_row : nullptr)) return rc;
  // dW1 and dW3 share their second operand: one launch has both, a tile of one beside the same tile of the other, and ends once.  A training step, us, apart /
  // together: 64 experts of 1024 x 512, six each, 300, 700, 1500, 3000, 5686 tokens 205 / 200, 242 / 236, 309 / 304, 382 / 367, 594 / 564; 64 of 768 x 448, two each, 489
  // tokens 155 / 148; 32 of 832 x 640, five each, 6991 603 / 588; 16 of 2048 x 1024, four each, 3000 566 / 557; 128 of 2048 x 768, eight each, 1600 816 / 809, 4000 1370 / 1373,
  // 8192 2213 / 2205, 16384 of a skewed router 4142 / 4120.  (As two planes of the grid, whose workgroups follow each other, 2645 tokens of it and 7222 of 32
  // of 1600 x 960 lost 2-3 %.)  Not where many tiles of one K step each do nothing but write: 200 to 450 tokens of the 128 experts 698 / 701.
  const int64_t tiles = El * ((F + WBM - 1) / WBM) * ((D + WBN - 1) / WBN);
  const bool one_step = 4 * (tile_capacity - El - 1) <= El;  // 64 rows an expert
  if (dw1 && dw3 && (stages & STAGE_DW1) && (stages & STAGE_DW3) && !(one_step && tiles > 8 * (int64_t)resident_blocks()))
    return wgrad(dgate, rows, token_of_row, dw1, F, D, "grouped dw1 and dw3", nullptr, dup, dw3);
  if (dw1 && (stages & STAGE_DW1)) if (int rc = wgrad(dgate, rows, token_of_row, dw1, F, D, "grouped dw1")) return rc;
  if (dw3 && (stages & STAGE_DW3)) if (int rc = wgrad(dup, rows, token_of_row, dw3, F, D, "grouped dw3")) return rc;
  return MI355_OK;
}

}  // namespace mi355
