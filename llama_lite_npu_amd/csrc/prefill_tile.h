// Varlen causal FlashAttention-2 prefill for gfx950, over paged KV (block table) or over packed
// contiguous K/V (reference: lite_llama/kernels/flashattention2_nopad.py:9-166 and
// paged_chunk_flashattention.py:12-222).
//
// A workgroup of 4 wavefronts owns 128 score columns: up to 8 query heads of one KV head (the
// GQA group) times 16 * row_tiles query rows, 32 columns per wavefront. It walks the keys the
// block may see in tiles of 64 (two halves of 32 for the softmax). Per tile and wavefront:
//
//   S^T[key][col]  = K_tile[64 x 128] . Q^T[128 x 32]         32 x MFMA 16x16x32
//   causal mask, online softmax per column (fp32, exp2 domain, lazy rescale)
//   O^T[d][col]   += V_tile^T[128 x 64] . P^T[64 x 32]         32 x MFMA 16x16x32
//   l[col]        += 1^T . P^T                                   4 x MFMA 16x16x32
//
// Both products are computed transposed so that the accumulator layout of S^T (lane = column,
// 4 consecutive keys per lane group) is the B-operand layout of the second product: P stays in
// its lane, cast to fp16 like the reference's `p.to(v.dtype)` (flashattention2_nopad.py:150).
// The k index of one second-product MFMA runs over (keys 4g..4g+3 of a 16-key tile, then the
// same of the next tile) for lane group g, which is what two S^T accumulator tiles hold and what
// two transposing LDS reads of V deliver. The softmax denominator is one more MFMA against a
// tile of ones, which also reduces it across lane groups.
//
// K/V tiles go from HBM straight into LDS (global_load_lds_dwordx4, no registers in between),
// double buffered: the loads of tile t+1 are in flight while tile t is consumed, and one
// barrier per tile orders them. The direct load writes 64 lanes x 16 bytes contiguously, so
// rows are unpadded (256 bytes) and the 16-byte chunks of a row are XOR-swizzled instead: the
// lane that fills slot p of row r fetches chunk p ^ f(r) from memory. f differs for K (read
// back as 16-byte rows by 16 lanes of different rows) and V (read back transposed, 8 rows x
// 32 bytes at a time); both reads are then free of bank conflicts.
//
// In the fast tiles the score accumulators start from -m / c (m the running maximum of their
// column, c the softmax scale times log2 e) instead of zero, so the MFMA result times c is the
// exponent: a probability costs one multiply, one v_exp_f32 and half a packed conversion. q is not
// pre-multiplied by c: rounding q * c to fp16 would cost the scores 2^-12 of every channel's
// share. Whether the running maximum still holds is checked on the packed fp16
// probabilities (any above 2^kMaxP, or not finite, sends the sub-tile to general_tile), not by a
// column maximum over the fp32 scores.
//
// The accumulators are only ever rescaled in straight-line code (general_tile): a conditional
// rescale inside the key loop makes the compiler copy all 72 accumulator registers at the join
// on every tile. Tiles below the diagonal run in a loop of three straight-line blocks, each laid
// out as a pipeline with scheduling fences and group barriers: the eight K fragments of a
// half-tile are requested at once and each register is refilled with the other half's fragment as
// soon as its MFMA pair has issued; V fragments are requested a block ahead of their use; the
// exponentials of one half run beside the MFMAs of the other; the next tile's HBM -> LDS loads
// leave a quarter at a time between MFMA pairs instead of in one burst behind the barrier.
//
// q and the output move as whole 256-byte rows: q comes in through the direct HBM -> LDS load
// (into the half that tile 1 takes later) and is read back as fragments; the accumulators, which
// hold O^T (4 consecutive d of one row per lane), are transposed through LDS after the last tile
// and leave 4 rows per store instruction. Straight from registers, every q load and output store
// touched 16 rows with 64 / 32 bytes each.
//
// What bounds the loop is the port that issues vector instructions, and the power the chip may draw: a tile of
// 128-wide heads has 68 MFMAs of 16 cycles and, of four-cycle slots on that port, two for each of them, two for each of its
// 32 exponentials and one for each other vector instruction. So the tile of ones stays in registers, maxima of
// packed pairs take three operands and the page ids' address is a 32-bit offset, 14 instructions fewer. Passes: four
// prompts of 5000 to 8192 tokens, 64 / 8 heads, 2748 -> 2710 us, eight of 128 to 2048, two layers, 678 -> 671; 32 / 8 heads of
// 64, 4 x 4096 322 -> 315, four chunks of 512 rows over up to 8000 tokens of int8, two layers, 359 -> 348.
//
// About 235 registers per lane leave two wavefronts per SIMD: two workgroups share a compute
// unit and drift apart, so one's softmax (vector ALU) overlaps the other's MFMAs and a
// finishing block's prologue/epilogue hides behind its neighbour. Grid: x = kv head (times the
// head split), y = row block (long blocks first), z = sequence; with 8 kv heads a head's blocks
// all land on one XCD and share its L2.
#pragma once

#include <type_traits>

#include "common.h"
#include "head_dim.h"
#include "kv_fp8.h"
#include "prefill_rows.h"

namespace litekv {
inline namespace LITEKV_HD_NS {
namespace prefill_tile {

constexpr int kHD = LITEKV_HD;              // head dim of this build of the file
constexpr int kKSteps = kHD / 32;           // MFMA k steps of the first product
constexpr int kJTiles = kHD / 16;           // 16-row tiles of O^T; also K fragments per 32-key half
constexpr int kChunks = kHD / 8;            // 16-byte chunks of a staged row
constexpr int kRowsPerLoad = 64 / kChunks;  // rows one direct-load instruction (64 x 16 bytes) fills
constexpr int kLoadsPerWave = 16 / kRowsPerLoad;  // such instructions per wavefront, tile and operand

// XOR applied to the 16-byte chunk index of staged row r, for K (and q) and for V. A row of 256
// bytes covers all 64 banks, so consecutive rows must differ in the chunk; rows of 128 bytes
// alternate between the bank halves, so it is every second row that must.
// (Rows of 512 bytes cover the banks twice over: the map of 256-byte rows inside each half.)
__device__ __forceinline__ int k_swz(int r) { return kHD >= 128 ? (r & 15) : ((r >> 1) & 7); }
__device__ __forceinline__ int v_swz(int r) { return kHD >= 128 ? 2 * (r & 7) : 2 * ((r >> 1) & 3); }

// At head dim 256 a probability reaches the second product as two fp16 numbers, its rounding and
// what the rounding left, each with an MFMA of its own: prompts of that width have always been
// attended with fp32 probabilities. It costs half as many MFMAs again (the V fragments and their LDS
// reads are shared). The two hold p within 2^-23 of its value (v_exp_f32 is good for about as much),
// or within 2^-25, half of fp16's smallest step, if that is more. What the second bound means for a
// row depends on where its largest probability lies: it is put at 2^kMaxBias instead of 1, and may
// grow to 2^kMaxP before the row is rescaled, so that the bound is at most 2^-34 of it. (At 1, a
// row that is the sum over 12 000 keys 22.4 powers of two less likely than one of value 0 was off
// by 1.4e-2 of itself; at 2^9 by 3e-5, a sixteenth of the output's own rounding. 2^9 costs nothing;
// with 2^11 rows outgrow their bound more often, and four prompts of 300 to 2048 tokens, 16 / 4
// heads, take 2.5 % longer, with 2^13 a third.)
constexpr bool kTwoPartP = kHD == 256;
constexpr int kMaxBias = kTwoPartP ? 9 : 0;
constexpr int kMaxP = kTwoPartP ? 15 : 8;
// Workgroups per compute unit: bounded by registers at 64 and 128 (about 150 and 235 per lane), by
// LDS at 256 (two tiles of K and of V are 128 KiB), where a lane may then use all 512 registers (codes: four wavefronts)
// or 256 (fp16 rows: eight).
constexpr int kWgPerCu = kHD == 64 ? 3 : kHD == 128 ? 2 : 1;
// Immediate of s_waitcnt that waits for all but the n youngest vector memory requests.
constexpr int wait_vm(int n) { return 0x0F70 | (n & 15) | ((n >> 4) << 14); }

constexpr float kLog2eP = 1.4426950408889634f;

// Scales (times log2 e, times the K scale of a pool of codes) the tile arithmetic is made for: it
// takes maxima of unscaled scores (wrong below 0), and seeds the accumulators with a quotient by
// the scale (no number at 0, lost below fp32's normal range). Head dim 256 takes any scale, so what
// lies outside goes another way there.
__host__ __device__ constexpr bool tile_scale(float k_mul) { return k_mul >= 0x1p-100f && k_mul <= 0x1p100f; }

// The entry of a block-table row, `bt_stride` (at least 1) of them, that holds page pidx of 16 tokens. A length beyond the row
// re-reads its last entry, and so does a page in front of the row, which a sequence without a key (a context length of
// minus its rows or less) asks for: the caller's 32-bit byte offset would take -1 to be 4 GiB past the row.
__host__ __device__ __forceinline__ uint32_t table_entry(int pidx, int page_shift, int bt_stride) {
  const uint32_t at = (uint32_t)(pidx >> page_shift), last = (uint32_t)bt_stride - 1u;
  return at < last ? at : last;
}

// Where the keys of a sequence live.
struct PagedSource {
  const half_t *kv;             // pool [slots][2*Hkv][128], fp16 (or E4M3 codes, one byte each)
  const int32_t *block_table;   // [B][stride]
  int32_t bt_stride;
  int32_t num_kv_heads;
  int32_t num_pages;
  const float *scales;          // fp8 pool: value = code * scale, K heads then V heads
  int32_t page_shift;           // pages of 16 << page_shift tokens
};
// Shared-prefix decode (mode kSharedPrefix): the columns are (sequence, query head) pairs of one
// decode step, the keys are a slice of the pages every sequence starts with, and the result is
// a normalised fp32 partial row + log-sum-exp per column, for the decode merge.
// Prefill over key slices (mode kPagedPrefillSplit) writes the same kind of partial rows, one
// per (key slice, query row, head): `batch` then counts the query rows of the launch.
struct PrefixTask {
  float *part_o;            // [splits][batch][Hq][128]
  float *part_lse;          // [splits][batch][Hq]
  int64_t q_batch_stride;   // elements between the q rows of consecutive sequences
  int32_t batch;
  int32_t num_q_heads;
  int32_t prefix_keys;      // shared pages * 16
  int32_t keys_per_split;   // multiple of the key tile
};
struct PackedSource {
  const half_t *k;              // [T][Hkv][128]
  const half_t *v;
  int64_t k_stride, v_stride;   // elements per token
  const int32_t *seq_starts;    // [B]
};

constexpr int kKvTile = 64;
constexpr int kColTiles = 2;      // 16-column tiles per wavefront
constexpr int kTiledWaves = 4;    // wavefronts of a prefill workgroup (see prefill_waves)
constexpr int kWideWaves = 8;     // a shared prefix: twice the columns on every staged K/V tile (prefill: 2 to 5 % slower)
constexpr int kWgColTiles = kColTiles * kTiledWaves;
constexpr int kTileHalfs = kKvTile * kHD;  // one staged tile: 64 rows of 2 * kHD bytes

typedef __attribute__((address_space(3))) half_t lds_half_t;
typedef __attribute__((address_space(3))) half8_t lds_half8_t;
typedef __attribute__((address_space(3))) short4_t lds_short4_t;
typedef short short8_t __attribute__((ext_vector_type(8)));

// Plain maxima. This file is compiled with -fno-honor-nans, so the compiler does not wrap every
// operand in a NaN-quieting self-max and fuses pairs into v_max3_f32. (They must stay compiler
// instructions: an asm v_max3 reading an MFMA result gets none of the wait states that the
// compiler inserts between an MFMA and the first use of its result.)
__device__ __forceinline__ float vmax3(float a, float b, float c) {
  return __builtin_fmaxf(__builtin_fmaxf(a, b), c);
}
__device__ __forceinline__ float vmax2(float a, float b) { return __builtin_fmaxf(a, b); }
constexpr int kPagedPrefill = 0, kPackedPrefill = 1, kSharedPrefix = 2, kPagedPrefillFp8 = 3,
              kSharedPrefixFp8 = 4, kPagedPrefillInt8 = 5, kSharedPrefixInt8 = 6,
              kPagedPrefillSplit = 7, kPagedPrefillSplitFp8 = 8, kPagedPrefillSplitInt8 = 9;
// kPagedPrefillSplit: a launch with too few row blocks to fill the device (one request's chunk
// over a long history) cuts every block's keys into `key_slices` runs of tiles, one workgroup
// each; a slice leaves a normalised fp32 partial row + log-sum-exp per (query row, head), and a
// merge launch folds the slices of a row (prefill_split_merge_kernel in paged_prefill.hip).

// Column tiles per wavefront and wavefronts per workgroup of a prefill of 128 columns. Head dim 256 leaves one
// workgroup per CU (LDS), which as four wavefronts of two column tiles is a lone wavefront per SIMD: its
// softmax, LDS latencies and barrier waits stand in the open (MFMA busy 45 %). Eight wavefronts of one column tile
// are two per SIMD at 256 registers (MFMA busy 53 %). Every K and V fragment then feeds one column tile instead of two,
// and LDS, read twice as much, is busy 36 % instead of 16: 2.3 us a tile of keys, 2.5 before. A launch of few workgroups
// ends with its longest chain of tiles: 31 x 2.3 of the 76 us below. Kernel time, 16 / 4 heads, four to eight
// wavefronts: 4 prompts of 459 to 1951 tokens 82 -> 76 us; passes with the epilogue, 300 tokens 26.3 -> 21.9, 16 x 500..700
// 153 -> 132, 64 rows over 2000 cached tokens 54.5 -> 48.3. Codes keep four: their conversion needs the registers (eight
// spill, and take 0.98 to 1.02 of the time).
constexpr int prefill_ct(int mode) {
  return kHD == 256 && (mode == kPagedPrefill || mode == kPackedPrefill) ? 1 : kColTiles;
}
constexpr int prefill_waves(int mode) { return kWgColTiles / prefill_ct(mode); }

// Head dim 256: the 16 query rows of column tile t of a block (see prefill_tile_body, whose names these
// are), in fp32 (prefill_rows.h); `lds` as there.
template <int KV, bool PAGED, int ROWS>
__device__ __forceinline__ void tile_by_rows(uint32_t lds, const half_t *q, int64_t q_stride, half_t *out,
                                             int64_t out_stride, const PagedSource &paged,
                                             const PackedSource &packed, int b, int q_start, int q_len, int ctx,
                                             int m0, int t, int row_tiles, int head0, int heads_here, int group,
                                             int h, float scale_log2) {
  const int head = t / row_tiles;
  const int row0 = m0 + (t - head * row_tiles) * 16;
  if (head >= heads_here || row0 >= q_len) return;
  const int hq = h * group + head0 + head;
  constexpr bool CODES = KV != kKvF16;
  auto kv_row = [&](int tok, bool value) -> const void * {
    if constexpr (PAGED) {
      const int shift = 4 + paged.page_shift;
      int at = tok >> shift;
      at = at < paged.bt_stride ? at : paged.bt_stride - 1;  // a length beyond the row re-reads its last entry
      int pid = paged.block_table[(int64_t)b * paged.bt_stride + at];
      pid = pid < 0 ? 0 : (pid >= paged.num_pages ? paged.num_pages - 1 : pid);
      const int64_t slot = ((int64_t)pid << shift) + (tok & ((1 << shift) - 1));
      return (const char *)paged.kv +
             (slot * 2 * paged.num_kv_heads + (value ? paged.num_kv_heads : 0) + h) * kHD * (CODES ? 1 : 2);
    } else {
      return value ? packed.v + (int64_t)(q_start + tok) * packed.v_stride + h * kHD
                   : packed.k + (int64_t)(q_start + tok) * packed.k_stride + h * kHD;
    }
  };
  const int64_t at = (int64_t)hq * kHD;
  const int rows = q_len - row0 < 16 ? q_len - row0 : 16;
#pragma unroll 1
  for (int r = 0; r < rows; r += ROWS) {
    prefill_rows::attend_rows<KV, ROWS>(lds, q + (int64_t)(q_start + row0 + r) * q_stride + at, q_stride,
                                  out + (int64_t)(q_start + row0 + r) * out_stride + at, out_stride,
                                  rows - r < ROWS ? rows - r : ROWS, ctx + row0 + r + 1,
                                  kv_row, scale_log2, CODES ? paged.scales[h] : 1.0f,
                                  CODES ? paged.scales[paged.num_kv_heads + h] : 1.0f);
  }
}

// The body of the kernel, run by a workgroup of W wavefronts that stands at (block_x, block_y,
// block_z) of a grid block_y runs over grid_y values of; k_lds is the LDS byte address of its
// staging area (tile_lds_bytes<W>() bytes, 1 KiB aligned). A function, so that the decode step
// with a shared prefix can run it as one role of its launch (paged_decode.hip).
template <int W>
constexpr int tile_lds_bytes() { return (W == kWideWaves && kHD != 256 ? 6 : 4) * kTileHalfs * 2; }

template <int MODE, int W, int KG = 1, int CT = kColTiles>
__device__ __forceinline__ void prefill_tile_body(
    const uint32_t lds_base, const int block_x, const int block_y, const int block_z, const int grid_y,
    const half_t *__restrict__ q, int64_t q_stride, half_t *__restrict__ out, int64_t out_stride,
    const PagedSource &paged, const PackedSource &packed, const PrefixTask &prefix,
    const int32_t *__restrict__ q_starts_or_cu, const int32_t *__restrict__ q_lens_or_null,
    const int32_t *__restrict__ context_lens, int32_t group, int32_t head_splits,
    int32_t heads_per_wg, int32_t row_tiles, float scale_log2, const int key_slice = 0,
    const int key_slices = 1) {
  constexpr bool PAGED = MODE != kPackedPrefill;
  // causal prefill over one slice of the block's keys
  constexpr bool KSPLIT = MODE == kPagedPrefillSplit || MODE == kPagedPrefillSplitFp8 ||
                          MODE == kPagedPrefillSplitInt8;
  // An fp8 pool cannot take the direct HBM -> LDS load: its codes go through registers, are
  // converted to fp16 (exactly) and written to LDS in the same swizzled layout, so everything
  // after the staging is shared. The K scale joins the softmax scale, the V scale the final
  // normalisation, as in the decode kernel.
  constexpr bool FP8 = MODE == kPagedPrefillFp8 || MODE == kSharedPrefixFp8 ||
                       MODE == kPagedPrefillInt8 || MODE == kSharedPrefixInt8 ||
                       MODE == kPagedPrefillSplitFp8 || MODE == kPagedPrefillSplitInt8;  // 8-bit codes
  constexpr int KV = (MODE == kPagedPrefillInt8 || MODE == kSharedPrefixInt8 ||
                      MODE == kPagedPrefillSplitInt8) ? kKvInt8 : kKvFp8;
  constexpr bool SHARED = MODE == kSharedPrefix || MODE == kSharedPrefixFp8 || MODE == kSharedPrefixInt8;
  // (rows of 64 codes staged by 8 wavefronts would leave a lane 8 codes, half a 16-byte load)
  static_assert(W == kTiledWaves || (W == kWideWaves && (!FP8 || kHD == 128)),
                "eight wavefronts: fp16 K/V, or 8-bit codes at head dim 128");
  static_assert(kHD != 256 || (W == prefill_waves(MODE) && CT == prefill_ct(MODE) && !KSPLIT && !SHARED), "256: plain prefill only");
  // Rows of a 64-key tile one wavefront stages (a page, or half of one), and the direct-load
  // instructions that takes per operand.
  constexpr int kRowsPerWave = kKvTile / W;
  constexpr int kLoads = kRowsPerWave / kRowsPerLoad;
  static_assert(CT == kColTiles || (CT == 1 && KG == 1 && W == (kHD == 256 ? kWideWaves : kTiledWaves) && !SHARED),
                "one column tile a wavefront: a prefill");
  static_assert(KG == 1 || (KG == 2 && W == kTiledWaves && !KSPLIT && !SHARED && kHD != 256), "two key groups: a prefill");
  const int wave_in_wg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kgroup = KG == 2 ? wave_in_wg / W : 0;  // which half of the keys this wavefront attends
  const uint32_t k_lds = lds_base + (uint32_t)(kgroup * tile_lds_bytes<W>());
  // Two tiles of K, then two of V: tile t sits in half t % 2. (Eight wavefronts have a third
  // region of the same size behind them: room for their partial rows.)
  const uint32_t v_lds = k_lds + 4u * kTileHalfs;  // LDS byte addresses

  const int tid = threadIdx.x;
  const int wave = wave_in_wg - kgroup * W;
  const int lane = tid & 63;
  const int n = lane & 15;
  const int g = lane >> 4;
  const int h = block_x / head_splits;  // kv head
  const int head0 = (block_x - h * head_splits) * heads_per_wg;
  const int heads_here = (group - head0) < heads_per_wg ? (group - head0) : heads_per_wg;
  const int b = block_z;
  // q reaches the MFMA as the caller gave it: the products of fp16 q and K elements are exact and
  // summed in fp32, and the softmax scale (times log2 e, times the K scale of a pool of 8-bit
  // codes) multiplies the finished score in fp32 (k_mul). Folded into q instead, the product
  // would be rounded to fp16 once more: an error of 2^-12 of every channel's share of a score,
  // which rows with a few large channels of q and K (scores tens of log2 units apart) turn into
  // percent-level errors of their probabilities.
  float v_scale = 1.0f, k_mul = scale_log2;
  if constexpr (FP8) {
    k_mul *= paged.scales[h];
    v_scale = paged.scales[paged.num_kv_heads + h];
  }
  const float k_mul_inv = 1.0f / k_mul;

  // What the block works on: query rows m0.. of sequence b (prefill), or the column block
  // block_y of all (sequence, head) pairs against key slice block_z (shared prefix).
  //   kv_end  one past the last key the block may see      diag  last key every column sees
  //   tile0   first key tile (tiles are counted from it)   last_key  last key that exists
  int q_start = 0, q_len = 0, m0 = 0, ctx = 0, kv_end, diag, last_key;
  int tile0 = 0;
  int wg_barriers = 0;  // two key groups: barriers of the one with more tiles
  if constexpr (SHARED) {
    const int key_begin = block_z * prefix.keys_per_split;
    if (key_begin >= prefix.prefix_keys) return;
    kv_end = key_begin + prefix.keys_per_split;
    kv_end = kv_end < prefix.prefix_keys ? kv_end : prefix.prefix_keys;
    diag = kv_end - 1;
    last_key = prefix.prefix_keys - 1;
    tile0 = key_begin / kKvTile;
  } else {
    if (PAGED) {
      q_start = q_starts_or_cu[b];
      q_len = q_starts_or_cu[b + 1] - q_start;
    } else {
      q_start = packed.seq_starts[b];
      q_len = q_lens_or_null[b];
    }
    const int block_rows = 16 * row_tiles;
    // Long blocks first, all heads of a row block next to each other.
    m0 = (grid_y - 1 - block_y) * block_rows;
    if (m0 >= q_len) return;
    ctx = (PAGED && context_lens) ? context_lens[b] : 0;
    const int rows = (q_len - m0) < block_rows ? (q_len - m0) : block_rows;
    kv_end = ctx + m0 + rows;
    diag = ctx + m0;
    last_key = ctx + q_len - 1;
    if constexpr (KG == 2) {
      // The first group takes the first half of the tiles, the second the rest: as in a launch over key
      // slices, from no later than the last tile that every row of the block sees in full. (A block of
      // so few keys leaves the first group without any.)
      const int total = (kv_end + kKvTile - 1) / kKvTile;
      const int plain = (diag + 1) / kKvTile;
      const int last_start = plain > 0 ? plain - 1 : 0;
      const int mid = (total + 1) / 2 < last_start ? (total + 1) / 2 : last_start;
      wg_barriers = mid > total - mid ? mid : total - mid;
      if (kgroup == 0) {
        kv_end = mid * kKvTile;
      } else {
        tile0 = mid;
      }
    }
    if constexpr (KSPLIT) {
      // The tiles every row of the block sees in full (`plain` of them) are shared out among the
      // slices; the last slice also takes the tiles at the diagonal, and starts no later than
      // the last plain tile, so that each of its rows sees at least one key.
      const int total = (kv_end + kKvTile - 1) / kKvTile;
      const int plain = (diag + 1) / kKvTile;
      const int last_start = plain > 0 ? plain - 1 : 0;
      const int per = (plain + key_slices - 1) / key_slices;
      int t_begin = key_slice * per;
      t_begin = t_begin < last_start ? t_begin : last_start;
      int t_end = (key_slice + 1) * per;
      t_end = key_slice == key_slices - 1 ? total : (t_end < last_start ? t_end : last_start);
      if (t_end <= t_begin) {
        // Nothing for this slice: its partial rows say so (log-sum-exp -inf, a row of zeros).
        for (int t = wave * CT; t < wave * CT + CT; ++t) {
          const int head = t / row_tiles;
          const int row = m0 + (t - head * row_tiles) * 16 + n;
          if (head < heads_here && row < q_len) {
            const int64_t cell = ((int64_t)key_slice * prefix.batch + q_start + row) * prefix.num_q_heads +
                                 h * group + head0 + head;
            if (g == 0) prefix.part_lse[cell] = -INFINITY;
            float4_t *dst = (float4_t *)(prefix.part_o + cell * kHD) + g * (kHD / 16);
#pragma unroll
            for (int i = 0; i < kHD / 16; ++i) dst[i] = float4_t{0.f, 0.f, 0.f, 0.f};
          }
        }
        return;
      }
      tile0 = t_begin;
      kv_end = kv_end < t_end * kKvTile ? kv_end : t_end * kKvTile;
    }
  }
  const int n_tiles = (kv_end + kKvTile - 1) / kKvTile - tile0;

  // a wavefront's own part of the staging area, for what it does before and after the tiles
  constexpr uint32_t kOwnLds = (uint32_t)tile_lds_bytes<W>() / W;
  constexpr int kByRows = W == kWideWaves ? 8 : 16;  // rows of a tile attended together where it goes by rows
  static_assert(kHD != 256 || prefill_rows::lds_bytes(kByRows) <= kOwnLds, "rows attended together fit a wavefront's part");
  if constexpr (kHD == 256 && FP8) {
    if (!tile_scale(k_mul)) {  // the K scale's doing: the launch looked at softmax_scale itself
      for (int t = wave * CT; t < (wave + 1) * CT; ++t) {
        tile_by_rows<KV, PAGED, kByRows>(k_lds + wave * kOwnLds, q, q_stride, out, out_stride, paged, packed, b, q_start, q_len,
                                ctx, m0, t, row_tiles, head0, heads_here, group, h, scale_log2);
      }
      return;
    }
  }

  // ---- staging addresses -------------------------------------------------------------------
  // Direct-load instruction i of wavefront w fills tile rows kRowsPerWave * w + 4i .. +3 (one
  // page per wavefront, or half of one): lane l writes slot l % 16 of row 4i + l / 16.
  const int r_loc = lane / kChunks;
  const int slot = lane % kChunks;
  const int sub = (kRowsPerWave * wave) & 15;   // first row of this wavefront's rows inside their page
  const uint32_t k_pitch = PAGED ? 2u * paged.num_kv_heads * kHD * (FP8 ? 1u : 2u)
                                 : (uint32_t)packed.k_stride * 2u;
  const uint32_t v_pitch = PAGED ? k_pitch : (uint32_t)packed.v_stride * 2u;
  // byte offsets from the page (paged) or from the wavefront's first row (packed)
  uint32_t koff[kLoadsPerWave], voff[kLoadsPerWave];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int rip = kRowsPerLoad * i + r_loc;   // row among this wavefront's rows
    const int ck = slot ^ k_swz(sub + rip);      // the swizzle goes by the row of the tile
    const int cv = slot ^ v_swz(sub + rip);
    const int src_row = (PAGED ? sub : 0) + rip;
    koff[i] = src_row * k_pitch + (uint32_t)(h * kHD + 8 * ck) * 2u;
    voff[i] = src_row * v_pitch +
              (uint32_t)(((PAGED ? paged.num_kv_heads : 0) + h) * kHD + 8 * cv) * 2u;
  }
  const int32_t *table =
      PAGED ? paged.block_table + (SHARED ? 0 : (int64_t)b * paged.bt_stride) : nullptr;
  const int last_page = last_key >> 4;
  // The kernel works on 16-token pages: page j of them is part j % (1 << page_shift) of the
  // sequence's page j >> page_shift, whose tokens are contiguous in the pool.
  auto page_of = [&](int pidx) {
    const uint32_t at = table_entry(pidx, paged.page_shift, paged.bt_stride);
    int pid = *(const int32_t *)((const char *)table + 4u * at);  // (a 32-bit offset from a scalar base)
    pid = pid < 0 ? 0 : (pid >= paged.num_pages ? paged.num_pages - 1 : pid);
    return (pid << paged.page_shift) + (pidx & ((1 << paged.page_shift) - 1));
  };

  // Starts the loads of tile kt into its LDS half. The instruction is written as asm so that the
  // compiler does not make later LDS reads of the *other* half wait for it; the wait is the
  // explicit vmcnt(0) before the barrier that publishes the tile.
  // 8-bit pools: a row's codes are shared out among kLanesPerRow lanes, kRawVecs 16-byte vectors
  // of codes per lane and operand
  constexpr int kLanesPerRow = kWave / kRowsPerWave;
  constexpr int kCodesPerLane = kHD / kLanesPerRow;
  constexpr int kRawVecs = FP8 ? kCodesPerLane / 16 : 1;
  uint4_t raw_k[kRawVecs], raw_v[kRawVecs];  // this lane's codes of K and of V of the tile requested last
  auto issue_tile = [&](int kt) {
    const int row0 = (tile0 + kt) * kKvTile + kRowsPerWave * wave;  // first key of this wavefront's rows
    if constexpr (FP8) {
      // lane l: row l / kLanesPerRow of the wavefront's rows, kCodesPerLane codes of the head's row
      int pidx = (tile0 + kt) * 4 + (kRowsPerWave * wave) / 16;
      pidx = pidx < last_page ? pidx : last_page;
      const int pid = page_of(pidx);
      int tok = row0 + lane / kLanesPerRow;
      tok = tok < last_key ? tok : last_key;  // rows past the last key re-read it
      const int src_row = tok - pidx * kPageSize;
      const uint8_t *base = (const uint8_t *)paged.kv +
                            ((int64_t)pid * kPageSize + src_row) * (int64_t)k_pitch +
                            kCodesPerLane * (lane % kLanesPerRow);
      const uint8_t *kp = base + h * kHD;
      const uint8_t *vp = base + (paged.num_kv_heads + h) * kHD;
#pragma unroll
      for (int i = 0; i < kRawVecs; ++i) {
        raw_k[i] = *(const uint4_t *)(kp + 16 * i);
        raw_v[i] = *(const uint4_t *)(vp + 16 * i);
      }
      return;
    }
    const char *kbase, *vbase;
    int src0;  // key index the bases point at
    if (PAGED) {
      int pidx = (tile0 + kt) * 4 + (kRowsPerWave * wave) / 16;
      pidx = pidx < last_page ? pidx : last_page;
      const int pid = page_of(pidx);
      kbase = (const char *)paged.kv + (int64_t)pid * ((int64_t)kPageSize * k_pitch);
      vbase = kbase;
      src0 = pidx * kPageSize;
    } else {
      const int first = row0 < last_key ? row0 : last_key;
      kbase = (const char *)packed.k + (int64_t)(q_start + first) * k_pitch;
      vbase = (const char *)packed.v + (int64_t)(q_start + first) * v_pitch;
      src0 = first;
    }
    // (uniform, which the compiler does not see everywhere)
    const uint32_t dst =
        __builtin_amdgcn_readfirstlane((uint32_t)((kt & 1) * kTileHalfs + kRowsPerWave * wave * kHD) * 2u);
    auto load_rows = [&](uint32_t i, uint32_t ko, uint32_t vo) {
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(k_lds + dst + 1024u * i), "v"(ko), "s"(kbase)
                   : "memory", "m0");
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                   :
                   : "s"(v_lds + dst + 1024u * i), "v"(vo), "s"(vbase)
                   : "memory", "m0");
    };
    if (row0 + kRowsPerWave - 1 <= last_key) {
#pragma unroll
      for (int i = 0; i < kLoads; ++i) load_rows(i, koff[i], voff[i]);
    } else {
      // Only in the last tile of a sequence. Rows past the last key re-read it: finite values
      // that zero probabilities multiply.
      const int off0 = PAGED ? row0 - sub : row0;  // the key the offsets count from
#pragma unroll
      for (int i = 0; i < kLoads; ++i) {
        const int rip = kRowsPerLoad * i + r_loc;
        int tok = row0 + rip;
        tok = tok < last_key ? tok : last_key;
        const uint32_t back = (uint32_t)(row0 + rip - tok) - (uint32_t)(off0 - src0);
        // source row = offset row - back: inside the page / at the clamped packed row
        load_rows(i, koff[i] - back * k_pitch, voff[i] - back * v_pitch);
      }
    }
  };

  // q rows come in as whole 256-byte rows, 4 per direct-load instruction, into a region of the
  // LDS half that tile 1 will take (8 KiB per wavefront, private to it), swizzled like a K tile;
  // the fragments are read back from there. Requested before tile 0: vmcnt counts in order.
  uint32_t q_lds = 0;
  if constexpr (!SHARED) {
    static_assert(16 * CT * W <= 2 * kKvTile, "the q rows of the wavefronts fit a tile half of K and of V");
    q_lds = ((wave & (W / 2)) ? v_lds : k_lds) +
            (uint32_t)(kTileHalfs * 2 + (wave & (W / 2 - 1)) * (kTileHalfs * 4 / W));
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      const int t = wave * CT + u;
      const int head = t / row_tiles;
      const int row0 = m0 + (t - head * row_tiles) * 16;
      const int hq = h * group + head0 + (head < heads_here ? head : 0);
      const int first = row0 < q_len ? row0 : q_len - 1;
      const char *base = (const char *)(q + (int64_t)(q_start + first) * q_stride + (int64_t)hq * kHD);
#pragma unroll
      for (int i = 0; i < kLoadsPerWave; ++i) {
        int rip = kRowsPerLoad * i + r_loc;
        const int chunk = slot ^ k_swz(rip);
        rip = first + rip < q_len ? rip : q_len - 1 - first;  // rows past the end re-read the last one
        const uint32_t off = (uint32_t)rip * (uint32_t)q_stride * 2u + 16u * (uint32_t)chunk;
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(q_lds + (uint32_t)(32 * kHD) * u + 1024u * i), "v"(off), "s"(base)
                     : "memory", "m0");
      }
    }
  }
  issue_tile(0);

  // ---- this wavefront's columns: tile t = head (t / row_tiles), rows 16 * (t % row_tiles) ..
  half8_t qf[CT][kKSteps];
  int q_pos[CT];
  int out_row[CT];   // packed row index, or -1
  int out_head[CT];
#pragma unroll
  for (int u = 0; u < CT; ++u) {
    const int t = wave * CT + u;
    bool ok;
    int hq;
    const half_t *qrow;
    if constexpr (SHARED) {
      const int col = block_y * (16 * CT * W) + 16 * t + n;  // (sequence, head) pair
      ok = col < prefix.batch * group;
      const int seq = ok ? col / group : 0;
      hq = h * group + (ok ? col - seq * group : 0);
      q_pos[u] = kv_end - 1;
      out_row[u] = ok ? seq : -1;
      qrow = q + (int64_t)seq * prefix.q_batch_stride + (int64_t)hq * kHD + 8 * g;
    } else {
      const int head = t / row_tiles;
      const int row = m0 + (t - head * row_tiles) * 16 + n;
      ok = head < heads_here && row < q_len;
      hq = h * group + head0 + (head < heads_here ? head : 0);
      const int last = q_len - 1;
      q_pos[u] = ctx + (row < last ? row : last);
      out_row[u] = ok ? q_start + row : -1;
      qrow = q + (int64_t)(q_start + (ok ? row : 0)) * q_stride + (int64_t)hq * kHD + 8 * g;
    }
    out_head[u] = hq;
    if constexpr (!SHARED) continue;
#pragma unroll
    for (int kk = 0; kk < kKSteps; ++kk) {
      qf[u][kk] = ok ? *(const half8_t *)(qrow + 32 * kk) : half8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  if constexpr (!SHARED) {
    // the loads of tile 0 (K and V) were requested after q's
    if constexpr (FP8) {
      __builtin_amdgcn_s_waitcnt(wait_vm(2 * kRawVecs));
    } else {
      __builtin_amdgcn_s_waitcnt(wait_vm(2 * kLoads));
    }
#pragma unroll
    for (int u = 0; u < CT; ++u) {
#pragma unroll
      for (int kk = 0; kk < kKSteps; ++kk) {
        qf[u][kk] = *(const lds_half8_t *)(uintptr_t)(
            q_lds + (uint32_t)(32 * kHD) * u + (uint32_t)(n * 2 * kHD + 16 * ((4 * kk + g) ^ k_swz(n))));
      }
    }
  }

  float4_t acc[kJTiles][CT];
  float4_t dsum[CT];
  float m_run[CT];
  // Seed of the score accumulators in the fast tiles: -m_run (divided by k_mul), in all four
  // elements, so that the MFMA result is already the exponent.
  float4_t seed[CT];
#pragma unroll
  for (int u = 0; u < CT; ++u) {
    m_run[u] = -INFINITY;
    seed[u] = float4_t{0.f, 0.f, 0.f, 0.f};
    dsum[u] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < kJTiles; ++j) acc[j][u] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  half8_t ones = half8_t{1, 1, 1, 1, 1, 1, 1, 1};
  asm volatile("" : "+v"(ones));  // in registers: left alone, the constant is moved into them again in every tile

  // Swizzled read addresses (LDS bytes) for the tile half in use; they flip between the halves
  // once per tile (the loop below the diagonal takes two tiles at offsets of its own instead).
  // K, A operand of S^T: row 16m + n, chunk (4kk + g) ^ n.
  // (Rows of 512 bytes: the swizzle stays inside a 256-byte half, so the second half's addresses are
  // the first's plus a constant.)
  constexpr int kKAddrs = kHD == 256 ? kKSteps / 2 : kKSteps, kVAddrs = kHD == 256 ? kJTiles / 2 : kJTiles;
  uint32_t k_addr[kKAddrs];
#pragma unroll
  for (int kk = 0; kk < kKAddrs; ++kk) {
    k_addr[kk] = k_lds + 2u * (uint32_t)(n * kHD + 8 * ((4 * kk + g) ^ k_swz(n)));
  }
  // V^T, A operand of O^T: row 32 s2 + 4g + n/4 (+16), halfs 16j + 4(n%4); chunk pair j ^ (r%8).
  const int v_row = 4 * g + (n >> 2);
  uint32_t v_addr[kVAddrs];
#pragma unroll
  for (int j = 0; j < kVAddrs; ++j) {
    v_addr[j] = v_lds + 2u * (uint32_t)(v_row * kHD + 8 * ((2 * j) ^ v_swz(v_row)) + 4 * (n & 3));
  }
  int flip = kTileHalfs * 2;  // bytes to the other half
  auto flip_halves = [&]() {
#pragma unroll
    for (int kk = 0; kk < kKAddrs; ++kk) k_addr[kk] += flip;
#pragma unroll
    for (int j = 0; j < kVAddrs; ++j) v_addr[j] += flip;
    flip = -flip;
  };
  auto k_at = [&](int kk) -> uint32_t { return k_addr[kk % kKAddrs] + 256u * (uint32_t)(kk / kKAddrs); };
  auto v_at = [&](int j) -> uint32_t { return v_addr[j % kVAddrs] + 256u * (uint32_t)(j / kVAddrs); };

  float4_t st[2][CT];
  half8_t pk[CT];
  half8_t pk_lo[CT];  // kTwoPartP: what the rounding of pk left

  // S^T of 32 keys (rows 32 s2 .. +31 of the staged K tile) against this wavefront's columns.
  auto scores_into = [&](float4_t (&st)[2][CT], int s2, auto seeded_tag) {
    constexpr bool SEEDED = decltype(seeded_tag)::value;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int u = 0; u < CT; ++u) st[m][u] = SEEDED ? seed[u] : float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < kKSteps; ++kk) {
        const half8_t a =
            *(const lds_half8_t *)(uintptr_t)(k_at(kk) + 2u * (32 * s2 + 16 * m) * kHD);
#pragma unroll
        for (int u = 0; u < CT; ++u) st[m][u] = mfma_16x16x32(a, qf[u][kk], st[m][u]);
      }
    }
  };
  // -inf on the keys column u may not see; key0 = first key of the sub-tile.
  auto mask_sub = [&](int u, int key0) {
    const int lim = q_pos[u] - key0 - 4 * g;  // key offset 16m + i is visible iff <= lim
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (16 * m + i > lim) st[m][u][i] = -INFINITY;
      }
    }
  };
  // Column maxima of `st`, in scaled (log2) units.
  auto column_max_of = [&](const float4_t (&st)[2][CT], int u) {
    float mx = vmax3(st[0][u][0], st[0][u][1], st[0][u][2]);
    mx = vmax3(mx, st[0][u][3], st[1][u][0]);
    mx = vmax3(mx, st[1][u][1], st[1][u][2]);
    mx = vmax2(mx, st[1][u][3]);
    return max_over_lane_groups(mx) * k_mul;  // k_mul > 0: max and scaling commute
  };
  // p = 2^(s * scale - m), cast to fp16, in B-operand order.
  typedef float float2_t __attribute__((ext_vector_type(2)));
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  // General path: p = 2^(s * k_mul - m) from unseeded scores.
  auto put_pair = [&](float2_t p, half8_t &hi, half8_t &lo, int at) {
    const half2_t ph = __builtin_convertvector(p, half2_t);
    hi[at] = ph[0];
    hi[at + 1] = ph[1];
    if constexpr (kTwoPartP) {
      const half2_t pl = __builtin_convertvector(p - __builtin_convertvector(ph, float2_t), half2_t);
      lo[at] = pl[0];
      lo[at + 1] = pl[1];
    }
  };
  auto exponentials_of = [&](const float4_t (&st)[2][CT], half8_t (&pk)[CT],
                             half8_t (&pk_lo)[CT], int u) {
    const float neg_m = -m_run[u];
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        put_pair(float2_t{fast_exp2(__builtin_fmaf(st[m][u][i], k_mul, neg_m)),
                          fast_exp2(__builtin_fmaf(st[m][u][i + 1], k_mul, neg_m))},
                 pk[u], pk_lo[u], 4 * m + i);
      }
    }
  };
  // Fast path: the scores were seeded with -m / k_mul, so they are the exponents up to that factor.
  auto exponentials_seeded = [&](const float4_t (&st)[2][CT], half8_t (&pk)[CT],
                                 half8_t (&pk_lo)[CT], int u) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        put_pair(float2_t{fast_exp2(st[m][u][i] * k_mul), fast_exp2(st[m][u][i + 1] * k_mul)}, pk[u],
                 pk_lo[u], 4 * m + i);
      }
    }
  };
  // One MFMA with the probabilities of a column tile (two where they come in two parts).
  auto mfma_p = [&](half8_t a, half8_t hi, half8_t lo, float4_t c) -> float4_t {
    c = mfma_16x16x32(a, hi, c);
    if constexpr (kTwoPartP) c = mfma_16x16x32(a, lo, c);
    return c;
  };
  // True if any probability of the sub-tile exceeds 2^kMaxP (or is not finite): the running maximum
  // is then too low for these keys and the sub-tile has to be redone with a rescale. Probabilities
  // are non-negative, so their fp16 bit patterns order like their values.
  auto overflowed = [&](const half8_t (&pk)[CT]) -> bool {
    // (`maximum` has a form of three packed operands, which the other maximum of fp16 pairs has not)
    auto pair = [&](int i) {
      const half8_t &p = pk[i / 4 % CT];
      return half2_t{p[2 * (i & 3)], p[2 * (i & 3) + 1]};
    };
    half2_t mx2 = pair(0);
#pragma unroll
    for (int i = 1; i < 4 * CT; i += 2) {
      mx2 = __builtin_elementwise_maximum(mx2, pair(i));
      if (i + 1 < 4 * CT) mx2 = __builtin_elementwise_maximum(mx2, pair(i + 1));
    }
    const uint32_t bits = __builtin_bit_cast(uint32_t, mx2);
    const uint32_t top = (bits & 0xffffu) > (bits >> 16) ? (bits & 0xffffu) : (bits >> 16);
    return __builtin_amdgcn_ballot_w64(top > (uint32_t)(15 + kMaxP) << 10) != 0;  // fp16 bits of 2^kMaxP
  };
  // O^T += V^T . P^T,  l += 1^T . P^T for keys 32 s2 .. +31 of the staged V tile.
  auto accumulate_sub = [&](int s2) {
#pragma unroll
    for (int u = 0; u < CT; ++u) dsum[u] = mfma_p(ones, pk[u], pk_lo[u], dsum[u]);
#pragma unroll
    for (int j = 0; j < kJTiles; ++j) {
      const uint32_t at = v_at(j) + 2u * 32 * s2 * kHD;
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t *)(uintptr_t)at);
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_short4_t *)(uintptr_t)(at + 2u * 16 * kHD));
      const short8_t both = short8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      const half8_t a = __builtin_bit_cast(half8_t, both);
#pragma unroll
      for (int u = 0; u < CT; ++u) acc[j][u] = mfma_p(a, pk[u], pk_lo[u], acc[j][u]);
    }
  };
  // V^T fragment j (A operand: d rows 16j.., keys 32 s2 + {4g..4g+3, 16+4g..}) of the staged tile.
  auto load_vfrag = [&](int j, int s2, uint32_t half) -> half8_t {
    const uint32_t at = v_at(j) + half + 2u * 32 * s2 * kHD;
    const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t *)(uintptr_t)at);
    const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (lds_short4_t *)(uintptr_t)(at + 2u * 16 * kHD));
    const short8_t both = short8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(half8_t, both);
  };
  auto scores_sub = [&](int s2) { scores_into(st, s2, std::false_type{}); };
  auto column_max = [&](int u) { return column_max_of(st, u); };
  auto exponentials = [&](int u) { exponentials_of(st, pk, pk_lo, u); };
  float4_t st1[2][CT];  // scores of the second half of a fast tile
  half8_t pk1[CT], pk1_lo[CT];

  // Publishes tile kt (already requested) and requests tile kt + 1 into the other half.
  auto sync_and_prefetch = [&](int kt, bool issue_next = true) {
    if constexpr (FP8) {
      // The codes of tile kt (requested a tile ago) become fp16 rows in its LDS half: 16-byte
      // chunk c of row r goes where the direct load of the fp16 path would have put it.
      const int r = sub + lane / kLanesPerRow;   // row inside the page: what the swizzle goes by
      const uint32_t row_at =
          (uint32_t)((kt & 1) * kTileHalfs + (kRowsPerWave * wave + lane / kLanesPerRow) * kHD) * 2u;
#pragma unroll
      for (int j = 0; j < kCodesPerLane / 8; ++j) {
        const int chunk = (kCodesPerLane / 8) * (lane % kLanesPerRow) + j;
        const uint4_t ck = raw_k[j >> 1], cv = raw_v[j >> 1];
        const half8_t kh = codes_to_half<KV>((j & 1) ? uint2_t{ck[2], ck[3]} : uint2_t{ck[0], ck[1]});
        const half8_t vh = codes_to_half<KV>((j & 1) ? uint2_t{cv[2], cv[3]} : uint2_t{cv[0], cv[1]});
        *(lds_half8_t *)(uintptr_t)(k_lds + row_at + 16u * (uint32_t)(chunk ^ k_swz(r))) = kh;
        *(lds_half8_t *)(uintptr_t)(v_lds + row_at + 16u * (uint32_t)(chunk ^ v_swz(r))) = vh;
      }
    }
    __builtin_amdgcn_s_waitcnt(wait_vm(0));  // this wavefront's part of tile kt is in LDS
    __syncthreads();                     // ... and everyone's; everyone is done with tile kt-1
    if (issue_next && kt + 1 < n_tiles) issue_tile(kt + 1);
  };
  // The same loads for a tile that lies wholly inside the sequence's keys, split in two steps so
  // that they can ride between MFMAs instead of leaving in one burst behind the barrier:
  // tile_bases() reads the page id (scalar), issue_rows(i) requests row group i of K and of V.
  const char *next_kbase = nullptr, *next_vbase = nullptr;
  uint32_t next_dst = 0;
  // The page ids of two tiles' eight pages, one per lane (lane l: page l % 8 of tiles kt, kt + 1), requested
  // behind the barrier of the tile before the first that needs them, whose MFMAs cover the trip: as a scalar
  // value read on the spot the id cost every tile a round trip to memory in front of its first MFMA. (In front
  // of a barrier it is waited for there, as it is once where the loop is entered. With the request in front of the
  // even tiles' barriers, eight prompts of 128 to 2048 tokens, 64 / 8 heads, two layers, took 673 us instead of 668, four
  // of 5000 to 8192 2724 instead of 2714.)
  auto page_ids_of_tiles = [&](int kt) -> int {
    if constexpr (!PAGED) return 0;
    int pidx = (tile0 + kt) * 4 + (lane & 7);
    pidx = pidx < last_page ? pidx : last_page;
    return page_of(pidx);
  };
  auto tile_bases = [&](int kt, int half, int ids, int first) {  // half: kt % 2; ids: lanes first .. first + 3 those of tile kt
    const int row0 = (tile0 + kt) * kKvTile + kRowsPerWave * wave;
    if (PAGED) {
      const int pid = __builtin_amdgcn_readlane(ids, first + (kRowsPerWave * wave) / 16);
      next_kbase = (const char *)paged.kv + (int64_t)pid * ((int64_t)kPageSize * k_pitch);
      next_vbase = next_kbase;
    } else {
      next_kbase = (const char *)packed.k + (int64_t)(q_start + row0) * k_pitch;
      next_vbase = (const char *)packed.v + (int64_t)(q_start + row0) * v_pitch;
    }
    next_dst = (uint32_t)(half * kTileHalfs + kRowsPerWave * wave * kHD) * 2u;
  };
  auto issue_rows = [&](int i) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(k_lds + next_dst + 1024u * i), "v"(koff[i]), "s"(next_kbase)
                 : "memory", "m0");
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(v_lds + next_dst + 1024u * i), "v"(voff[i]), "s"(next_vbase)
                 : "memory", "m0");
  };

  // General sub-tiles of tile kt from `first` on: causal mask, and the accumulators are rescaled
  // to the new running maximum unconditionally (straight-line code: a branch around the
  // rescale makes the compiler copy every accumulator at the join, on every tile). Used for the
  // first tile and wherever the fast loop saw a maximum grow.
  auto general_tile = [&](int kt, int first) {
#pragma unroll
    for (int s2 = 0; s2 < 2; ++s2) {
      const int key0 = (tile0 + kt) * kKvTile + 32 * s2;
      if (s2 < first) continue;
      if (key0 >= kv_end) break;  // nothing visible in the second half
      scores_sub(s2);
      // Masked only where a row of the block does not see all 32 keys: 64 vector instructions a tile that the first
      // tile and the upper half of the one at the diagonal do without (16 x 1024 tokens, 32 / 8 heads of 64, 126 -> 124 us,
      // 64 x 256 78 -> 75.5; 64 / 8 heads, eight prompts of 128 to 2048 691 -> 685).
      if (key0 + 31 > diag) {
#pragma unroll
        for (int u = 0; u < CT; ++u) mask_sub(u, key0);
      }
#pragma unroll
      for (int u = 0; u < CT; ++u) {
        const float m_new = vmax2(m_run[u], column_max(u) - (float)kMaxBias);
        const float alpha = fast_exp2(m_run[u] - m_new);
        m_run[u] = m_new;
        const float sd = -m_new * k_mul_inv;
        seed[u] = float4_t{sd, sd, sd, sd};
        dsum[u] *= alpha;
#pragma unroll
        for (int j = 0; j < kJTiles; ++j) acc[j][u] *= alpha;
        exponentials(u);
      }
      accumulate_sub(s2);
    }
  };

  // Fast tiles kt .. kt_end-1: they proceed only while no column maximum exceeds the running one
  // by more than 8 (6 at head dim 256; p stays below 2^kMaxP, inside fp16 and fp32 range), so the
  // accumulators are touched by nothing but MFMAs. Returns 0 at kt_end, else 1 + the sub-tile of tile kt that
  // has to be redone with a rescale.
  int kt = 1;
  auto fast_tiles = [&](int kt_end, auto masked_tag) -> int {
    constexpr bool MASKED = decltype(masked_tag)::value;
    for (; kt < kt_end; ++kt) {
      sync_and_prefetch(kt);
      flip_halves();
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int key0 = (tile0 + kt) * kKvTile + 32 * s2;
        if (MASKED && key0 >= kv_end) break;
        scores_into(st, s2, std::true_type{});
        if (MASKED && key0 + 31 > diag) {
#pragma unroll
          for (int u = 0; u < CT; ++u) mask_sub(u, key0);
        }
#pragma unroll
        for (int u = 0; u < CT; ++u) exponentials_seeded(st, pk, pk_lo, u);
        if (overflowed(pk)) return 1 + s2;
        accumulate_sub(s2);
      }
    }
    return 0;
  };

  // Fast tiles below the diagonal: both halves' scores first, one growth check, then the halves'
  // exponentials and second products, so that in each basic block MFMAs of one half can run
  // beside the vector ALU work of the other. Returns like fast_tiles (a grown tile is redone
  // from its first half).
  constexpr int kIssueEvery = kJTiles / kLoads;  // MFMA pairs between two row groups of the next tile
  // Two tiles an iteration, tile 2i + 1 in the second half of the staging area and tile 2i + 2 in the first: the halves
  // are offsets of the LDS reads, and neither the addresses nor the page ids cost vector instructions in each tile (14 fewer;
  // passes as above, 2825 -> 2802 us, 516 -> 509 the chunk over 7601 tokens, 592 -> 584 over int8, 324 -> 320 at 64). Taken
  // up at an odd tile; taken up and left with the addresses on the half of tile kt - 1, like fast_tiles, or where tile
  // kt is to be redone on its own.
  auto plain_tile = [&](auto half_tag, int ids, int &ids_next) -> int {  // ids: of the odd tile's kt + 1, kt + 2
    constexpr bool kOdd = decltype(half_tag)::value;
    constexpr uint32_t kAt = kOdd ? 2u * kTileHalfs : 0u;
    sync_and_prefetch(kt, FP8);
    if constexpr (!FP8) {
      tile_bases(kt + 1, kOdd ? 0 : 1, ids, kOdd ? 0 : 4);
      if constexpr (kOdd) ids_next = page_ids_of_tiles(kt + 3);
    }
    // Block 1: scores of both halves, the first half's exponentials beside the second half's
    // MFMAs, and the first half's V fragments requested before the block ends.
    // Region 1: all eight K fragments of the first half are requested at once.
    auto load_kfrag = [&](int s2, int i) -> half8_t {   // fragment i = (kk = i / 2, m = i % 2)
      return *(const lds_half8_t *)(uintptr_t)(k_at(i >> 1) + kAt + 2u * (32 * s2 + 16 * (i & 1)) * kHD);
    };
    half8_t kf[kJTiles];
#pragma unroll
    for (int i = 0; i < kJTiles; ++i) kf[i] = load_kfrag(0, i);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
#pragma unroll
      for (int u = 0; u < CT; ++u) st[m][u] = st1[m][u] = seed[u];
    }
    __builtin_amdgcn_sched_barrier(0);
    // Region 2: the first half's MFMAs; each fragment register takes the second half's
    // fragment once its pair is issued. Four accumulators in rotation: no MFMA waits for
    // the one before it.
    half8_t kf1[kJTiles];
#pragma unroll
    for (int i = 0; i < kJTiles; ++i) {
#pragma unroll
      for (int u = 0; u < CT; ++u) st[i & 1][u] = mfma_16x16x32(kf[i], qf[u][i >> 1], st[i & 1][u]);
      kf1[i] = load_kfrag(1, i);
      if constexpr (!FP8) {
        if (i % kIssueEvery == kIssueEvery - 1) issue_rows(i / kIssueEvery);
      }
    }
#pragma unroll
    for (int i = 0; i < kJTiles; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, CT, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (!FP8 && i % kIssueEvery == kIssueEvery - 1) __builtin_amdgcn_sched_group_barrier(0x020, 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    // Region 3: the second half's MFMAs beside the first half's exponentials; the first
    // half's V fragments are requested on the way.
    // (Head dim 256: the exponentials stand in front of the MFMAs in the source here and below; behind
    // them, the scheduler started them late and a tile took 3 % longer.)
    half8_t vf[kJTiles];
    if constexpr (kHD == 256) {
#pragma unroll
      for (int u = 0; u < CT; ++u) exponentials_seeded(st, pk, pk_lo, u);
    }
#pragma unroll
    for (int i = 0; i < kJTiles; ++i) {
#pragma unroll
      for (int u = 0; u < CT; ++u) st1[i & 1][u] = mfma_16x16x32(kf1[i], qf[u][i >> 1], st1[i & 1][u]);
      vf[i] = load_vfrag(i, 0, kAt);
    }
    if constexpr (kHD != 256) {
#pragma unroll
      for (int u = 0; u < CT; ++u) exponentials_seeded(st, pk, pk_lo, u);
    }
    const bool over_a = overflowed(pk);
#pragma unroll
    for (int i = 0; i < kJTiles; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, CT, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
    }
    if (over_a) return 1;
    // Block 2: second product of the first half beside the second half's exponentials; each
    // fragment register takes the second half's fragment as soon as its MFMAs are issued.
    half8_t vf2[kJTiles];
    if constexpr (kHD == 256) {
#pragma unroll
      for (int u = 0; u < CT; ++u) exponentials_seeded(st1, pk1, pk1_lo, u);
    }
#pragma unroll
    for (int u = 0; u < CT; ++u) dsum[u] = mfma_p(ones, pk[u], pk_lo[u], dsum[u]);
#pragma unroll
    for (int j = 0; j < kJTiles; ++j) {
#pragma unroll
      for (int u = 0; u < CT; ++u) acc[j][u] = mfma_p(vf[j], pk[u], pk_lo[u], acc[j][u]);
      vf2[j] = load_vfrag(j, 1, kAt);
    }
    if constexpr (kHD != 256) {
#pragma unroll
      for (int u = 0; u < CT; ++u) exponentials_seeded(st1, pk1, pk1_lo, u);
    }
    const bool over_b = overflowed(pk1);
#pragma unroll
    for (int i = 0; i < kJTiles; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, kTwoPartP ? 2 * CT : CT, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, kTwoPartP ? 2 * CT : CT, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 8, 0);
    if (over_b) return 2;
    // Block 3: second product of the second half.
#pragma unroll
    for (int u = 0; u < CT; ++u) dsum[u] = mfma_p(ones, pk1[u], pk1_lo[u], dsum[u]);
#pragma unroll
    for (int j = 0; j < kJTiles; ++j) {
#pragma unroll
      for (int u = 0; u < CT; ++u) acc[j][u] = mfma_p(vf2[j], pk1[u], pk1_lo[u], acc[j][u]);
    }
    return 0;
  };
  auto fast_plain_tiles = [&](int kt_end) -> int {
    int ids = 0;  // of tiles kt + 1, kt + 2
    if constexpr (!FP8) {
      if (kt < kt_end) ids = page_ids_of_tiles(kt + 1);
    }
    while (kt < kt_end) {
      int ids_next = 0;
      int grew = plain_tile(std::true_type{}, ids, ids_next);
      if (grew == 0) ++kt;
      if (grew != 0 || kt >= kt_end) {
        flip_halves();
        return grew;
      }
      grew = plain_tile(std::false_type{}, ids, ids_next);
      if (grew != 0) return grew;
      ++kt;
      ids = ids_next;
    }
    return 0;
  };

  {
    // Tiles whose last key is at or below the block's first row need no mask.
    int n_plain = (diag + 1) / kKvTile - tile0;
    n_plain = n_plain < n_tiles ? n_plain : n_tiles;
    sync_and_prefetch(0);
    general_tile(0, 0);
    while (kt < n_tiles) {
      int n_spread = (last_key + 1) / kKvTile - 1 - tile0;   // tiles kt < n_spread: tile kt + 1 is full
      n_spread = n_spread < n_tiles - 1 ? n_spread : n_tiles - 1;
      n_spread = n_spread < n_plain ? n_spread : n_plain;
      // (an even tile, behind one that was redone, goes the other way too)
      int grew = kt & 1 ? fast_plain_tiles(n_spread) : 0;
      if (grew == 0) grew = fast_tiles((kt & 1) == 0 && kt < n_spread ? kt + 1 : n_tiles, std::true_type{});
      if (grew != 0) {
        general_tile(kt, grew - 1);
        ++kt;
      }
    }
  }

  if constexpr (KG == 2) {
    // Each group finishes one of a wavefront's two column tiles: it hands the other's accumulators,
    // denominators and maxima to the wavefront of the same columns in the other group, through the
    // staging area, and folds in what it is given.
    typedef __attribute__((address_space(3))) float4_t lds_float4_t;
    typedef __attribute__((address_space(3))) float lds_float_t;
    for (int i = n_tiles > 1 ? n_tiles : 1; i < wg_barriers; ++i) __syncthreads();
    __syncthreads();  // every wavefront is done with its last tile
    constexpr uint32_t kHandBytes = 64 * (16 * kJTiles + 8);  // per wavefront: [kJTiles][64] float4, then [2][64] floats
    constexpr int kOutPitch = 2 * kHD + 16;
    static_assert(2 * W * (kHandBytes + 16 * kOutPitch) <= 2 * tile_lds_bytes<W>(), "fits the staging area");
    const uint32_t give = lds_base + (uint32_t)wave_in_wg * kHandBytes;
    const uint32_t take = lds_base + (uint32_t)(wave_in_wg ^ W) * kHandBytes;
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      if (u != kgroup) {
#pragma unroll
        for (int j = 0; j < kJTiles; ++j) *(lds_float4_t *)(uintptr_t)(give + 1024u * j + 16u * lane) = acc[j][u];
        *(lds_float_t *)(uintptr_t)(give + 1024u * kJTiles + 4u * lane) = dsum[u][0];
        *(lds_float_t *)(uintptr_t)(give + 1024u * kJTiles + 256u + 4u * lane) = m_run[u];
      }
    }
    __syncthreads();
    const float d_in = *(const lds_float_t *)(uintptr_t)(take + 1024u * kJTiles + 4u * lane);
    const float m_in = *(const lds_float_t *)(uintptr_t)(take + 1024u * kJTiles + 256u + 4u * lane);
    const float m_own = kgroup ? m_run[1] : m_run[0];
    const float d_own = kgroup ? dsum[1][0] : dsum[0][0];
    const float m_all = vmax2(m_own, m_in);  // finite: the second group's rows all see a key
    const float w_own = fast_exp2(m_own - m_all), w_in = fast_exp2(m_in - m_all);
    const float inv = v_scale / (d_own * w_own + d_in * w_in);
    const uint32_t mine = lds_base + 2u * W * kHandBytes + (uint32_t)(wave_in_wg * 16 * kOutPitch);
#pragma unroll
    for (int j = 0; j < kJTiles; ++j) {
      const float4_t in = *(const lds_float4_t *)(uintptr_t)(take + 1024u * j + 16u * lane);
      const float4_t own = kgroup ? acc[j][1] : acc[j][0];
      half4_t o;
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = (half_t)((own[i] * w_own + in[i] * w_in) * inv);
      *(__attribute__((address_space(3))) half4_t *)(uintptr_t)(mine + (uint32_t)(n * kOutPitch + 8 * g) + 32u * j) = o;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int t = wave * CT + kgroup;
    const int head = t / row_tiles;
    const int row0 = m0 + (t - head * row_tiles) * 16;
    half_t *o_tile = out + (int64_t)(q_start + row0) * out_stride + (int64_t)(h * group + head0 + head) * kHD + 8 * slot;
#pragma unroll
    for (int step = 0; step < kLoadsPerWave; ++step) {
      const int r = kRowsPerLoad * step + r_loc;
      const half8_t row = *(const lds_half8_t *)(uintptr_t)(mine + (uint32_t)(r * kOutPitch + 16 * slot));
      if (head < heads_here && row0 + r < q_len) *(half8_t *)(o_tile + (int64_t)r * out_stride) = row;
    }
    return;
  }
  if constexpr (!SHARED && !KSPLIT) {
    // The accumulators hold O^T: a lane has 4 consecutive d of one row, so stored directly every
    // store instruction would touch 16 rows with 32 bytes each. The rows go through LDS instead
    // (the K/V tiles are done with) and leave as whole 256-byte rows, 4 rows per instruction.
    constexpr int kOutPitch = 2 * kHD + 16;  // bytes; at 128: 68 dwords, a half-wave's 8-byte writes hit 64 banks
    __syncthreads();                              // every wavefront is done reading the last tile
    const uint32_t mine = kHD == 256 ? k_lds + (uint32_t)wave * kOwnLds
                                     : ((wave & 2) ? v_lds : k_lds) + (uint32_t)((wave & 1) * CT * 16 * kOutPitch);
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      const float inv = v_scale / dsum[u][0];
      const uint32_t at = mine + (uint32_t)((u * 16 + n) * kOutPitch + 8 * g);
#pragma unroll
      for (int j = 0; j < kJTiles; ++j) {
        *(__attribute__((address_space(3))) half4_t *)(uintptr_t)(at + 32u * j) =
            half4_t{(half_t)(acc[j][u][0] * inv), (half_t)(acc[j][u][1] * inv),
                    (half_t)(acc[j][u][2] * inv), (half_t)(acc[j][u][3] * inv)};
      }
    }
    // lane l carries chunk l % kChunks of row l / kChunks + kRowsPerLoad * step
    const int chunk = slot, r4 = r_loc;
    // Head dim 256: not 0 (but not a number) once an output of the tile was not finite
    float odd[CT] = {};
#pragma unroll
    for (int u = 0; u < CT; ++u) {
#pragma unroll
      for (int step = 0; step < kLoadsPerWave; ++step) {
        const int r = kRowsPerLoad * step + r4;
        const half8_t row = *(const lds_half8_t *)(uintptr_t)(mine + (uint32_t)((u * 16 + r) * kOutPitch + 16 * chunk));
        const int t = wave * CT + u;
        const int head = t / row_tiles;
        const int qrow_idx = m0 + (t - head * row_tiles) * 16 + r;
        if (head < heads_here && qrow_idx < q_len) {
          *(half8_t *)(out + (int64_t)(q_start + qrow_idx) * out_stride + (int64_t)out_head[u] * kHD +
                       8 * chunk) = row;
        }
        if constexpr (kHD == 256) {
#pragma unroll
          for (int i = 0; i < 8; i += 2) {
            odd[u] = __builtin_amdgcn_fdot2(half2_t{row[i], row[i + 1]}, half2_t{0, 0}, odd[u], false);
          }
        }
      }
    }
    if constexpr (kHD == 256) {
      // A tile with an output that is not finite is attended again row by row, over what was just
      // written. An infinite value times a probability of 0 -- of a row that may not see its key, or
      // the second part of a probability that fp16 holds exactly -- is NaN above and must not be.
      // (Looking is a v_dot2_f32_f16 for two outputs on the way to their store: nothing to measure.)
      if (__builtin_expect(__builtin_amdgcn_ballot_w64(odd[0] + odd[CT - 1] != 0.f) != 0, false)) {
        __builtin_amdgcn_s_waitcnt(wait_vm(0));  // the rows' first stores come first
#pragma unroll 1
        for (int u = 0; u < CT; ++u) {
          tile_by_rows<FP8 ? KV : kKvF16, PAGED, kByRows>(mine, q, q_stride, out, out_stride, paged, packed, b, q_start, q_len, ctx,
                                                 m0, wave * CT + u, row_tiles, head0, heads_here, group, h, scale_log2);
        }
      }
    }
    return;
  }
  if constexpr (SHARED || KSPLIT) {
    // The partial rows (fp32, normalised) leave as whole rows like the output of a prefill block:
    // a lane holds 4 consecutive elements of each of its column's 16-element groups, so stored
    // straight from registers one instruction would touch 16 rows with 64 bytes each. One column
    // tile at a time goes through this wavefront's part of the K/V staging area (the tiles are
    // done with) and leaves 1 KiB per instruction.
    constexpr int kPartPitch = 4 * kHD + 16;           // bytes; rows 4 banks apart: a 16-lane group's writes hit 64 banks
    constexpr int kRowLanes = kHD / 4;                 // lanes that carry one row (16 bytes each)
    constexpr int kRowsPerStore = kWave / kRowLanes;   // rows one store instruction writes
    __syncthreads();                                   // every wavefront is done reading the last tile
    const uint32_t mine = k_lds + (uint32_t)(wave * 16 * kPartPitch);
    typedef __attribute__((address_space(3))) float4_t lds_float4_t;
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      const float inv = v_scale / dsum[u][0];
      // the partial row of this lane's column (the same in its four lane groups), or -1
      const int piece = SHARED ? block_z : key_slice;  // which partial of the row this block writes
      const int cell = out_row[u] >= 0
                           ? (piece * prefix.batch + out_row[u]) * prefix.num_q_heads + out_head[u]
                           : -1;
      if (g == 0 && cell >= 0) {
        // read once, by the merge launch: streaming stores (see store_state in paged_decode.hip)
        __builtin_nontemporal_store((m_run[u] + fast_log2(dsum[u][0])) * 0.6931471805599453f,
                                    prefix.part_lse + cell);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");   // the reads of the tile before are done
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int j = 0; j < kJTiles; ++j) {
        *(lds_float4_t *)(uintptr_t)(mine + (uint32_t)(n * kPartPitch + 4 * (16 * j + 4 * g))) =
            float4_t{acc[j][u][0] * inv, acc[j][u][1] * inv, acc[j][u][2] * inv, acc[j][u][3] * inv};
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int step = 0; step < 16 / kRowsPerStore; ++step) {
        const int r = kRowsPerStore * step + lane / kRowLanes;      // column of the tile = row staged
        const int c = lane % kRowLanes;
        const int row_cell = __shfl(cell, r, kWave);
        const float4_t x = *(const lds_float4_t *)(uintptr_t)(mine + (uint32_t)(r * kPartPitch + 16 * c));
        if (row_cell >= 0) {
          __builtin_nontemporal_store(x, (float4_t *)(prefix.part_o + (int64_t)row_cell * kHD + 4 * c));
        }
      }
    }
    return;
  }
#pragma unroll
  for (int u = 0; u < CT; ++u) {
    const float inv = v_scale / dsum[u][0];
    if (out_row[u] >= 0) {
      half_t *o = out + (int64_t)out_row[u] * out_stride + (int64_t)out_head[u] * kHD + 4 * g;
#pragma unroll
      for (int j = 0; j < kJTiles; ++j) {
        *(half4_t *)(o + 16 * j) =
            half4_t{(half_t)(acc[j][u][0] * inv), (half_t)(acc[j][u][1] * inv),
                    (half_t)(acc[j][u][2] * inv), (half_t)(acc[j][u][3] * inv)};
      }
    }
  }
}

// CT: column tiles per wavefront. One instead of two, 64 score columns a workgroup, for launches that would
// leave most of the device idle (see narrow_fits in paged_prefill.hip). Bound by the chain of its few key tiles.
template <int MODE, int CT = prefill_ct(MODE)>
__global__ __launch_bounds__(prefill_waves(MODE) * kWave, kWgPerCu *prefill_waves(MODE) / kTiledWaves) void varlen_prefill_tiled_kernel(
    const half_t *__restrict__ q, int64_t q_stride, half_t *__restrict__ out, int64_t out_stride,
    PagedSource paged, PackedSource packed, PrefixTask prefix,
    const int32_t *__restrict__ q_starts_or_cu, const int32_t *__restrict__ q_lens_or_null,
    const int32_t *__restrict__ context_lens, int32_t group, int32_t head_splits,
    int32_t heads_per_wg, int32_t row_tiles, float scale_log2, int32_t key_slices) {
  __shared__ __attribute__((aligned(1024))) half_t lds_all[tile_lds_bytes<prefill_waves(MODE)>() / 2];
  if constexpr (MODE == kPagedPrefillSplit || MODE == kPagedPrefillSplitFp8 ||
                MODE == kPagedPrefillSplitInt8) {
    // blockIdx.y = row block * key_slices + slice: the slices of a block are neighbours
    const int by = (int)blockIdx.y / key_slices;
    prefill_tile_body<MODE, prefill_waves(MODE), 1, CT>((uint32_t)(uintptr_t)(lds_half_t *)lds_all, (int)blockIdx.x, by,
                               (int)blockIdx.z, (int)gridDim.y / key_slices, q, q_stride, out, out_stride,
                               paged, packed, prefix, q_starts_or_cu, q_lens_or_null, context_lens, group,
                               head_splits, heads_per_wg, row_tiles, scale_log2,
                               (int)blockIdx.y - by * key_slices, key_slices);
  } else {
    prefill_tile_body<MODE, prefill_waves(MODE), 1, CT>((uint32_t)(uintptr_t)(lds_half_t *)lds_all, (int)blockIdx.x, (int)blockIdx.y,
                               (int)blockIdx.z, (int)gridDim.y, q, q_stride, out, out_stride, paged, packed,
                               prefix, q_starts_or_cu, q_lens_or_null, context_lens, group, head_splits,
                               heads_per_wg, row_tiles, scale_log2);
  }
}

// The same for a launch of no more workgroups than compute units: eight wavefronts, two groups of four
// that attend half of the block's keys each (see KG in prefill_tile_body). One workgroup of four on a
// compute unit is a lone wavefront per SIMD, whose softmax and barrier waits nothing covers; this gives
// every SIMD two and halves the chain of tiles. The groups meet in LDS, where key slices (separate
// workgroups) pay for partial rows in memory and a merge launch. One request's chunk of 512 rows, 64 / 8
// heads, over 7601 cached tokens: 159 -> 132 us (826 -> 994 TFLOP/s); 1008 rows, 32 / 8 heads of 64, over 7177: 105 ->
// 89; 256 workgroups, 64 / 8 heads: 1.1 us a key tile with one group, 1.0 with two. Bound by the tile loop's
// instruction mix, as the launch of many workgroups is.
template <int MODE>
__global__ __launch_bounds__(2 * kTiledWaves *kWave, 2) void varlen_prefill_two_group_kernel(
    const half_t *__restrict__ q, int64_t q_stride, half_t *__restrict__ out, int64_t out_stride,
    PagedSource paged, PackedSource packed, PrefixTask prefix,
    const int32_t *__restrict__ q_starts_or_cu, const int32_t *__restrict__ q_lens_or_null,
    const int32_t *__restrict__ context_lens, int32_t group, int32_t head_splits,
    int32_t heads_per_wg, int32_t row_tiles, float scale_log2, int32_t) {
  __shared__ __attribute__((aligned(1024))) half_t lds_all[tile_lds_bytes<kTiledWaves>()];  // two staging areas
  prefill_tile_body<MODE, kTiledWaves, 2>((uint32_t)(uintptr_t)(lds_half_t *)lds_all, (int)blockIdx.x, (int)blockIdx.y,
                             (int)blockIdx.z, (int)gridDim.y, q, q_stride, out, out_stride, paged, packed,
                             prefix, q_starts_or_cu, q_lens_or_null, context_lens, group, head_splits,
                             heads_per_wg, row_tiles, scale_log2);
}

}  // namespace prefill_tile
}  // namespace LITEKV_HD_NS
}  // namespace litekv
