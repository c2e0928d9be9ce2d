// Host side of the varlen causal prefill and of the shared-prefix pass of a decode step: argument
// checks, launch shapes and the C ABI. The kernel is in prefill_tile.h.
#include "prefill_tile.h"

namespace litekv {
inline namespace LITEKV_HD_NS {
using namespace prefill_tile;

static int validate_prefill(const char *what, const void *q, int64_t q_stride, const void *out,
                            int64_t out_stride, int32_t batch, int32_t hq, int32_t hkv,
                            int32_t head_dim, int32_t max_q_len) {
  LITEKV_REQUIRE(batch >= 0 && batch <= 65535, "%s: batch %d out of [0, 65535]", what, batch);
  LITEKV_REQUIRE(head_dim == kHD, "%s: head_dim %d unsupported (32, 64, 128 or 256)", what,
                 head_dim);
  LITEKV_REQUIRE(hq > 0 && hkv > 0 && hq % hkv == 0 && hq <= 65535,
                 "%s: num_q_heads %d / num_kv_heads %d invalid", what, hq, hkv);
  LITEKV_REQUIRE(hq / hkv <= kMaxGroup, "%s: %d query heads per kv head unsupported (max %d)", what,
                 hq / hkv, kMaxGroup);
  LITEKV_REQUIRE(max_q_len >= 0, "%s: max_q_len %d < 0", what, max_q_len);
  if (batch == 0 || max_q_len == 0) return LITEKV_OK;
  LITEKV_REQUIRE(q && out, "%s: null pointer", what);
  LITEKV_REQUIRE(aligned16(q) && aligned16(out), "%s: q and out must be 16-byte aligned", what);
  const int64_t row = (int64_t)hq * head_dim;
  LITEKV_REQUIRE(q_stride >= row && q_stride % 8 == 0 && out_stride >= row && out_stride % 8 == 0,
                 "%s: token strides (%lld, %lld) invalid", what, (long long)q_stride,
                 (long long)out_stride);
  // q rows are staged with 32-bit byte offsets from the block's first row
  LITEKV_REQUIRE(q_stride < (1 << 25), "%s: q token stride %lld too large", what, (long long)q_stride);
  return LITEKV_OK;
}

// Whether a 256-wide prefill goes to the tiled kernel: all of them but rows it cannot address
// (16-byte stores of the output, 32-bit offsets into q) and scales its arithmetic is not made for
// (tile_scale: 0, below 0, not a number), which stay with the general kernel. Four prompts of 300
// to 2048 tokens, 16 / 4 heads: 9198 us there, without matrix instructions and with every K row
// read by one lane at a time, 76 us here.
[[maybe_unused]] static bool tiled_256(int64_t q_stride, int64_t out_stride, int32_t num_kv_heads,
                                       float softmax_scale) {
  return q_stride < (1 << 25) && out_stride % 8 == 0 && num_kv_heads <= 1024 &&
         tile_scale(softmax_scale * kLog2eP);
}

// How a GQA group of `group` heads is cut into workgroups.
struct PrefillShape {
  int head_splits, heads_per_wg, row_tiles;
  unsigned row_blocks;
};
static PrefillShape prefill_shape(int group, int max_q_len, int wg_col_tiles = kWgColTiles) {
  PrefillShape s;
  s.head_splits = (group + wg_col_tiles - 1) / wg_col_tiles;
  s.heads_per_wg = (group + s.head_splits - 1) / s.head_splits;
  s.row_tiles = wg_col_tiles / s.heads_per_wg;
  s.row_blocks = (unsigned)((max_q_len + 16 * s.row_tiles - 1) / (16 * s.row_tiles));
  return s;
}

// Folds the key slices of a split prefill: one wavefront per (query row, head) reads the row's
// `slices` log-sum-exps and partial rows (fp32, normalised per slice) and writes the fp16 row.
// A slice without keys has log-sum-exp -inf and weight 0; the last slice always has keys.
__global__ __launch_bounds__(4 * kWave) void prefill_split_merge_kernel(
    const float *__restrict__ part_o, const float *__restrict__ part_lse, half_t *__restrict__ out,
    int64_t out_stride, int64_t num_tokens, int32_t num_q_heads, int32_t slices) {
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t id = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (id >= num_tokens * num_q_heads) return;  // whole wavefronts
  const int64_t token = id / num_q_heads;
  const int head = (int)(id - token * num_q_heads);
  const int64_t piece_stride = num_tokens * num_q_heads;  // cells between the slices of a row
  const float l = lane < slices ? part_lse[lane * piece_stride + id] : -INFINITY;
  float mx = l;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, xor_lane(mx, off));
  const float w = lane < slices ? fast_exp2((l - mx) * 1.4426950408889634f) : 0.f;
  float den = w;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) den += xor_lane(den, off);
  if (2 * lane >= kHD) return;
  float o0 = 0.f, o1 = 0.f;
  for (int sidx = 0; sidx < slices; ++sidx) {  // in slice order: the sum does not depend on timing
    const float ws = __shfl(w, sidx, kWave);
    const float2 r = *(const float2 *)(part_o + (sidx * piece_stride + id) * kHD + 2 * lane);
    o0 += ws * r.x;
    o1 += ws * r.y;
  }
  const float inv = 1.0f / den;
  typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
  *(half2_t *)(out + token * out_stride + (int64_t)head * kHD + 2 * lane) =
      half2_t{(half_t)(o0 * inv), (half_t)(o1 * inv)};
}

static size_t prefill_split_workspace_bytes(int64_t num_tokens, int32_t num_q_heads, int32_t key_slices) {
  if (num_tokens <= 0 || num_q_heads <= 0 || key_slices <= 1) return 0;
  return (size_t)key_slices * (size_t)num_tokens * (size_t)num_q_heads * (kHD + 1) * sizeof(float);
}

// Compute units of the current device.
static int device_cus() {
  static thread_local int cached_device = -1, cached_cus = 0;  // compute units of the current device
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = -2;
  if (dev != cached_device) {
    int cus = 0;
    if (dev < 0 || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0) {
      cus = 256;
    }
    cached_device = dev;
    cached_cus = cus;
  }
  return cached_cus;
}

// Whether the blocks of a launch of `wgs` workgroups (counted as if every sequence had max_q_len rows, in
// `row_blocks` blocks) whose rows see up to `max_keys` keys are attended by two groups of wavefronts each
// (varlen_prefill_two_group_kernel): where a workgroup would have its compute unit to itself, the narrow
// form does not take it, and half of the key tiles saves more than the larger workgroup and the meeting of
// the groups cost. That is from 10 tiles on; over codes, whose conversion the groups share, from 4; where
// a sequence has one or two blocks of 128-wide fp16 rows and the launch streams its K and V, from 24. Time with
// two groups / one, 136 to 256 workgroups, 1 to 32 sequences, 64 / 8, 16 / 8 and 32 / 4 heads: 4 tiles 0.97 to 1.04
// (fp8 0.94 to 0.99), 9 1.01 to 1.04 (0.95 to 0.97), 10 0.96 to 1.02, 16 0.92 to 0.98, 32 0.88 to 0.95, 128 0.85 to
// 0.94; one or two blocks a sequence: 9 1.03 to 1.09, 16 0.96 to 1.03, 24 0.94 to 1.00; 32 / 8 heads of 64: 9 1.00 to 1.03,
// 10 0.94 to 0.98, 128 0.79 to 0.91. (The width of a block table says little about the keys: 8 chunks of 64 rows,
// nothing cached, in a table of 2048 pages took 8.2 us in two groups, 6.6 in one.)
static bool two_key_groups(int64_t wgs, unsigned row_blocks, int64_t max_keys, bool codes) {
  const int from = codes ? 4 : kHD == 128 && row_blocks <= 2 ? 24 : 10;
  return kHD != 256 && max_keys > (from - 1) * kKvTile && wgs <= device_cus();
}

// Whether a launch of `wgs` workgroups of 128 columns runs with 64 columns a workgroup, one column tile
// per wavefront, instead: where that still leaves at most one workgroup per compute unit. Twice as many
// wavefronts with half of a key tile's products and exponentials each, and less to load, normalise and store around
// them: 0.68 to 0.95 of the time with 128 columns (32 to 128 workgroups, 1 to 128 key tiles, the layouts above). One
// request, us with 128 columns and with 64: 203 rows of a fresh prompt, 16 / 8 heads, 9.2, 7.6; 64 rows, 64 / 8 heads,
// 5.3, 4.4; 128 rows over 2048 tokens 40.1, 30.5; 32 / 8 heads of 64, 256 rows 7.3, 5.8. With more
// workgroups the K and V tiles staged twice cost as much as that saves (400 rows, 64 / 8 heads: 200 workgroups).
static bool narrow_fits(int64_t wgs) {
  return kHD != 256 && 2 * wgs <= device_cus();
}

// Whether narrow workgroups would bring K and V in from memory twice at a cost: those of more than 4 heads per kv
// head share the heads of a block, not its rows, and land on different XCDs, so where every sequence has one block
// (of 128-wide fp16 rows) nothing else keeps its K and V near. From 7/16 of the compute units and 13 key tiles a
// workgroup on (or where nobody says how many, 0) that costs more than the rest saves: 16 rows a sequence, 64 / 8
// heads, time with 64 columns / with 128: 112 workgroups 16 tiles 0.97, 64 tiles 1.05, 128 workgroups 12 tiles 1.00, 16
// 1.05, 32 1.12 (41 us with 128); 96 workgroups 0.82 to 0.96; 16 / 8 heads 0.84 to 0.96, codes and rows of 64 0.73 to
// 0.87. In 8 key slices, two sequences of 30 000 tokens: 77.3 us with 128 columns, 84.1 with 64.
static bool narrow_reads_twice(int64_t wgs, int group, unsigned row_blocks, int64_t max_keys, bool codes) {
  return kHD == 128 && !codes && group > kTiledWaves && row_blocks == 1 && 16 * wgs >= 7 * device_cus() &&
         (max_keys <= 0 || max_keys > 12 * kKvTile);
}

// Key slices for a paged prefill whose row blocks alone would not fill the device, if the longest
// row sees `max_kv_len` keys: the count (at most kMaxPrefillKeySlices) with the smallest estimated
// time, 1 (do not split) unless that is at least 5 % less than unsplit. The estimate, in
// microseconds, head dim 128 (fits to one request's chunk of 64 to 512 rows over 0 to 32k cached
// tokens, 64 query / 8 kv heads): a workgroup walks max_kv_len / 64 / n key tiles at 1.0 us each
// while it has its compute unit to itself (0.75 us with 64 columns, narrow_fits; 0.95 uncut in two groups of
// wavefronts, two_key_groups) and at 1.7 us once the launch has more workgroups than compute units (two share
// one), times the rounds the launch needs on the device's resident slots; a cut costs the merge launch, 6 us, and
// a partial row (fp32) written and read back per query row, head and slice at 6 MB/us. Rows of 64: 0.6 us a
// tile with 64 columns as with 128 (priced at 0.45, chunks of 8 to 64 rows over 1000 tokens were left uncut: 12.1 us, 8.6
// in eight slices; over int8 15.7, 8.9). Over 1121 shapes (8 to 512 rows, 200 to 30 000 tokens, 1 to 4 chunks, the
// layouts above and 32 / 8 heads of 64, codes among them) the choice takes 1.019 times as long as the best count, rows of
// 64 1.020 (1.042 before). (One chunk over 30 000
// tokens, plain against sliced:
// 128 rows 364 -> 148 us, 256 rows 388 -> 269 us, 512 rows 480 -> 485 us; 128 rows over 2048 tokens
// 30.5 -> 25.5 us in four slices; 512 rows over 2048 tokens in two slices 48 -> 62 us and 128 rows of a
// fresh prompt in eight 14 -> 29 us, which the estimate rules out.)
static int32_t prefill_key_slices(int32_t batch, int32_t num_q_heads, int32_t num_kv_heads,
                                  int32_t max_q_len, int64_t max_kv_len) {
  if (batch <= 0 || num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads != 0 ||
      max_q_len <= 0 || max_kv_len <= 0 || num_q_heads / num_kv_heads > kMaxGroup) {
    return 1;
  }
  const PrefillShape s = prefill_shape(num_q_heads / num_kv_heads, max_q_len);
  const int64_t wgs = (int64_t)num_kv_heads * s.head_splits * s.row_blocks * batch;
  const int64_t cus = device_cus();
  const int64_t slots = cus * kWgPerCu;
  if (2 * wgs > slots) return 1;
  const double tile_us = kHD == 64 ? 0.6 : 1.0;
  const double tiles = (double)((max_kv_len + kKvTile - 1) / kKvTile);
  const double partial_us = (double)batch * max_q_len * num_q_heads * (kHD + 1) * 2.0 * sizeof(float) / 6.0e6;
  auto estimate = [&](int64_t n) {
    const int64_t resident = wgs * n;
    const double per_tile = narrow_fits(resident) ? (kHD == 64 ? 1.0 : 0.75) * tile_us
                            : n == 1 && two_key_groups(resident, s.row_blocks, max_kv_len, false) ? 0.95 * tile_us
                            : resident <= cus ? tile_us
                                              : 1.7 * tile_us * (double)((resident + slots - 1) / slots);
    return tiles / (double)n * per_tile + (n > 1 ? 6.0 + partial_us * (double)n : 0.0);
  };
  const double unsplit = estimate(1);
  int64_t best = 1;
  double best_us = 0.95 * unsplit;
  for (int64_t n = 2; n <= kMaxPrefillKeySlices; ++n) {
    const double t = estimate(n);
    if (t < best_us) {
      best = n;
      best_us = t;
    }
  }
  return (int32_t)best;
}

// Causal chunk attention over paged KV; `kv_scales` selects the fp8 pool.
static int launch_paged_prefill(const char *what, const void *q, int64_t q_token_stride,
                                const void *kv_pool, const float *kv_scales,
                                const int32_t *block_table, int32_t block_table_stride,
                                const int32_t *cu_q_lens, const int32_t *context_lens, void *out,
                                int64_t out_token_stride, int32_t batch, int32_t num_q_heads,
                                int32_t num_kv_heads, int32_t head_dim, int32_t page_size,
                                int64_t num_pages, int32_t max_q_len, float softmax_scale,
                                void *stream, int format, const PrefillKeySplit &split) {
  const bool fp8 = format != kKvF16;  // a pool of 8-bit codes
  LITEKV_REQUIRE(split.key_slices >= 1 && split.key_slices <= kMaxPrefillKeySlices,
                 "%s: key_slices %d out of [1, %d]", what, split.key_slices, kMaxPrefillKeySlices);
  LITEKV_REQUIRE(split.key_slices == 1 || head_dim == 128 || head_dim == 64,
                 "%s: key slices take head_dim 64 or 128", what);
#if LITEKV_HD == 128
  const PrefillBuild *build = head_dim == 64 ? &hd64_prefill()
                              : head_dim == 256 && tiled_256(q_token_stride, out_token_stride, num_kv_heads,
                                                                 softmax_scale)
                                  ? &hd256_prefill()
                                  : nullptr;
  if (build != nullptr) {  // another head dim's build of this file
    return build->paged(what, q, q_token_stride, kv_pool, kv_scales, block_table, block_table_stride, cu_q_lens,
                        context_lens, out, out_token_stride, batch, num_q_heads, num_kv_heads, head_dim,
                        page_size, num_pages, max_q_len, softmax_scale, stream, format, split);
  }
#endif
  if (head_dim != kHD && generic_head_dim(head_dim)) {  // see generic_attention.hip
    LITEKV_REQUIRE(max_q_len >= 0, "%s: max_q_len %d < 0", what, max_q_len);
    LITEKV_REQUIRE(batch == 0 || max_q_len == 0 || (kv_pool && block_table && cu_q_lens),
                   "%s: null pointer", what);
    LITEKV_REQUIRE(!fp8 || kv_scales, "%s: null pointer (kv_scales)", what);
    GenericLaunch g;
    g.q = q;
    g.q_row_stride = q_token_stride;
    g.out = out;
    g.out_row_stride = out_token_stride;
    g.kv_pool = const_cast<void *>(kv_pool);
    g.scales = kv_scales;
    g.format = format;
    g.block_table = block_table;
    g.bt_stride = block_table_stride;
    g.page_size = page_size;
    g.num_pages = num_pages;
    g.cu_q_lens = cu_q_lens;
    g.context_lens = context_lens;
    g.batch = batch;
    g.rows_per_seq = max_q_len;
    g.num_q_heads = num_q_heads;
    g.num_kv_heads = num_kv_heads;
    g.head_dim = head_dim;
    g.softmax_scale = softmax_scale;
    g.stream = stream;
    return launch_generic_attention(what, g);
  }
  int rc = validate_prefill(what, q, q_token_stride, out, out_token_stride, batch, num_q_heads,
                            num_kv_heads, head_dim, max_q_len);
  if (rc != LITEKV_OK) return rc;
  const int page_shift = page_shift_of(page_size);
  LITEKV_REQUIRE(page_shift >= 0, "%s: page_size %d unsupported (16, 32, 64, 128 or 256)", what, page_size);
  if (batch == 0 || max_q_len == 0) {
    clear_error();
    return LITEKV_OK;
  }
  LITEKV_REQUIRE(kv_pool && block_table && cu_q_lens, "%s: null pointer", what);
  LITEKV_REQUIRE(!fp8 || kv_scales, "%s: null pointer (kv_scales)", what);
  LITEKV_REQUIRE(aligned16(kv_pool), "%s: kv_pool must be 16-byte aligned", what);
  LITEKV_REQUIRE(block_table_stride >= 1, "%s: block_table_stride %d < 1", what, block_table_stride);
  LITEKV_REQUIRE(num_pages >= 1 && num_pages <= 0x7fffffffLL / page_size,
                 "%s: num_pages %lld out of range", what, (long long)num_pages);
  LITEKV_REQUIRE(num_kv_heads <= 1024, "%s: num_kv_heads %d > 1024", what, num_kv_heads);
  PagedSource paged{static_cast<const half_t *>(kv_pool), block_table, block_table_stride,
                    num_kv_heads, (int32_t)num_pages, kv_scales, page_shift};
  PackedSource packed{nullptr, nullptr, 0, 0, nullptr};
  const int group = num_q_heads / num_kv_heads;
#if LITEKV_HD != 256
  if (split.key_slices > 1) {
    // every block's keys in key_slices runs of tiles, one workgroup each, then the merge
    const int slices = split.key_slices;
    const int64_t rows = split.num_tokens;
    LITEKV_REQUIRE(rows >= 1 && rows * num_q_heads * slices <= 0x7fffffffLL,
                   "%s: num_tokens %lld out of range for %d key slices", what, (long long)rows, slices);
    const size_t need = prefill_split_workspace_bytes(rows, num_q_heads, slices);
    LITEKV_REQUIRE(split.workspace != nullptr && aligned16(split.workspace) && split.workspace_bytes >= need,
                   "%s: workspace of %zu bytes needed for %d key slices, got %zu", what, need, slices,
                   split.workspace_bytes);
    PrefillShape s = prefill_shape(group, max_q_len);
    // 64 columns a workgroup (narrow_fits); short slices (at most 16 tiles, as far as the block table can
    // say) up to twice as many: 128 rows, 64 / 8 heads, in 4 slices over 2048 tokens 29.6, 25.5 us, over 8192
    // 54.7, 56.2, over 30 000 169.7, 181.0.
    const int64_t wgs = (int64_t)num_kv_heads * s.head_splits * s.row_blocks * slices * batch;
    const int64_t slice_keys = (int64_t)block_table_stride * page_size / slices;  // at most, by the table
    const bool narrow = (narrow_fits(wgs) || (wgs <= device_cus() && slice_keys <= 16 * kKvTile)) &&
                        !narrow_reads_twice(wgs, group, s.row_blocks, slice_keys, fp8);
    if (narrow) s = prefill_shape(group, max_q_len, kTiledWaves);
    LITEKV_REQUIRE((uint64_t)s.row_blocks * slices <= 65535u, "%s: max_q_len %d too large for %d key slices",
                   what, max_q_len, slices);
    float *part_o = static_cast<float *>(split.workspace);
    float *part_lse = part_o + (size_t)slices * rows * num_q_heads * kHD;
    const PrefixTask task{part_o, part_lse, 0, (int32_t)rows, num_q_heads, 0, 0};
    const dim3 grid((unsigned)(num_kv_heads * s.head_splits), s.row_blocks * (unsigned)slices, (unsigned)batch);
    auto launch_slices = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grid, dim3(kTiledWaves * kWave), 0, static_cast<hipStream_t>(stream),
                         static_cast<const half_t *>(q), q_token_stride, static_cast<half_t *>(out),
                         out_token_stride, paged, packed, task, cu_q_lens, (const int32_t *)nullptr,
                         context_lens, group, s.head_splits, s.heads_per_wg, s.row_tiles,
                         softmax_scale * kLog2eP, slices);
    };
    auto by_width = [&](auto mode_tag) {
      constexpr int MODE = decltype(mode_tag)::value;
      if (narrow) {
        launch_slices(varlen_prefill_tiled_kernel<MODE, 1>);
      } else {
        launch_slices(varlen_prefill_tiled_kernel<MODE>);
      }
    };
    if (format == kKvInt8) {
      by_width(std::integral_constant<int, kPagedPrefillSplitInt8>{});
    } else if (format == kKvFp8) {
      by_width(std::integral_constant<int, kPagedPrefillSplitFp8>{});
    } else {
      by_width(std::integral_constant<int, kPagedPrefillSplit>{});
    }
    int rc2 = check_launch(what);
    if (rc2 != LITEKV_OK) return rc2;
    const int64_t merge_rows = rows * num_q_heads;
    hipLaunchKernelGGL(prefill_split_merge_kernel, dim3((unsigned)((merge_rows + 3) / 4)), dim3(4 * kWave), 0,
                       static_cast<hipStream_t>(stream), part_o, part_lse, static_cast<half_t *>(out),
                       out_token_stride, rows, num_q_heads, slices);
    return check_launch(what);
  }
#endif  // LITEKV_HD != 256
  PrefillShape s = prefill_shape(group, max_q_len);
  LITEKV_REQUIRE(s.row_blocks <= 65535u, "%s: max_q_len %d too large", what, max_q_len);
  dim3 grid((unsigned)(num_kv_heads * s.head_splits), s.row_blocks, (unsigned)batch);
  auto launch = [&](auto mode_tag) {
    constexpr int MODE = decltype(mode_tag)::value;
    auto with = [&](auto kernel, int waves) {
      hipLaunchKernelGGL(kernel, grid, dim3(waves * kWave), 0, static_cast<hipStream_t>(stream),
                         static_cast<const half_t *>(q), q_token_stride, static_cast<half_t *>(out),
                         out_token_stride, paged, packed, PrefixTask{}, cu_q_lens,
                         (const int32_t *)nullptr, context_lens, group, s.head_splits, s.heads_per_wg,
                         s.row_tiles, softmax_scale * kLog2eP, 1);
    };
#if LITEKV_HD != 256
    const int64_t max_keys = context_lens != nullptr ? split.max_kv_len : max_q_len;
    const int64_t wgs = (int64_t)grid.x * grid.y * grid.z;
    if (narrow_fits(wgs) && !narrow_reads_twice(wgs, group, s.row_blocks, max_keys, fp8)) {
      s = prefill_shape(group, max_q_len, kTiledWaves);
      grid = dim3((unsigned)(num_kv_heads * s.head_splits), s.row_blocks, (unsigned)batch);
      with(varlen_prefill_tiled_kernel<MODE, 1>, kTiledWaves);
      return;
    }
    if (two_key_groups(wgs, s.row_blocks, max_keys, fp8)) {
      with(varlen_prefill_two_group_kernel<MODE>, 2 * kTiledWaves);
      return;
    }
#endif
    with(varlen_prefill_tiled_kernel<MODE>, prefill_waves(MODE));
  };
  if (format == kKvInt8) {
    launch(std::integral_constant<int, kPagedPrefillInt8>{});
  } else if (format == kKvFp8) {
    launch(std::integral_constant<int, kPagedPrefillFp8>{});
  } else {
    launch(std::integral_constant<int, kPagedPrefill>{});
  }
  return check_launch(what);
}

// Causal attention over packed, contiguous K/V.
static int launch_varlen_prefill(const void *q, int64_t q_token_stride, const void *k,
                                 int64_t k_token_stride, const void *v, int64_t v_token_stride,
                                 const int32_t *seq_starts, const int32_t *seq_lens, void *out,
                                 int64_t out_token_stride, int32_t batch, int32_t num_q_heads,
                                 int32_t num_kv_heads, int32_t head_dim, int32_t max_seq_len,
                                 int64_t num_tokens, float softmax_scale, void *stream) {
#if LITEKV_HD == 128
  const PrefillBuild *build =
      head_dim == 64 ? &hd64_prefill()
      : head_dim == 256 && tiled_256(q_token_stride, out_token_stride, num_kv_heads, softmax_scale) &&
              k_token_stride < (1 << 25) && v_token_stride < (1 << 25)
          ? &hd256_prefill()
          : nullptr;
  if (build != nullptr) {  // another head dim's build of this file
    return build->varlen(q, q_token_stride, k, k_token_stride, v, v_token_stride, seq_starts, seq_lens, out,
                         out_token_stride, batch, num_q_heads, num_kv_heads, head_dim, max_seq_len,
                         num_tokens, softmax_scale, stream);
  }
#endif
  if (head_dim != kHD && generic_head_dim(head_dim)) {  // see generic_attention.hip
    LITEKV_REQUIRE(max_seq_len >= 0, "varlen_prefill: max_seq_len %d < 0", max_seq_len);
    GenericLaunch g;
    g.q = q;
    g.q_row_stride = q_token_stride;
    g.out = out;
    g.out_row_stride = out_token_stride;
    g.k = k;
    g.v = v;
    g.k_stride = k_token_stride;
    g.v_stride = v_token_stride;
    g.seq_starts = seq_starts;
    g.q_lens = seq_lens;
    g.batch = num_tokens == 0 ? 0 : batch;
    g.rows_per_seq = max_seq_len;
    g.num_q_heads = num_q_heads;
    g.num_kv_heads = num_kv_heads;
    g.head_dim = head_dim;
    g.softmax_scale = softmax_scale;
    g.stream = stream;
    return launch_generic_attention("varlen_prefill", g);
  }
  int rc = validate_prefill("varlen_prefill", q, q_token_stride, out, out_token_stride, batch,
                            num_q_heads, num_kv_heads, head_dim, max_seq_len);
  if (rc != LITEKV_OK) return rc;
  if (batch == 0 || max_seq_len == 0 || num_tokens == 0) {
    clear_error();
    return LITEKV_OK;
  }
  LITEKV_REQUIRE(k && v && seq_starts && seq_lens, "varlen_prefill: null pointer");
  LITEKV_REQUIRE(aligned16(k) && aligned16(v), "varlen_prefill: k and v must be 16-byte aligned");
  const int64_t row = (int64_t)num_kv_heads * head_dim;
  LITEKV_REQUIRE(k_token_stride >= row && k_token_stride % 8 == 0 && v_token_stride >= row &&
                     v_token_stride % 8 == 0,
                 "varlen_prefill: k/v token strides (%lld, %lld) invalid",
                 (long long)k_token_stride, (long long)v_token_stride);
  LITEKV_REQUIRE(k_token_stride < (1 << 25) && v_token_stride < (1 << 25),
                 "varlen_prefill: k/v token strides (%lld, %lld) too large",
                 (long long)k_token_stride, (long long)v_token_stride);
  PagedSource paged{nullptr, nullptr, 0, num_kv_heads, 1, nullptr};
  PackedSource packed{static_cast<const half_t *>(k), static_cast<const half_t *>(v),
                      k_token_stride, v_token_stride, seq_starts};
  const int group = num_q_heads / num_kv_heads;
  PrefillShape s = prefill_shape(group, max_seq_len);
  LITEKV_REQUIRE(s.row_blocks <= 65535u, "varlen_prefill: max_seq_len %d too large", max_seq_len);
  dim3 grid((unsigned)(num_kv_heads * s.head_splits), s.row_blocks, (unsigned)batch);
  auto launch = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, grid, dim3(waves * kWave), 0, static_cast<hipStream_t>(stream),
                       static_cast<const half_t *>(q), q_token_stride, static_cast<half_t *>(out),
                       out_token_stride, paged, packed, PrefixTask{}, seq_starts, seq_lens,
                       (const int32_t *)nullptr, group, s.head_splits, s.heads_per_wg, s.row_tiles,
                       softmax_scale * kLog2eP, 1);
  };
#if LITEKV_HD != 256
  const int64_t wgs = (int64_t)grid.x * grid.y * grid.z;
  if (narrow_fits(wgs) && !narrow_reads_twice(wgs, group, s.row_blocks, max_seq_len, false)) {
    s = prefill_shape(group, max_seq_len, kTiledWaves);
    grid = dim3((unsigned)(num_kv_heads * s.head_splits), s.row_blocks, (unsigned)batch);
    launch(varlen_prefill_tiled_kernel<kPackedPrefill, 1>, kTiledWaves);
    return check_launch("varlen_prefill");
  }
  if (two_key_groups(wgs, s.row_blocks, max_seq_len, false)) {
    launch(varlen_prefill_two_group_kernel<kPackedPrefill>, 2 * kTiledWaves);
    return check_launch("varlen_prefill");
  }
#endif
  launch(varlen_prefill_tiled_kernel<kPackedPrefill>, prefill_waves(kPackedPrefill));
  return check_launch("varlen_prefill");
}
}  // namespace LITEKV_HD_NS

#if LITEKV_HD == 64
const PrefillBuild &hd64_prefill() {
  static const PrefillBuild build{launch_paged_prefill, launch_varlen_prefill, prefill_key_slices};
  return build;
}
#elif LITEKV_HD == 256
const PrefillBuild &hd256_prefill() {
  static const PrefillBuild build{launch_paged_prefill, launch_varlen_prefill, nullptr};
  return build;
}
#endif
}  // namespace litekv

#if LITEKV_HD == 128  // the C ABI lives in the head dim 128 build of this file

extern "C" int litekv_paged_prefill(const void *q, int64_t q_token_stride, const void *kv_pool,
                                    const int32_t *block_table, int32_t block_table_stride,
                                    const int32_t *cu_q_lens, const int32_t *context_lens,
                                    void *out, int64_t out_token_stride, int32_t batch,
                                    int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                    int32_t page_size, int64_t num_pages, int32_t max_q_len,
                                    float softmax_scale, void *stream) {
  return litekv::launch_paged_prefill("paged_prefill", q, q_token_stride, kv_pool, nullptr, block_table,
                                      block_table_stride, cu_q_lens, context_lens, out,
                                      out_token_stride, batch, num_q_heads, num_kv_heads, head_dim,
                                      page_size, num_pages, max_q_len, softmax_scale, stream,
                                      litekv::kKvF16, litekv::PrefillKeySplit{});
}

extern "C" int litekv_paged_prefill_bounded(const void *q, int64_t q_token_stride, const void *kv_pool,
                                            const float *kv_scales, int32_t pool_is_int8,
                                            const int32_t *block_table, int32_t block_table_stride,
                                            const int32_t *cu_q_lens, const int32_t *context_lens,
                                            void *out, int64_t out_token_stride, int32_t batch,
                                            int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                            int32_t page_size, int64_t num_pages, int32_t max_q_len,
                                            int64_t max_kv_len, float softmax_scale, void *stream) {
  const int format = kv_scales == nullptr ? litekv::kKvF16 : pool_is_int8 ? litekv::kKvInt8 : litekv::kKvFp8;
  const char *what = format == litekv::kKvF16    ? "paged_prefill"
                     : format == litekv::kKvInt8 ? "paged_prefill_int8"
                                                 : "paged_prefill_fp8";
  litekv::PrefillKeySplit split;
  split.max_kv_len = max_kv_len;
  return litekv::launch_paged_prefill(what, q, q_token_stride, kv_pool, kv_scales, block_table,
                                      block_table_stride, cu_q_lens, context_lens, out,
                                      out_token_stride, batch, num_q_heads, num_kv_heads, head_dim,
                                      page_size, num_pages, max_q_len, softmax_scale, stream, format, split);
}

extern "C" size_t litekv_paged_prefill_split_workspace_bytes(int64_t num_tokens, int32_t num_q_heads,
                                                             int32_t head_dim, int32_t key_slices) {
  if (head_dim != 128 && head_dim != 64) return 0;
  if (num_tokens <= 0 || num_q_heads <= 0 || key_slices <= 1) return 0;
  return (size_t)key_slices * (size_t)num_tokens * (size_t)num_q_heads * (size_t)(head_dim + 1) * sizeof(float);
}

extern "C" int32_t litekv_paged_prefill_key_slices(int32_t batch, int32_t num_q_heads,
                                                   int32_t num_kv_heads, int32_t head_dim,
                                                   int32_t max_q_len, int64_t max_kv_len) {
  if (head_dim == 64) {
    return litekv::hd64_prefill().key_slices(batch, num_q_heads, num_kv_heads, max_q_len, max_kv_len);
  }
  if (head_dim != 128) return 1;
  return litekv::prefill_key_slices(batch, num_q_heads, num_kv_heads, max_q_len, max_kv_len);
}

extern "C" int litekv_paged_prefill_split(const void *q, int64_t q_token_stride, const void *kv_pool,
                                          const int32_t *block_table, int32_t block_table_stride,
                                          const int32_t *cu_q_lens, const int32_t *context_lens,
                                          void *out, int64_t out_token_stride, int32_t batch,
                                          int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                          int32_t page_size, int64_t num_pages, int32_t max_q_len,
                                          int64_t num_tokens, int32_t key_slices, void *workspace,
                                          size_t workspace_bytes, float softmax_scale, void *stream) {
  litekv::PrefillKeySplit split;
  split.key_slices = key_slices;
  split.workspace = workspace;
  split.workspace_bytes = workspace_bytes;
  split.num_tokens = num_tokens;
  return litekv::launch_paged_prefill("paged_prefill_split", q, q_token_stride, kv_pool, nullptr,
                                      block_table, block_table_stride, cu_q_lens, context_lens, out,
                                      out_token_stride, batch, num_q_heads, num_kv_heads, head_dim,
                                      page_size, num_pages, max_q_len, softmax_scale, stream,
                                      litekv::kKvF16, split);
}

extern "C" int litekv_paged_prefill_split_q8(const void *q, int64_t q_token_stride, const void *kv_pool,
                                             const float *kv_scales, int32_t pool_is_int8,
                                             const int32_t *block_table, int32_t block_table_stride,
                                             const int32_t *cu_q_lens, const int32_t *context_lens,
                                             void *out, int64_t out_token_stride, int32_t batch,
                                             int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                             int32_t page_size, int64_t num_pages, int32_t max_q_len,
                                             int64_t num_tokens, int32_t key_slices, void *workspace,
                                             size_t workspace_bytes, float softmax_scale, void *stream) {
  litekv::PrefillKeySplit split;
  split.key_slices = key_slices;
  split.workspace = workspace;
  split.workspace_bytes = workspace_bytes;
  split.num_tokens = num_tokens;
  return litekv::launch_paged_prefill(pool_is_int8 ? "paged_prefill_split_int8" : "paged_prefill_split_fp8", q,
                                      q_token_stride, kv_pool, kv_scales, block_table, block_table_stride,
                                      cu_q_lens, context_lens, out, out_token_stride, batch, num_q_heads,
                                      num_kv_heads, head_dim, page_size, num_pages, max_q_len,
                                      softmax_scale, stream, pool_is_int8 ? litekv::kKvInt8 : litekv::kKvFp8,
                                      split);
}

extern "C" int litekv_paged_prefill_fp8(const void *q, int64_t q_token_stride, const void *kv_pool,
                                        const float *kv_scales, const int32_t *block_table,
                                        int32_t block_table_stride, const int32_t *cu_q_lens,
                                        const int32_t *context_lens, void *out,
                                        int64_t out_token_stride, int32_t batch,
                                        int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                        int32_t page_size, int64_t num_pages, int32_t max_q_len,
                                        float softmax_scale, void *stream) {
  return litekv::launch_paged_prefill("paged_prefill_fp8", q, q_token_stride, kv_pool, kv_scales,
                                      block_table, block_table_stride, cu_q_lens, context_lens, out,
                                      out_token_stride, batch, num_q_heads, num_kv_heads, head_dim,
                                      page_size, num_pages, max_q_len, softmax_scale, stream,
                                      litekv::kKvFp8, litekv::PrefillKeySplit{});
}

extern "C" int litekv_paged_prefill_int8(const void *q, int64_t q_token_stride, const void *kv_pool,
                                         const float *kv_scales, const int32_t *block_table,
                                         int32_t block_table_stride, const int32_t *cu_q_lens,
                                         const int32_t *context_lens, void *out,
                                         int64_t out_token_stride, int32_t batch,
                                         int32_t num_q_heads, int32_t num_kv_heads, int32_t head_dim,
                                         int32_t page_size, int64_t num_pages, int32_t max_q_len,
                                         float softmax_scale, void *stream) {
  return litekv::launch_paged_prefill("paged_prefill_int8", q, q_token_stride, kv_pool, kv_scales,
                                      block_table, block_table_stride, cu_q_lens, context_lens, out,
                                      out_token_stride, batch, num_q_heads, num_kv_heads, head_dim,
                                      page_size, num_pages, max_q_len, softmax_scale, stream,
                                      litekv::kKvInt8, litekv::PrefillKeySplit{});
}

extern "C" int litekv_varlen_prefill(const void *q, int64_t q_token_stride, const void *k,
                                     int64_t k_token_stride, const void *v, int64_t v_token_stride,
                                     const int32_t *seq_starts, const int32_t *seq_lens, void *out,
                                     int64_t out_token_stride, int32_t batch, int32_t num_q_heads,
                                     int32_t num_kv_heads, int32_t head_dim, int32_t max_seq_len,
                                     int64_t num_tokens, float softmax_scale, void *stream) {
  return litekv::launch_varlen_prefill(q, q_token_stride, k, k_token_stride, v, v_token_stride,
                                       seq_starts, seq_lens, out, out_token_stride, batch,
                                       num_q_heads, num_kv_heads, head_dim, max_seq_len, num_tokens,
                                       softmax_scale, stream);
}
#endif  // LITEKV_HD == 128
