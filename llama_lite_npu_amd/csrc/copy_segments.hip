// Several small device arrays copied in one launch: what a replayed decode step uploads into its
// graph's fixed tensors (token ids, positions, slots, lengths, request ids, block-table rows).
//
// Launch-bound: seven arrays of a few hundred bytes each. As seven copies on the stream they ran
// one after the other in front of every replayed step: 28 layers for one sequence of 778 tokens took
// 293 us a step with them and 281 with this launch.
// One grid row per array; a block takes 4 KiB of it (a thread four 4-byte words: block-table rows
// have any width, so rows are only 4-byte aligned), the largest array decides how many.
#include "common.h"

namespace litekv {

constexpr int kMaxSegments = 8;
constexpr int kSegmentThreads = 256;
constexpr int kWordsPerThread = 4;

struct SegmentList {
  litekv_copy_segment s[kMaxSegments];
};

__global__ __launch_bounds__(kSegmentThreads) void copy_segments_kernel(SegmentList list) {
  const litekv_copy_segment s = list.s[blockIdx.y];
  const uint32_t row_words = (uint32_t)(s.row_bytes >> 2);
  const uint32_t words = (uint32_t)s.rows * row_words;
  const uint32_t first = blockIdx.x * (kSegmentThreads * kWordsPerThread) + threadIdx.x;
  uint32_t x[kWordsPerThread];
#pragma unroll
  for (int i = 0; i < kWordsPerThread; ++i) {
    const uint32_t w = first + i * kSegmentThreads;
    const uint32_t row = w / row_words, col = w - row * row_words;
    if (w < words) x[i] = *(const uint32_t *)((const char *)s.src + row * s.src_pitch + 4 * (int64_t)col);
  }
#pragma unroll
  for (int i = 0; i < kWordsPerThread; ++i) {
    const uint32_t w = first + i * kSegmentThreads;
    const uint32_t row = w / row_words, col = w - row * row_words;
    if (w < words) *(uint32_t *)((char *)s.dst + row * s.dst_pitch + 4 * (int64_t)col) = x[i];
  }
}

}  // namespace litekv

extern "C" int litekv_copy_segments(const litekv_copy_segment *segments, int32_t count, void *stream) {
  using namespace litekv;
  const char *what = "copy_segments";
  LITEKV_REQUIRE(count >= 0 && count <= kMaxSegments, "%s: count %d out of [0, %d]", what, count, kMaxSegments);
  LITEKV_REQUIRE(count == 0 || segments != nullptr, "%s: null pointer", what);
  SegmentList list{};
  int n = 0;
  int64_t most = 0;
  for (int i = 0; i < count; ++i) {
    const litekv_copy_segment &s = segments[i];
    LITEKV_REQUIRE(s.rows >= 0 && s.row_bytes >= 0, "%s: segment %d has a negative size", what, i);
    if (s.rows == 0 || s.row_bytes == 0) continue;
    LITEKV_REQUIRE(s.src && s.dst, "%s: null pointer (segment %d)", what, i);
    LITEKV_REQUIRE(((reinterpret_cast<uintptr_t>(s.src) | reinterpret_cast<uintptr_t>(s.dst) |
                     (uint64_t)s.row_bytes | (uint64_t)s.src_pitch | (uint64_t)s.dst_pitch) & 3) == 0,
                   "%s: segment %d is not in whole 4-byte words", what, i);
    LITEKV_REQUIRE(s.rows == 1 || (s.src_pitch >= s.row_bytes && s.dst_pitch >= s.row_bytes),
                   "%s: segment %d: a pitch is smaller than its row", what, i);
    LITEKV_REQUIRE(s.row_bytes <= 0x40000000 && s.rows <= 0x40000000 / s.row_bytes,
                   "%s: segment %d is larger than 1 GiB", what, i);
    const int64_t words = s.rows * (s.row_bytes >> 2);
    most = words > most ? words : most;
    list.s[n++] = s;
  }
  if (n == 0) {
    clear_error();
    return LITEKV_OK;
  }
  const int64_t per_block = kSegmentThreads * kWordsPerThread;
  hipLaunchKernelGGL(copy_segments_kernel, dim3((unsigned)((most + per_block - 1) / per_block), (unsigned)n),
                     dim3(kSegmentThreads), 0, static_cast<hipStream_t>(stream), list);
  return check_launch(what);
}
