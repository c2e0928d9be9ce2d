// The column tiles of a 256-wide prefill that the matrix pipeline of prefill_tile.h does not serve:
// neighbouring query rows of one query head (a tile has 16), in fp32 without matrix instructions, as the general
// kernel (generic_attention.hip) computes them, whatever the scale and the values are. Run by one
// whole wavefront in the place of its tile.
//
// Bound by LDS reads and fp32 arithmetic: four prompts of 300 to 2048 tokens, 16 / 4 heads, every tile by
// rows, 8 at a time by eight wavefronts, 2.9 ms (16 by four 5.2, the general kernel 9.2, the matrix pipeline 0.08). It
// stands here so that the launch needs no second kernel and no look at device data from the host.
#pragma once

#include "common.h"
#include "kv_fp8.h"

namespace litekv {
namespace prefill_rows {

constexpr int kDim = 256;
// Per wavefront: 20.25 KiB for 16 rows attended together, 10.25 for 8. (A row's result does not depend on it.)
constexpr int lds_bytes(int rows) { return (rows * kDim + kWave * (rows + 1)) * 4; }

typedef __attribute__((address_space(3))) float lds_float_t;

// Orders this wavefront's LDS accesses for the compiler (the LDS unit keeps one wavefront's order).
__device__ __forceinline__ void lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// q, out: the first row (`rows` of them, 1 .. ROWS); that row sees keys 0 .. keys0 - 1, each
// further row one key more. kv_row(token, value): address of the token's K or V row of the kv head
// (fp16, or codes of format KV). lds: lds_bytes(ROWS) bytes of this wavefront's own.
template <int KV, int ROWS, typename KvRow>
__device__ __forceinline__ void attend_rows(uint32_t lds, const half_t *q, int64_t q_stride, half_t *out,
                                            int64_t out_stride, int rows, int keys0, KvRow kv_row,
                                            float scale_log2, float k_scale, float v_scale) {
  const int lane = threadIdx.x & (kWave - 1);
  lds_float_t *qs = (lds_float_t *)(uintptr_t)lds;                         // [ROWS][kDim]
  lds_float_t *ps = (lds_float_t *)(uintptr_t)(lds + 4u * ROWS * kDim);   // [kWave][ROWS + 1]
  auto load8 = [&](const void *row, int d8) -> half8_t {
    if constexpr (KV == kKvF16) {
      return *((const half8_t *)row + d8);
    } else {
      return codes_to_half<KV>(*((const uint2_t *)row + d8));
    }
  };
  lds_fence();
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {  // rows past the last repeat it and are not written
    const half_t *row = q + (int64_t)(r < rows ? r : rows - 1) * q_stride;
#pragma unroll
    for (int c = 0; c < kDim / kWave; ++c) {
      qs[r * kDim + lane + kWave * c] = (float)row[lane + kWave * c] * scale_log2;
    }
  }
  lds_fence();
  float m[ROWS], den[ROWS], acc[ROWS][kDim / kWave];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    m[r] = -INFINITY;
    den[r] = 0.f;
#pragma unroll
    for (int c = 0; c < kDim / kWave; ++c) acc[r][c] = 0.f;
  }
  const int n_keys = keys0 + rows - 1;
  for (int t0 = 0; t0 < n_keys; t0 += kWave) {
    const int tok = t0 + lane;  // this lane's key
    const void *k_row = kv_row(tok < n_keys ? tok : n_keys - 1, false);
    float s[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) s[r] = 0.f;
    for (int d8 = 0; d8 < kDim / 8; ++d8) {
      const half8_t k8 = load8(k_row, d8);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
#pragma unroll
        for (int e = 0; e < 8; ++e) s[r] += qs[r * kDim + 8 * d8 + e] * (float)k8[e];
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
      // key 0 is in every row's first step: the running maximum is the maximum of real scores
      const float sv = tok < keys0 + (r < rows ? r : rows - 1) ? s[r] * k_scale : -INFINITY;
      float mx = sv;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, xor_lane(mx, off));
      const float m_new = fmaxf(m[r], mx);
      const float alpha = fast_exp2(m[r] - m_new);
      const float p = fast_exp2(sv - m_new);
      float sum = p;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) sum += xor_lane(sum, off);
      den[r] = den[r] * alpha + sum;
      m[r] = m_new;
#pragma unroll
      for (int c = 0; c < kDim / kWave; ++c) acc[r][c] *= alpha;
      ps[lane * (ROWS + 1) + r] = p;
    }
    lds_fence();
    const int n_here = n_keys - t0 < kWave ? n_keys - t0 : kWave;
    for (int j = 0; j < n_here; ++j) {
      const void *v_row = kv_row(t0 + j, true);
      float v[kDim / kWave];
#pragma unroll
      for (int c = 0; c < kDim / kWave; ++c) {
        const int d = lane + kWave * c;
        v[c] = (float)load8(v_row, d / 8)[d % 8];
      }
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        // (a probability of 0 does not keep an infinite value out: 0 * inf is NaN)
        const bool sees = t0 + j < keys0 + (r < rows ? r : rows - 1);
        const float p = ps[j * (ROWS + 1) + r];
#pragma unroll
        for (int c = 0; c < kDim / kWave; ++c) acc[r][c] += sees ? p * v[c] : 0.f;
      }
    }
    lds_fence();
  }
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    if (r < rows) {
      const float inv = v_scale / den[r];
#pragma unroll
      for (int c = 0; c < kDim / kWave; ++c) {
        out[(int64_t)r * out_stride + lane + kWave * c] = (half_t)(acc[r][c] * inv);
      }
    }
  }
}

}  // namespace prefill_rows
}  // namespace litekv
