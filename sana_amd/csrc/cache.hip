// The small passes around a streamed chunk's kernels: the cache of the chunks before, read and written.
#include "common.h"

namespace sana {
namespace {

// state += past, and the state of this chunk alone to save_vk / save_ks ([B*h][d][d] and [B*h][d]; state [B*h][d + 1][d]).
// Bound by its launch: 2 MB at 20 heads of 112.  Two copies and two additions, one each for the d rows of products and the row of
// key sums, were 5 us each; this is 5.5 in all.
__global__ __launch_bounds__(256) void state_cache_kernel(f32x4_t* __restrict__ state, const f32x4_t* __restrict__ past_vk,
                                                          const f32x4_t* __restrict__ past_ks, f32x4_t* __restrict__ save_vk,
                                                          f32x4_t* __restrict__ save_ks, int64_t total, int d) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // four values; d % 4 == 0
  if (i >= total) return;
  const int row4 = d / 4, per = (d + 1) * row4, products = d * row4;
  const int64_t bh = i / per;
  const int e = (int)(i - bh * per);
  const bool ks = e >= products;
  const int64_t at = ks ? bh * row4 + (e - products) : bh * products + e;
  const f32x4_t s = state[i];
  if (save_vk) (ks ? save_ks : save_vk)[at] = s;
  if (past_vk) state[i] = s + (ks ? past_ks : past_vk)[at];
}

// dst[b][p][c] = src[b][c][p], 16-bit values: 64 x 64 tiles through LDS, 128-byte loads along p (any alignment), 16-byte stores.
// An elementwise copy between the two layouts takes 23 us for 1560 x 2240, this 6 (7 MB read, 7 written).
__global__ __launch_bounds__(256) void transpose16_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int P,
                                                          int C, int64_t src_b, int64_t src_c, int64_t dst_b, int64_t dst_p) {
  constexpr int PITCH = 66;
  __shared__ uint16_t tile[64 * PITCH];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int p0 = blockIdx.x * 64, c0 = blockIdx.y * 64;
  const uint16_t* s = src + (int64_t)blockIdx.z * src_b + p0 + lane;
  uint16_t v[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int c = c0 + wave + 4 * i;
    v[i] = c < C && p0 + lane < P ? s[(int64_t)c * src_c] : (uint16_t)0;
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) tile[(wave + 4 * i) * PITCH + lane] = v[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = threadIdx.x + 256 * i, p = idx >> 3, c = (idx & 7) * 8;
    if (p0 + p >= P || c0 + c >= C) continue;  // C % 8 == 0
    u32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = tile[(c + 2 * e) * PITCH + p] | ((uint32_t)tile[(c + 2 * e + 1) * PITCH + p] << 16);
    *reinterpret_cast<u32x4_t*>(dst + (int64_t)blockIdx.z * dst_b + (int64_t)(p0 + p) * dst_p + c0 + c) = o;
  }
}

}  // namespace
}  // namespace sana

using namespace sana;

#define SANA_API extern "C" __attribute__((visibility("default")))

SANA_API int sana_hip_state_cache(float* state, const float* past_vk, const float* past_ks, float* save_vk, float* save_ks,
                                  int B, int h, int d, void* stream) {
  if (!state || B <= 0 || h <= 0 || d <= 0 || !past_vk != !past_ks || !save_vk != !save_ks) return SANA_ERR_ARG;
  if (d % 4 || d > 1024) return SANA_ERR_SHAPE;
  for (const void* p : {(const void*)state, (const void*)past_vk, (const void*)past_ks, (const void*)save_vk, (const void*)save_ks})
    if (!aligned16(p)) return SANA_ERR_ALIGN;
  if (!past_vk && !save_vk) return SANA_OK;
  const int64_t total = (int64_t)B * h * (d + 1) * (d / 4), groups = (total + 255) / 256;
  if (groups > 0x7fffffff) return SANA_ERR_SHAPE;
  hipLaunchKernelGGL(state_cache_kernel, dim3((unsigned)groups), dim3(256), 0, static_cast<hipStream_t>(stream),
                     reinterpret_cast<f32x4_t*>(state), reinterpret_cast<const f32x4_t*>(past_vk),
                     reinterpret_cast<const f32x4_t*>(past_ks), reinterpret_cast<f32x4_t*>(save_vk),
                     reinterpret_cast<f32x4_t*>(save_ks), total, d);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

SANA_API int sana_hip_transpose16(const void* src, void* dst, int B, int P, int C, int64_t src_b, int64_t src_c, int64_t dst_b,
                                  int64_t dst_p, void* stream) {
  if (!src || !dst || B <= 0 || P <= 0 || C <= 0) return SANA_ERR_ARG;
  if (C % 8 || B > 65535 || (C + 63) / 64 > 65535) return SANA_ERR_SHAPE;
  if (src_b < 0 || src_c < 0 || dst_b < 0 || dst_p < C) return SANA_ERR_ARG;
  if (!aligned16(dst) || dst_b % 8 || dst_p % 8 || (reinterpret_cast<uintptr_t>(src) & 1)) return SANA_ERR_ALIGN;
  hipLaunchKernelGGL(transpose16_kernel, dim3((unsigned)((P + 63) / 64), (unsigned)((C + 63) / 64), (unsigned)B), dim3(256), 0,
                     static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), P, C,
                     src_b, src_c, dst_b, dst_p);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}
