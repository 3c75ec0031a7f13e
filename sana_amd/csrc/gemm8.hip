#include "gemm8.h"

#include <algorithm>

namespace sana {
namespace {

template <int NB, typename T>
int launch_nb(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
              int64_t ldw, int64_t ldc, int epilogue, const Taps* taps, hipStream_t s) {
  const int64_t tiles_t = (M + 255) / 256, tiles_c = (N + 64 * NB - 1) / (64 * NB);
  if (tiles_t * tiles_c > (1 << 30)) return SANA_ERR_SHAPE;
  const dim3 grid((unsigned)std::min<int64_t>(tiles_t * tiles_c, 256)), block(512);  // one workgroup per compute unit
  const Taps none = {0, 0, 0, 0, 0, nullptr};
#define SANA_LAUNCH8(EPI, TAPS, TP)                                                                                   \
  hipLaunchKernelGGL((gemm8_kernel<EPI, NB, TAPS, T>), grid, block, 0, s, a, w, ep, c, M, N, K, lda, ldw, ldc, (int)tiles_t, \
                     (int)tiles_c, TP)
  if (taps) {
    if constexpr (NB != 2 && !is_f16<T>) {
      if (epilogue != SANA_EPI_GATE_RES) return SANA_ERR_ARG;
      if (taps->zero_last) SANA_LAUNCH8(SANA_EPI_GATE_RES, 2, *taps);
      else SANA_LAUNCH8(SANA_EPI_GATE_RES, 1, *taps);
      return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
    } else {
      return SANA_ERR_ARG;
    }
  }
  switch (epilogue) {
    case SANA_EPI_NONE: SANA_LAUNCH8(SANA_EPI_NONE, 0, none); break;
    case SANA_EPI_BIAS: SANA_LAUNCH8(SANA_EPI_BIAS, 0, none); break;
    case SANA_EPI_BIAS_SILU: SANA_LAUNCH8(SANA_EPI_BIAS_SILU, 0, none); break;
    case SANA_EPI_GATE_RES: SANA_LAUNCH8(SANA_EPI_GATE_RES, 0, none); break;
    case SANA_EPI_QKV_STATE:
      if constexpr (NB == 4 && !is_f16<T>) {
        SANA_LAUNCH8(SANA_EPI_QKV_STATE, 0, none);
        break;
      }
      return SANA_ERR_ARG;
    default: return SANA_ERR_ARG;
  }
#undef SANA_LAUNCH8
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

}  // namespace

// Against the one-wave-per-SIMD kernel that split 16-bit GEMMs before (gemm4_kernel, int8 weights only now), with the epilogue launch, us,
// weights cold: 1024 x 2240 x 5600 in five ranges 47.9 / 45.6, 600 in seven 36.8 / 35.0, 500 x 1152 x 5600 in eight 31.5 / 29.7; same bits.
int gemm8_planes_launch(const uint16_t* a, const uint16_t* w, float* planes, int M, int N, int K, int64_t lda, int64_t ldw, bool f16,
                        int tiles, int rem, int ranges, hipStream_t s) {
  const int tiles_t = (M + 255) / 256, tiles_c = (N + 191) / 192;
  const dim3 grid((unsigned)(tiles_t * tiles_c), (unsigned)ranges), block(512);
  const Taps split = {0, 0, 0, tiles, rem, nullptr};
  uint16_t* c = reinterpret_cast<uint16_t*>(planes);
  if (f16)
    hipLaunchKernelGGL((gemm8_kernel<SANA_EPI_PLANES, 3, 0, F16>), grid, block, 0, s, a, w, EpiArgs{}, c, M, N, K, lda, ldw, (int64_t)N, tiles_t,
                       tiles_c, split);
  else
    hipLaunchKernelGGL((gemm8_kernel<SANA_EPI_PLANES, 3, 0, BF16>), grid, block, 0, s, a, w, EpiArgs{}, c, M, N, K, lda, ldw, (int64_t)N, tiles_t,
                       tiles_c, split);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

int gemm8_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                 int64_t ldw, int64_t ldc, int epilogue, bool f16, int nb, const Taps* taps, hipStream_t s) {
#define SANA_NB8(NB)                                                                                            \
  return f16 ? launch_nb<NB, F16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, taps, s)                             \
             : launch_nb<NB, BF16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, taps, s)
  switch (nb) {
    case 2: SANA_NB8(2);
    case 3: SANA_NB8(3);
    case 4: SANA_NB8(4);
    default: return SANA_ERR_ARG;
  }
#undef SANA_NB8
}

}  // namespace sana
