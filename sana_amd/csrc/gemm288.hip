#include "gemm288.h"

#include <algorithm>

namespace sana {
namespace {

template <typename T>
int launch_288(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
               int64_t ldw, int64_t ldc, int epilogue, const Taps* taps, hipStream_t s) {
  const int64_t tiles_t = (M + 255) / 256, tiles_c = (N + 287) / 288;
  if (tiles_t * tiles_c > (1 << 30)) return SANA_ERR_SHAPE;
  const dim3 grid((unsigned)std::min<int64_t>(tiles_t * tiles_c, 256)), block(512);  // one workgroup per compute unit
  const Taps none = {0, 0, 0, 0, 0, nullptr};
#define SANA_LAUNCH288(EPI, TAPS, TP)                                                                                 \
  hipLaunchKernelGGL((gemm288_kernel<EPI, TAPS, T>), grid, block, 0, s, a, w, ep, c, M, N, K, lda, ldw, ldc, (int)tiles_t, \
                     (int)tiles_c, TP)
  if (taps) {
    if constexpr (!is_f16<T>) {
      if (epilogue != SANA_EPI_GATE_RES) return SANA_ERR_ARG;
      if (taps->zero_last) SANA_LAUNCH288(SANA_EPI_GATE_RES, 2, *taps);
      else SANA_LAUNCH288(SANA_EPI_GATE_RES, 1, *taps);
      return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
    } else {
      return SANA_ERR_ARG;
    }
  }
  switch (epilogue) {
    case SANA_EPI_NONE: SANA_LAUNCH288(SANA_EPI_NONE, 0, none); break;
    case SANA_EPI_BIAS: SANA_LAUNCH288(SANA_EPI_BIAS, 0, none); break;
    case SANA_EPI_BIAS_SILU: SANA_LAUNCH288(SANA_EPI_BIAS_SILU, 0, none); break;
    case SANA_EPI_GATE_RES: SANA_LAUNCH288(SANA_EPI_GATE_RES, 0, none); break;
    default: return SANA_ERR_ARG;
  }
#undef SANA_LAUNCH288
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

}  // namespace

int gemm288_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                   int64_t ldw, int64_t ldc, int epilogue, bool f16, const Taps* taps, hipStream_t s) {
  return f16 ? launch_288<F16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, taps, s)
             : launch_288<BF16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, taps, s);
}

}  // namespace sana
