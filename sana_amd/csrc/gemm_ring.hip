#include "gemm_ring.h"

#include <algorithm>

namespace sana {
namespace {

template <int WM, int WN, int TM, int TN, int ST, bool WHOLE, typename T>
int launch_ring(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                int64_t ldw, int64_t ldc, int epilogue, hipStream_t s) {
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  const int tiles_t = (M + BM - 1) / BM, tiles_c = (N + BN - 1) / BN;
  const dim3 grid((unsigned)(tiles_t * tiles_c)), block(64 * WM * WN);
  // An XCD works on an eighth of the tiles, g token tiles x the rest: the shape that reads the fewest operand rows.
  const int per = std::max(1, tiles_t * tiles_c / 8);
  int group = 1;
  int64_t best = INT64_MAX;
  for (int g = 1; g <= std::min(tiles_t, 64); ++g) {
    const int64_t cost = (int64_t)g * BM + (int64_t)((per + g - 1) / g) * BN;
    if (cost < best) best = cost, group = g;
  }
#define SANA_LAUNCH_R(EPI)                                                                                              \
  hipLaunchKernelGGL((gemm_ring_kernel<WM, WN, TM, TN, ST, WHOLE, EPI, T>), grid, block, 0, s, a, w, ep, c, M, N, K, lda, ldw, ldc, \
                     tiles_t, tiles_c, group)
  switch (epilogue) {
    case SANA_EPI_NONE: SANA_LAUNCH_R(SANA_EPI_NONE); break;
    case SANA_EPI_BIAS: SANA_LAUNCH_R(SANA_EPI_BIAS); break;
    case SANA_EPI_BIAS_SILU: SANA_LAUNCH_R(SANA_EPI_BIAS_SILU); break;
    case SANA_EPI_GATE_RES: SANA_LAUNCH_R(SANA_EPI_GATE_RES); break;
    default: return SANA_ERR_ARG;
  }
#undef SANA_LAUNCH_R
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

}  // namespace

int gemm_ring_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                     int64_t ldw, int64_t ldc, int epilogue, bool f16, int bm, int bn, hipStream_t s) {
#define SANA_RING(WM, WN, TM, TN, ST, WHOLE)                                                                           \
  if (bm == 16 * TM * WM && bn == 16 * TN * WN)                                                                        \
  return f16 ? launch_ring<WM, WN, TM, TN, ST, WHOLE, F16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, s)            \
             : launch_ring<WM, WN, TM, TN, ST, WHOLE, BF16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, s)
  // 64 x 64 where at most half the compute units would have a tile: each in two workgroups of 32 channels.  A compute unit takes 70 - 75
  // bytes/ns of such operands, whatever the ring's depth (8 and 10 stages: the same per k-tile, 1.1 and 1.9 us more in front of the
  // first), so a k-tile takes as long as its bytes: 12 KB 0.16 us, 16 KB 0.22.  us: 256 x 1152 x 1152 7.4 -> 6.0, x 2880
  // 13.4 -> 10.3, 144 x 2240 x 2240 11.7 -> 9.1; 32 tokens x 64 channels 6.2, 10.5, 9.6.  From 129 tiles on two workgroups would
  // share a compute unit: 512 x 1152 x 1152 7.4 in 64 x 64, 8.7 in halves.
  if (bm == 64 && bn == 64 && ((M + 63) / 64) * (int64_t)((N + 63) / 64) <= kHalvedTiles) bn = 32;
  SANA_RING(4, 1, 1, 2, 6, true);  // 64 x 32, 72 KB
  SANA_RING(2, 2, 2, 2, 5, true);  // 64 x 64, 80 KB: two workgroups per compute unit
  SANA_RING(2, 4, 2, 2, 6, true);  // 64 x 128
  SANA_RING(2, 4, 3, 2, 5, true);  // 96 x 128
  SANA_RING(2, 4, 4, 2, 4, true);  // 128 x 128
  // 128 x 160.  The other loop (with 4 x 2 or 2 x 2 waves) needs 800 cycles a k-tile where this needs 977, but at 224 workgroups
  // the chip then lowers its clock for what runs beside it as well: a step with int8 weights at 2048 rows takes 1721 us
  // with that loop and 1642 with this one, at 1160 and 1245 W.
  SANA_RING(4, 1, 2, 10, 4, false);
  SANA_RING(4, 2, 3, 4, 4, true);  // 192 x 128
  SANA_RING(4, 2, 4, 4, 3, true);  // 256 x 128
#undef SANA_RING
  return SANA_ERR_ARG;
}

}  // namespace sana
