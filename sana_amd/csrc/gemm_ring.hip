#include "gemm_ring.h"

#include <algorithm>

namespace sana {
namespace {

template <int WM, int WN, int TM, int TN, int ST, bool WHOLE, bool RANGES, typename T>
int launch_loop(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                int64_t ldw, int64_t ldc, int epilogue, uint32_t prefetch, const KRanges& kr, hipStream_t s) {
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
  hipLaunchKernelGGL((gemm_ring_kernel<WM, WN, TM, TN, ST, WHOLE, RANGES, EPI, T>), grid, block, 0, s, a, w, ep, c, M, N, K, lda, ldw, \
                     ldc, tiles_t, tiles_c, group, prefetch, kr)
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

// Weights ahead of the ring (and the loop over whole k-tiles, which gains by it), or not.  It pays where the workgroups of several
// token tiles read the same weights side by side.  One or two token tiles: nearly every weight is read once, and reading it ahead,
// into another XCD's cache, only adds to the traffic.  A last token tile of few rows: its workgroups, whose other rows are zeros,
// run ahead of the others and are their prefetch.  Nearly all compute units at work: the loads ahead compete with the ring's; with
// a full last tile that is 12 % less on one card and up to 8 % more on another, so that only a partly filled one decides.
// us, with / without: 72 x 6720 x 2240 14.2 / 11.1, 144 x 4480 x 2240 12.8 / 10.8, 256 x 11200 x 2240 29.8 / 26.5, 400 x 6720 x 2240 21.7 / 19.3,
// 800 x 6720 x 2240 32.3 / 29.4, 1088 x 3456 x 1152 13.9 / 12.9; 256 x 2240 x 2240 12.2 / 13.1, 512 x 1152 x 2880 12.8 / 15.3,
// 1024 x 1152 x 2880 17.8 / 21.8, 1024 x 2240 x 2240 18.7 / 20.8, 2400 x 1152 x 2880 22.8 / 26.1.
bool prefetch_pays(int bm, int bn, int M, int K, int64_t tiles_t, int64_t tiles_c) {
  const int last = (int)(M - (tiles_t - 1) * bm);  // rows of the last token tile
  if (bn == 32) return tiles_t > 3 || (tiles_t > 1 && 2 * last > bm);
  if (K >= 4096 && tiles_t > 7) return true;
  if (tiles_t <= 2 || last <= bm / (tiles_t > 4 ? 4 : tiles_t == 4 && bm == 64 ? 3 : 2)) return false;
  const int64_t busy = bm > 96 ? 212 : 216;  // workgroups
  return bm * bn <= 64 * 64 || tiles_t * tiles_c <= busy || tiles_t >= (bm == 64 ? 10 : 16) ||
         (bm > 64 && bm <= 128 && 4 * last > 3 * bm);
}

// AHEAD: the tile has the loop over whole k-tiles too.
template <int WM, int WN, int TM, int TN, int ST, bool AHEAD, bool RANGES, typename T>
int launch_ring(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                int64_t ldw, int64_t ldc, int epilogue, const KRanges& kr, hipStream_t s) {
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN;
  if constexpr (AHEAD) {
    // Dense weights of less than 2 GB; a loop too short for it to catch up loses (768 x 960, 1500 tokens 8.1 us without, 9.1 with).
    const bool ahead = ldw == K && (int64_t)N * K < ((int64_t)1 << 30) && K >= 1024 &&
                       prefetch_pays(BM, BN, M, K, (M + BM - 1) / BM, (N + BN - 1) / BN);
    // (64 x 32 gains by the loop without it too: 136 x 1152 x 2880 11.1 us in half k-tiles, 9.9; but 200 x 1536 x 64 2.8, 3.3)
    if (ahead || (BN == 32 && K >= 1024))
      return launch_loop<WM, WN, TM, TN, ST, true, RANGES, T>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue,
                                                              ahead ? (uint32_t)N * (uint32_t)K * 2u : 0u, kr, s);
  }
  return launch_loop<WM, WN, TM, TN, ST, false, RANGES, T>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, 0, kr, s);
}

}  // namespace

int gemm_ring_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                     int64_t ldw, int64_t ldc, int epilogue, bool f16, int bm, int bn, const KRanges& kr, hipStream_t s) {
#define SANA_RING(WM, WN, TM, TN, ST, AHEAD, RANGES)                                                                           \
  if (bm == 16 * TM * WM && bn == 16 * TN * WN && (kr.ranges > 1) == RANGES)                                                   \
  return f16 ? launch_ring<WM, WN, TM, TN, ST, AHEAD, RANGES, F16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, kr, s)        \
             : launch_ring<WM, WN, TM, TN, ST, AHEAD, RANGES, BF16>(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, kr, s)
  // 64 x 32: the plan's choice where 64 x 64 gives at most half the compute units a tile.  A compute unit takes 70 - 75
  // bytes/ns of such operands, whatever the ring's depth (8 and 10 stages: the same per k-tile, 1.1 and 1.9 us more in front of the
  // first), so a k-tile takes as long as its bytes: 12 KB 0.16 us, 16 KB 0.22.  us: 256 x 1152 x 1152 7.4 -> 6.0, x 2880
  // 13.4 -> 10.3, 144 x 2240 x 2240 11.7 -> 9.1; 32 tokens x 64 channels 6.2, 10.5, 9.6.  From 129 tiles on two workgroups would
  // share a compute unit: 512 x 1152 x 1152 7.4 in 64 x 64, 8.7 in halves.
  SANA_RING(4, 1, 1, 2, 6, true, false);   // 64 x 32, 72 KB
  SANA_RING(2, 2, 2, 2, 5, true, false);   // 64 x 64, 80 KB: two workgroups per compute unit
  SANA_RING(2, 4, 2, 2, 6, true, false);   // 64 x 128
  SANA_RING(2, 4, 3, 2, 5, true, false);   // 96 x 128
  SANA_RING(2, 4, 4, 2, 4, true, false);   // 128 x 128
  // 128 x 160.  The loop over whole k-tiles (with 4 x 2 or 2 x 2 waves) needs 800 cycles a k-tile where this needs 977, but at 224
  // workgroups the chip then lowers its clock for what runs beside it as well: a step with int8 weights at 2048 rows takes 1721 us
  // with that loop and 1642 with this one, at 1160 and 1245 W.
  SANA_RING(4, 1, 2, 10, 4, false, false);
  // 160 x 192: the 300 tokens of a prompt by the keys and values of a few blocks, two tiles of 256 rows a fifth longer than these.  us, weights
  // cold (each call others, tokens the same): 300 x 18432 x 1152 25.4 / 22.4 (23.7 / 20.5), 300 x 17920 x 2240 41.5 / 36.6 (37.7 / 33.9).  In 320 x 96,
  // with more operand bytes, 23.3 and 39.4; in 2 x 6 waves 23.2 and 36.6.
  SANA_RING(2, 2, 5, 6, 3, false, false);
  SANA_RING(4, 2, 3, 4, 4, true, false);   // 192 x 128
  SANA_RING(4, 2, 4, 4, 3, false, false);  // 256 x 128 (whole k-tiles: 0 - 12 % more, 1 - 4 % less at K = 5600)
  // sums over ranges of k (GEMMs that the split kernel was taken for; gemm.hip, split_way)
  SANA_RING(4, 1, 1, 2, 6, true, true);
  SANA_RING(2, 2, 2, 2, 5, true, true);
  SANA_RING(2, 4, 3, 2, 5, true, true);
  SANA_RING(4, 2, 3, 4, 4, true, true);
#undef SANA_RING
  return SANA_ERR_ARG;
}

}  // namespace sana
