// The 16-bit GEMM for many tokens: 256 tokens x 64*NB channels per workgroup, eight waves (two per SIMD) in
// alternation, operands by direct global -> LDS loads.
#pragma once
#include <type_traits>

#include "gemm_common.h"

namespace sana {
namespace {

// 4 outputs of one row -> packed, per the epilogue kind (the gated residual is applied at store time)
template <int EPI, typename T>
__device__ __forceinline__ u32x2_t g8_pack4(f32x4_t a, const float* bv) {
  float v[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = EPI != SANA_EPI_NONE ? a[r] + bv[r] : a[r];
  u32x2_t o = {pk16<T>(v[0], v[1]), pk16<T>(v[2], v[3])};
  if (EPI == SANA_EPI_BIAS_SILU) {  // on the rounded linear output, as the reference
    float x[4] = {lo16<T>(o.x), hi16<T>(o.x), lo16<T>(o.y), hi16<T>(o.y)};
#pragma unroll
    for (int r = 0; r < 4; ++r) x[r] *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.44269504088896341f * x[r]));
    o.x = pk16<T>(x[0], x[1]);
    o.y = pk16<T>(x[2], x[3]);
  }
  return o;
}

// k / v column tile of the fused qkv projection (SANA_EPI_QKV_STATE).  The tile's 256 weight rows are, per wave
// column, [K of head 4T + wn | V of it] (32 rows each, see sana_hip_qkv_state_rows), so MFMA tiles 0 and 1 of a wave
// are K and tiles 2 and 3 are V.  Instead of storing k and v, the wave contracts them over its 128 tokens: S[dv][dk] +=
// v[n][dv] * relu(k[n][dk]) and ksum[dk] += relu(k[n][dk]) with v and k rounded to bf16 first (what the unfused path
// stores and reads back), products in fp32 on the MFMA.  The contraction index of the MFMA is the token, and which
// token sits in which k slot is free as long as both operands agree: the 8 tokens a lane holds for one channel (j =
// 0 .. 7) ARE one operand fragment, only in the wrong lane, so it takes one trip through the wave's 16 KB of LDS:
// written at [channel][token group ^ channel % 16] (conflict-free both ways), read back as [channel = lane % 16][token
// group 4 m + lane / 16] for the m-th MFMA of a chain of four.  The two token halves of the workgroup are added through
// LDS and the sum goes to this token tile's slot of the partial states, which a second kernel adds up in tile order
// (deterministic, no atomics).
__device__ __forceinline__ void g8_state_tile(f32x4_t (&acc)[4][8], const float (&bv)[16], unsigned char* smem,
                                              const EpiArgs& ep, int m0, int n0, int wave, int lane) {
  const int wm = wave >> 2, wn = wave & 3, fr = lane & 15, fg = lane >> 4;
  unsigned char* stg = smem + wave * 16384;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      u32x4_t o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = pack_bf16(acc[i][2 * e][r] + bv[4 * i + r], acc[i][2 * e + 1][r] + bv[4 * i + r]);
        if (i < 2) o[e] = relu_pk16(o[e]);
      }
      const int row = 32 * (i >> 1) + 8 * fg + 4 * (i & 1) + r;
      *reinterpret_cast<u32x4_t*>(stg + row * 256 + ((fr ^ (row & 15)) << 4)) = o;
    }
  // (wave-private LDS is in order: the reads below see the writes above.)  The products are formed transposed (rows =
  // dk, columns = dv): a lane ends with four consecutive dk of one dv, i.e. 16-byte stores into the [dv][dk] state.
  f32x4_t S[2][2], Ks[2];  // S[a][b]: dk 16 a + 4 fg + r, dv 16 b + fr;  Ks[a]: dk 16 a + 4 fg + r
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int r = 0; r < 4; ++r) Ks[a][r] = 0.f, S[a][0][r] = 0.f, S[a][1][r] = 0.f;
  const u32x4_t ones = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
#pragma unroll
  for (int m = 0; m < 4; ++m) {
    const int slot = ((4 * m + fg) ^ fr) << 4;
    u32x4_t kf[2], vf[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      kf[b] = *reinterpret_cast<const u32x4_t*>(stg + (16 * b + fr) * 256 + slot);
      vf[b] = *reinterpret_cast<const u32x4_t*>(stg + (32 + 16 * b + fr) * 256 + slot);
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      S[a][0] = mfma_16x16x32_bf16(kf[a], vf[0], S[a][0]);
      S[a][1] = mfma_16x16x32_bf16(kf[a], vf[1], S[a][1]);
      Ks[a] = mfma_16x16x32_bf16(kf[a], ones, Ks[a]);
    }
  }
  // add the two token halves: the wave with wm = 1 hands its 24 values per lane to the one with wm = 0
  f32x4_t* xch = reinterpret_cast<f32x4_t*>(stg) + lane;
  if (wm == 1) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      xch[(a * 3 + 0) * 64] = S[a][0];
      xch[(a * 3 + 1) * 64] = S[a][1];
      xch[(a * 3 + 2) * 64] = Ks[a];
    }
  }
  __syncthreads();
  if (wm == 0) {
    const f32x4_t* oth = reinterpret_cast<const f32x4_t*>(smem + (wave + 4) * 16384) + lane;
    const int head = 4 * ((n0 - ep.q_pad) >> 8) + wn;
    const int tile_m = m0 >> 8;
    const int bi = tile_m / ep.tiles_per_batch, split = tile_m - bi * ep.tiles_per_batch;
    if (head < ep.heads) {
      float* o = ep.part + (((int64_t)bi * ep.heads + head) * ep.tiles_per_batch + split) * (33 * 32);
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int dk0 = 16 * a + 4 * fg;
#pragma unroll
        for (int b = 0; b < 2; ++b)
          *reinterpret_cast<f32x4_t*>(o + (16 * b + fr) * 32 + dk0) = S[a][b] + oth[(a * 3 + b) * 64];
        if (fr == 0) *reinterpret_cast<f32x4_t*>(o + 32 * 32 + dk0) = Ks[a] + oth[(a * 3 + 2) * 64];
      }
    }
  }
}

// What bounds it: the matrix pipes' power.  At 16384 x 11200 x 2240 a k-tile takes 2160 cycles (2048 of MFMAs) at a clock
// that settles at 1.68 - 1.8 GHz on random operands; a tile's epilogue costs ~6000 cycles, ~13000 with SiLU (two quarter-rate
// transcendentals per output), and nothing else is exposed.  Against the one-wave-per-SIMD kernel with register-staged
// operands that it replaced (2657 cycles per k-tile, 8600 / 15700 of epilogue, 3200 of prologue), us on one card: 16384
// tokens, inverted conv + SiLU 646 -> 589, bias only 612 -> 562, qkv 378 -> 350, proj 147 -> 139, point conv 343 -> 333.
//
// Waves (wm, wn) = (wave / 4, wave % 4): 128 tokens x 16*NB channels each = 8 x NB tiles of v_mfma_f32_16x16x32 (the
// weight tile is the row operand: a lane owns one token and, by the order in which weight rows are placed in LDS, 8
// contiguous channels per pair of MFMA tiles).  A SIMD holds one wave of wm = 0 and one of wm = 1.
//
// LDS: two stages of a k-tile of 64 per operand, rows of 128 bytes, the 16-byte piece index XORed with (row / 2) % 8 (16
// rows of one piece then hit all banks once).  Operands arrive by direct loads (1 KB = 8 rows per wave and instruction;
// the swizzle and the weight row order are applied to the global address), no staging registers, no LDS stores.
//
// A k-tile is two phases, the first 64 and the last 64 of the wave's tokens.  A phase is a memory half -- read its
// fragments (W and A rows 0-63; A rows 64-127), request the operand part read in the phase BEFORE for two k-tiles on, wait
// until the part the NEXT phase reads has landed -- and a matrix half (16 * NB MFMAs with raised priority), each ended by a
// barrier; the waves with wm = 1 run half a phase behind, so that on every SIMD one wave multiplies while the other
// fetches.  A wave's fragment reads are waited for inside the memory half, so what one phase read may be overwritten from
// the next phase on, and a requested part has two to three phases (2000 - 3000 cycles) to land.  (Four phases, one per
// quadrant of the sub-tile, cost 2340 cycles per k-tile: 36 cycles of barrier and first-read latency per half.)  The
// order of the products of an output is the k order, as in all GEMMs of this library.
//
// Workgroups are persistent (one per compute unit, every 256th tile): the first two k-tiles of the next tile are
// requested in front of a tile's epilogue, whose rows go through 8 KB (NB = 4) per wave beside the stages and leave those to
// the loads.  At NB = 3 the four waves of a wm share the rows: a wave's 48 channels are 96 bytes, and 64-byte sectors written half by one
// wave and half by another made the epilogue 8 - 9 us a tile, whatever it computes, where the wider tile of NB = 4 takes 6.  us, so /
// now, weights cold: 2048 x 5760 x 1152 SiLU 31.3 / 28.2, 4096 x 5760 x 1152 SiLU 59.4 / 50.8, 1024 x 11200 x 2240 SiLU 51.0 / 48.5, 2916 x 6720 x
// 2240 84.6 / 78.0, 4680 x 2240 x 2240 bias 46.1 / 43.1, gated 48.3 / 47.6.  (The residual touched from within the loop, six k-tiles in front of
// the epilogue: 1 us more a launch.)
template <int EPI, int NB, int TAPS = 0, typename T = BF16>
__global__ __launch_bounds__(512) void gemm8_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                    const EpiArgs ep, uint16_t* __restrict__ C, int M, int N, int K,
                                                    int64_t lda, int64_t ldw, int64_t ldc, int tiles_t, int tiles_c,
                                                    const Taps tp) {
  constexpr bool PLANES = EPI == SANA_EPI_PLANES;
  if constexpr (PLANES) {  // this grid row's range of k-tiles
    const int z = blockIdx.y, kt0 = z * tp.split_tiles + min(z, tp.split_rem);
    A += 64 * kt0, W += 64 * kt0;
    K = min(K - 64 * kt0, 64 * (tp.split_tiles + (z < tp.split_rem)));
  }
  constexpr int BM = 256, BN = 64 * NB;
  constexpr int A_STAGE = BM * 128, W_STAGE = BN * 128, W_BASE = 2 * A_STAGE;
  constexpr int NP = (NB + 1) / 2;  // pieces of 8 (the last one of 4 if NB is odd) channels per lane and token
  constexpr int STORES = 4 * NB;    // store instructions of an epilogue, per wave
  // The epilogue's rows, 32 at a time: per wave its 16*NB channels; NB = 3, whose 96 bytes a wave are no whole 64-byte sectors: the
  // tile's 192 channels by the four waves of a wm, in two buffers.
  constexpr bool SHARED = NB == 3;
  constexpr int OUT_ROW = SHARED ? 2 * BN : 32 * NB, OUT_BYTES = 32 * OUT_ROW, OUT_BUF = SHARED ? 2 * OUT_BYTES : 0;
  static_assert(!PLANES || NB == 3, "rows of 48 floats a wave");
  static_assert(EPI != SANA_EPI_QKV_STATE || (NB == 4 && !is_f16<T> && !TAPS), "the fused qkv projection: 256-wide bf16 tiles");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[W_BASE + 2 * W_STAGE + (SHARED ? 4 : 8) * OUT_BYTES];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  // The lane index, hidden from the optimiser: what is derived from it per tile (load offsets, epilogue addresses) would
  // otherwise be hoisted out of the tile loop and occupy registers across the main loop.
  auto lane_id = [&]() {
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));
    return l;
  };

  // ---- direct loads.  A lane carries piece (lane % 8) of LDS row 8 * wave + lane / 8 (+ 64 h + 128 m for operand half h).
  // LDS row l of a wave column's 16*NB weight rows is row l % 16 = 4 g + r of MFMA tile i = l / 16 and holds channel
  // 32 (i / 2) + 8 g + 4 (i % 2) + r of the column -- or 32 (i / 2) + 4 g + r for the last tile of an odd NB.
  auto w_dst = [&](int q) {  // LDS byte offset of W load q inside a stage (a scalar)
    const int gi = wave + 8 * q;
    return gi * 8 * 128;
  };
  const int KT = (K + 63) >> 6;
  // k pieces past K (K % 64 != 0) and k-tiles past the last one are loaded from outside the resource, i.e. as zeros
  constexpr uint32_t kOut = 0x80000000u;
  const int tap_b = TAPS ? (int)(tp.stride * lda * 2) : 0;
  const int last_tap = TAPS ? K / tp.kc - 1 : 0;

  // per tile
  int m0 = 0, n0 = 0;
  const uint16_t *base_a = A, *base_w = W;          // buffer resources of the operands: first row, bytes
  int bytes_a = 0, bytes_w = 0;
  uint32_t va[2][2], vw[NB];  // vector offsets; rows past M / N lie outside the resource: zeros
  uint32_t tail_mask = 0;
  int a_kin = 0, a_tapk = 0, a_tap = 0;             // TAPS: its column inside the tap, byte offset of (tap, column), tap
  uint32_t zlast[2][2] = {{0, 0}, {0, 0}};          // TAPS == 2: rows whose last tap reads zeros

  auto poison = [&](int kl) {  // kl: the k-tile about to be loaded
    if (kl >= KT - 1) {
      const uint32_t x = kl >= KT ? kOut : tail_mask;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < 2; ++m) va[h][m] |= x;
#pragma unroll
      for (int q = 0; q < NB; ++q) vw[q] |= x;
    }
  };
  auto advance = [&](int kl) {  // the loads go on to k-tile kl
    if (TAPS) {
      a_kin += 64;
      a_tapk += 128;
      if (a_kin >= tp.kc) {
        a_kin = 0;
        a_tapk += tap_b - tp.kc * 2;
        ++a_tap;
        if (TAPS == 2 && a_tap == last_tap) {
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < 2; ++m) va[h][m] |= zlast[h][m];
        }
      }
    }
    poison(kl);
  };
  auto load_a = [&](int h, int st, int kl) {
    const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base_a), 0, bytes_a, 0x00020000);
#pragma unroll
    for (int m = 0; m < 2; ++m)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_a, (__attribute__((address_space(3))) void*)(smem + st * A_STAGE + (128 * m + 64 * h + 8 * wave) * 128), 16,
          (int)(TAPS ? va[h][m] + (uint32_t)a_tapk : va[h][m]), TAPS ? 0 : kl * 128, 0, 0);
  };
  auto load_w = [&](int st, int kl) {
    const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base_w), 0, bytes_w, 0x00020000);
#pragma unroll
    for (int q = 0; q < NB; ++q)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rsrc_w, (__attribute__((address_space(3))) void*)(smem + W_BASE + st * W_STAGE + w_dst(q)), 16, (int)vw[q], kl * 128, 0, 0);
  };

  const int total = tiles_t * tiles_c;
  auto start_tile = [&](int id) {  // resources and offsets of a tile, and the loads in front of its first phase
    gemm_tile_of(id, tiles_t, tiles_c, K >= 4096 ? 8 : 4, BM, BN, m0, n0);
    m0 = gemm_uniform(__builtin_amdgcn_readfirstlane(m0));
    n0 = gemm_uniform(__builtin_amdgcn_readfirstlane(n0));
    const int a_last = min(BM, M - m0) - 1, w_last = min(BN, N - n0) - 1;
    const int64_t a_bytes = TAPS ? (tp.rows > m0 ? ((tp.rows - m0 - 1) * lda + tp.kc) * 2 : 0) : ((int64_t)a_last * lda + K) * 2;
    base_a = gemm_uniform(A + (int64_t)m0 * lda), bytes_a = gemm_uniform((int)a_bytes);
    base_w = gemm_uniform(W + (int64_t)n0 * ldw), bytes_w = gemm_uniform((int)(((int64_t)w_last * ldw + K) * 2));
    const int lane = lane_id(), lr = lane >> 3;
    const int piece = (lane & 7) ^ (4 * (wave & 1) + (lr >> 1));  // the global k piece of this lane's place in LDS
    const uint32_t la0 = ((uint32_t)(8 * wave + lr) * (uint32_t)lda + 8 * piece) * 2;
    tail_mask = 8 * piece >= K - (KT - 1) * 64 ? kOut : 0u;
    auto w_off = [&](int q) -> uint32_t {
      const int row = 8 * (wave + 8 * q) + lr, l = row % (16 * NB), i = l >> 4, g = (l >> 2) & 3;
      const int chan = 32 * (i >> 1) + ((NB & 1) && i == NB - 1 ? 4 * g : 8 * g + 4 * (i & 1)) + (l & 3);
      return ((uint32_t)(row - l + chan) * (uint32_t)ldw + 8 * piece) * 2;
    };
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < 2; ++m) va[h][m] = la0 + (uint32_t)(128 * m + 64 * h) * (uint32_t)lda * 2;
#pragma unroll
    for (int q = 0; q < NB; ++q) vw[q] = w_off(q);
    a_kin = a_tapk = a_tap = 0;
    if (TAPS == 2 && tp.zero_last) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int r = m0 + 128 * m + 64 * h + 8 * wave + lr;
          zlast[h][m] = r < M && tp.zero_last[r / tp.stride] ? kOut : 0u;
        }
    }
    poison(0);  // (K <= 64)
    load_w(0, 0);
    load_a(0, 0, 0);
    load_a(1, 0, 0);
    advance(1);
    load_w(1, 1);
    load_a(0, 1, 1);
  };

  // ---- fragments and accumulators
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)smem;
  const int lane0 = threadIdx.x & 63, fr0 = lane0 & 15, key = (fr0 >> 1) & 7;
  uint32_t ra[2], rw[2];  // LDS byte addresses of this lane's fragments, per k-step of 32; all else is an immediate
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int col = ((4 * ks + (lane0 >> 4)) ^ key) << 4;
    ra[ks] = lds0 + (128 * wm + fr0) * 128 + col;
    rw[ks] = lds0 + W_BASE + (16 * NB * wn + fr0) * 128 + col;
  }
  u32x4_t fa[2][4], fb[2][NB];
  f32x4_t acc[NB][8];
  constexpr bool HAS_BIAS = EPI != SANA_EPI_NONE && !PLANES;

  constexpr int LOADS = 4 + NB;  // per wave and k-tile
#define G8_PIN() __builtin_amdgcn_sched_barrier(0)
  auto read_b = [&](auto st_c) {
    constexpr int O = decltype(st_c)::value * W_STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      fb[ks][0] = gemm_lds_read<O>(rw[ks]);
      fb[ks][1] = gemm_lds_read<O + 2048>(rw[ks]);
      if constexpr (NB > 2) fb[ks][2] = gemm_lds_read<O + 4096>(rw[ks]);
      if constexpr (NB > 3) fb[ks][3] = gemm_lds_read<O + 6144>(rw[ks]);
    }
  };
  auto read_a = [&](auto st_c, auto h_c) {
    constexpr int O = decltype(st_c)::value * A_STAGE + decltype(h_c)::value * 8192;
    fa[0][0] = gemm_lds_read<O>(ra[0]);
    fa[0][1] = gemm_lds_read<O + 2048>(ra[0]);
    fa[0][2] = gemm_lds_read<O + 4096>(ra[0]);
    fa[0][3] = gemm_lds_read<O + 6144>(ra[0]);
    fa[1][0] = gemm_lds_read<O>(ra[1]);
    fa[1][1] = gemm_lds_read<O + 2048>(ra[1]);
    fa[1][2] = gemm_lds_read<O + 4096>(ra[1]);
    fa[1][3] = gemm_lds_read<O + 6144>(ra[1]);
  };
  auto wait_a = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(fa[0][0]), "+v"(fa[0][1]), "+v"(fa[0][2]), "+v"(fa[0][3]), "+v"(fa[1][0]), "+v"(fa[1][1]),
                   "+v"(fa[1][2]), "+v"(fa[1][3])::"memory");
  };
  auto wait_b = [&]() {
#pragma unroll
    for (int i = 0; i < NB; ++i) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fb[0][i]), "+v"(fb[1][i])::"memory");
  };
  auto mfmas = [&](int h) {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int j = ((ks * NB + i) & 1) ? 3 - jj : jj;  // every MFMA shares an operand with the one before
          gemm_mfma<T>(acc[i][4 * h + j], fb[ks][i], fa[ks][j]);
        }
  };
  auto half_end = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    G8_PIN();
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;

  // Wait until at most N loads are outstanding -- or, while `behind` (what is waited for was requested in front of the
  // previous tile's stores), N loads and those stores.
  auto wait_loads = [&](auto n_c, bool behind) {
    constexpr int N_ = decltype(n_c)::value;
    if (behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_ + STORES) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N_) : "memory");
  };
  using L = std::integral_constant<int, LOADS>;
  auto ktile = [&](auto st_c, int kt) {  // LDS stage of this k-tile
    constexpr int ST = decltype(st_c)::value;
    // phase 1
    read_b(st_c);
    read_a(st_c, C0{});
    load_a(1, ST ^ 1, kt + 1);
    wait_loads(L{}, ST == 0 && kt == 0);
    wait_a();
    wait_b();
    half_end();
    __builtin_amdgcn_s_setprio(1);
    mfmas(0);
    __builtin_amdgcn_s_setprio(0);
    half_end();
    // phase 2
    read_a(st_c, C1{});
    advance(kt + 2);
    load_w(ST, kt + 2);
    load_a(0, ST, kt + 2);
    wait_loads(L{}, ST == 0 && kt == 0);
    wait_a();
    half_end();
    __builtin_amdgcn_s_setprio(1);
    mfmas(1);
    __builtin_amdgcn_s_setprio(0);
    half_end();
  };

  int id = blockIdx.x;
  bool fresh = true;  // no stores behind this tile's first loads
  start_tile(id);
  for (;;) {
    const int m0t = m0, n0t = n0;
    // bias of the lane's channels, packed
    u32x2_t bpk[NB];
    auto chan_of = [&](int i, int fg) {  // first of the four channels of MFMA tile i
      return n0t + wn * 16 * NB + 32 * (i >> 1) + ((NB & 1) && i == NB - 1 ? 4 * fg : 8 * fg + 4 * (i & 1));
    };
    if (HAS_BIAS) {
      const int fg = lane_id() >> 4;
#pragma unroll
      for (int i = 0; i < NB; ++i) {  // N % 8 == 0: four channels are in or out together
        const int n = chan_of(i, fg);
        bpk[i] = (ep.bias && n < N) ? *reinterpret_cast<const u32x2_t*>(ep.bias + n) : u32x2_t{0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // what the first phase reads (everything requested so far, if no stores lie in between)
    if (fresh) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS + STORES) : "memory");
    half_end();
    // the MFMAs are asm statements: whatever wrote the accumulators last is done before the first of them
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(acc[i][j]));
    asm volatile("s_nop 7" ::: "memory");
    if (wm == 1) half_end();  // half a phase behind
    int kt = K >> 30;  // 0, but not known to the compiler: it would peel the first round
#pragma clang loop unroll(disable)
    for (;;) {
      ktile(C0{}, kt);
      if (++kt >= KT) break;
      ktile(C1{}, kt);
      if (++kt >= KT) break;
    }
    // results of the last asm MFMAs; the zero-filling loads past the last k-tile
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_waitcnt vmcnt(0)" ::: "memory");
    if (wm == 0) half_end();
    half_end();
    if (HAS_BIAS) {
#pragma unroll
      for (int i = 0; i < NB; ++i) asm volatile("" : "+v"(bpk[i]));
    }

    // ---- epilogue
    const int lane = lane_id(), fr = lane & 15, fg = lane >> 4;
    id += gridDim.x;
    int n_end = N;
    float bv[4 * NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      bv[4 * i] = HAS_BIAS ? lo16<T>(bpk[i].x) : 0.f, bv[4 * i + 1] = HAS_BIAS ? hi16<T>(bpk[i].x) : 0.f;
      bv[4 * i + 2] = HAS_BIAS ? lo16<T>(bpk[i].y) : 0.f, bv[4 * i + 3] = HAS_BIAS ? hi16<T>(bpk[i].y) : 0.f;
    }
    if constexpr (EPI == SANA_EPI_QKV_STATE) {
      n_end = ep.q_cols;        // a q tile: stored like any biased output, columns past C dropped
      if (n0t >= ep.q_pad) {    // uniform per workgroup: a k / v tile.  Its epilogue needs the LDS.
        g8_state_tile(acc, bv, smem, ep, m0t, n0t, wave, lane);
        if (id >= total) return;
        __syncthreads();
        start_tile(id);
        fresh = true;
        continue;
      }
    }
    if constexpr (PLANES) {
      // 32 rows of the wave's 48 floats at a time through its eighth of the epilogue's LDS (swizzled: conflict-free both ways): whole
      // segments of 192 bytes leave, for the kernel that adds the planes up to find in the caches
      const int prows = min(128, M - m0t - 128 * wm);
      const __amdgpu_buffer_rsrc_t rsrc_p = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<float*>(C) + ((int64_t)blockIdx.y * M + m0t + 128 * wm) * N, 0, prows > 0 ? prows * N * 4 : 0, 0x00020000);
      const uint32_t corner = lds0 + W_BASE + 2 * W_STAGE + wave * 6144;
      auto place = [&](int row, int pc) -> uint32_t { return corner + row * 192 + ((pc ^ ((row >> 2) & 3)) << 4); };
      const uint32_t wr[3] = {place(fr, 2 * fg), place(fr, 2 * fg + 1), place(fr, 8 + fg)};
#pragma unroll
      for (int g = 0; g < 4; ++g) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
          gemm_lds_write<0>(wr[i], __builtin_bit_cast(u32x4_t, acc[i][2 * g]));
          gemm_lds_write<16 * 192>(wr[i], __builtin_bit_cast(u32x4_t, acc[i][2 * g + 1]));  // (the swizzle repeats every 16 rows)
        }
        u32x4_t o[6];
        int off[6];
#pragma unroll
        for (int s = 0; s < 6; ++s) {
          const int idx = lane + 64 * s, row = idx / 12, pc = idx - 12 * row, n = n0t + 48 * wn + 4 * pc;
          off[s] = n < N ? ((row + 32 * g) * N + n) * 4 : (int)kOut;
          o[s] = gemm_lds_read<0>(place(row, pc));  // (a wave's LDS accesses are in order)
        }
#pragma unroll
        for (int s = 0; s < 6; ++s) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(o[s])::"memory");
#pragma unroll
        for (int s = 0; s < 6; ++s) __builtin_amdgcn_raw_buffer_store_b128(o[s], rsrc_p, off[s], 0, 0);
      }
      return;  // (one tile a workgroup)
    }
    if (id < total) start_tile(id);
    fresh = false;
    constexpr bool GATED = EPI == SANA_EPI_GATE_RES;
    const int rows = min(BM, M - m0t);
    // (C per wave: its 128 rows reach twice as far in 32 bits as the tile's 256)
    const int wrows = min(128, rows - 128 * wm);
    const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
        C + (int64_t)(m0t + 128 * wm) * ldc, 0, wrows > 0 ? (int)((((int64_t)wrows - 1) * ldc + n_end) * 2) : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(GATED ? ep.res + (int64_t)m0t * ep.ldr : nullptr), 0,
        GATED ? (int)((((int64_t)rows - 1) * ep.ldr + n_end) * 2) : 0, 0x00020000);
    // The accumulator layout has consecutive lanes in different rows, which a store instruction would hand to memory as
    // 64 separate 16-byte pieces (measured ~100 cycles each, against ~12 for whole row segments), so the rows go
    // through the wave's own corner of LDS, 32 tokens at a time: written as the lane holds them, read back row by row.
    // (asm LDS accesses: see the fragment reads.)
    constexpr int PPR = OUT_ROW / 16;                 // 16-byte pieces of a row
    auto out_at = [&](int row, int pc) -> uint32_t {  // swizzled (NB = 3: within eight pieces): conflict-free both ways
      const int k = NB == 2 ? (row >> 2) & 3 : (row >> 1) & 7;
      return row * OUT_ROW + ((pc ^ k) << 4);
    };
    const uint32_t out0 = lds0 + W_BASE + 2 * W_STAGE + (SHARED ? wm : wave) * OUT_BYTES;
    const int pc0 = SHARED ? 2 * NB * wn : 0;         // the wave's first piece of a row
    uint32_t wr[NP], rd[NB];   // LDS addresses: written pieces of row fr; pieces read for store s of a round
    int coff[NB], roff[NB];    // byte offsets of store s of the first round in C and in the residual
    int row_s[NB], n_s[NB];
#pragma unroll
    for (int c = 0; c < NP; ++c)
      wr[c] = out0 + ((NB & 1) && c == NP - 1 ? out_at(fr, pc0 + 4 * c + (fg >> 1)) + 8 * (fg & 1) : out_at(fr, pc0 + 4 * c + fg));
#pragma unroll
    for (int s = 0; s < NB; ++s) {
      const int idx = lane + 64 * s, row = (SHARED ? 8 * wn : 0) + idx / PPR, pc = idx % PPR;
      rd[s] = out0 + out_at(row, pc);
      row_s[s] = 128 * wm + row;
      n_s[s] = n0t + (SHARED ? 0 : wn * 16 * NB) + 8 * pc;
      coff[s] = n_s[s] < n_end ? (row * (int)ldc + n_s[s]) * 2 : (int)kOut;
      roff[s] = n_s[s] < n_end ? (row_s[s] * (int)ep.ldr + n_s[s]) * 2 : (int)kOut;
    }
    u32x4_t res[GATED ? 4 : 1][NB], gate[NB];
    bool one_gate = true;
    if (GATED) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int s = 0; s < NB; ++s)
          res[g][s] = __builtin_bit_cast(
              u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, roff[s] + 64 * g * (int)ep.ldr, 0, 0));
      // gate rows: one per rows_per_gate rows of C; the whole tile has one unless a batch boundary runs through it
      const uint32_t one = is_f16<T> ? 0x3C003C00u : 0x3F803F80u;  // no gate: a plain residual add
#pragma unroll
      for (int s = 0; s < NB; ++s) gate[s] = u32x4_t{one, one, one, one};
      if (ep.gate) {
        const int g_first = m0t / ep.rows_per_gate;
        one_gate = (int64_t)(g_first + 1) * ep.rows_per_gate >= min(m0t + BM, M);
        if (one_gate) {
#pragma unroll
          for (int s = 0; s < NB; ++s)
            if (n_s[s] < n_end)
              gate[s] = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)g_first * ep.gate_stride + n_s[s]);
        }
      }
    }
    constexpr int CEPI = (GATED || EPI == SANA_EPI_QKV_STATE) ? SANA_EPI_BIAS : EPI;
    auto convert = [&](auto g_c) {  // round g: token tiles 2g, 2g + 1
      constexpr int g = decltype(g_c)::value;
      auto tile = [&](auto jj_c) {
        constexpr int jj = decltype(jj_c)::value, j = 2 * g + jj, O = jj * 16 * OUT_ROW + (g & 1) * OUT_BUF;  // (the swizzle repeats every 16 rows)
#pragma unroll
        for (int c = 0; c < NP; ++c) {
          if ((NB & 1) && c == NP - 1) {
            gemm_lds_write<O>(wr[c], g8_pack4<CEPI, T>(acc[2 * c][j], bv + 8 * c));
          } else {
            float a8[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) a8[r] = acc[2 * c][j][r], a8[4 + r] = acc[2 * c + 1 < NB ? 2 * c + 1 : 2 * c][j][r];
            gemm_lds_write<O>(wr[c], epi_pack8<CEPI, T>(a8, bv + 8 * c));
          }
        }
      };
      tile(C0{});
      tile(C1{});
    };
    auto store = [&](auto g_c) {
      constexpr int g = decltype(g_c)::value;
      if (SHARED) {  // (a wave that is here has read the round before the last, whose buffer the next round is written to)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        half_end();
      }
      u32x4_t o[NB];
#pragma unroll
      for (int s = 0; s < NB; ++s) o[s] = gemm_lds_read<(g & 1) * OUT_BUF>(rd[s]);  // (a wave's LDS accesses are in order)
#pragma unroll
      for (int s = 0; s < NB; ++s) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(o[s])::"memory");
#pragma unroll
      for (int s = 0; s < NB; ++s) {
        if constexpr (GATED) {
          u32x4_t gt8 = gate[s];
          if (ep.gate && !one_gate) {
            const int m = min(m0t + row_s[s] + 32 * g, M - 1);
            if (n_s[s] < n_end)
              gt8 = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)(m / ep.rows_per_gate) * ep.gate_stride + n_s[s]);
          }
          o[s] = gate_res8v<T>(o[s], gt8, res[g][s]);
        }
        // non-temporal: C of many tokens does not evict the operand panels from the L2s (16 x 1024 px step 8455 -> 8411 us,
        // 4096 px 8174 -> 8132)
        __builtin_amdgcn_raw_buffer_store_b128(o[s], rsrc_c, coff[s] + 64 * g * (int)ldc, 0, kBufferNt);
      }
    };
    using C2 = std::integral_constant<int, 2>;
    using C3 = std::integral_constant<int, 3>;
    convert(C0{});
    store(C0{});
    convert(C1{});
    store(C1{});
    convert(C2{});
    store(C2{});
    convert(C3{});
    store(C3{});
    if (id >= total) return;
  }
#undef G8_PIN
}

}  // namespace
}  // namespace sana
