// The 16-bit GEMM for many tokens in 256 x 288 tiles: the two-phase scheme of gemm8.h with the waves placed 4 x 2, for outputs
// whose columns fill the last round of workgroups better in this width (2240 channels: 8 x 288 instead of 12 x 192).
#pragma once
#include <type_traits>

#include "gemm_common.h"

namespace sana {
namespace {

__device__ __forceinline__ u32x2_t g288_read2(uint32_t addr) {
  u32x2_t v;
  asm volatile("ds_read_b64 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

// What bounds it: the matrix pipes' power where the rounds are full (16384 x 2240 x 5600: 306 us = 1.34 PFLOP/s with the gated
// residual at 1.88 GHz; 192-wide tiles, which it replaced there, 352), else the half phases: a k-tile takes 2670 cycles for 2304
// of MFMAs (3120 with the gated residual, at a higher clock).  What is not k-tiles -- first loads and epilogue -- is 11 k cycles a
// tile with a bias, 15 k with the gated residual, of 245 k and 288 k at K = 5600: the whole chip reads its residual and writes its rows at
// once, at memory rate.  (Counters at K = 2240 and 5600: profiles/kernels_cfg3_mfma_util.txt.)
//
// Waves (wm, wn) = (wave % 4, wave / 4): 64 tokens x 144 channels each = 4 x 9 tiles of v_mfma_f32_16x16x32 (the weight tile
// is the row operand: a lane owns one token and, by the order in which weight rows are placed in LDS, 8 contiguous channels
// per pair of MFMA tiles, 4 of the ninth).  The 128-token x 72-channel split of gemm8_kernel does not divide into MFMA tiles.
// A SIMD holds one wave of wn = 0 and one of wn = 1.
//
// LDS: two stages of a k-tile of 64, rows of 128 bytes, the 16-byte piece index XORed with (row / 2) % 8; the weight rows in
// two parts, MFMA tiles 0-3 and 4-8 of both wave columns.  A k-tile is two phases, one per part: a memory half -- read the
// fragments (A and the first part; the second part, A stays in registers), request the operands that the phase BEFORE read,
// wait until what the NEXT phase reads has landed -- and a matrix half (32 or 40 MFMAs with raised priority), each ended by a
// barrier; the waves with wn = 1 run half a phase behind.  Some of a phase's loads go out between its MFMAs (a memory half
// with six of them takes longer than the other wave's matrix half: 2 % on 16384 x 2240 x 5600).
// The order of the products of an output is the k order, as in all GEMMs of this library.
//
// Workgroups are persistent, one per compute unit: the first two k-tiles of the next tile, its bias and its gate row are
// requested in front of a tile's epilogue, whose rows go through the place of the second stage of the second weight part.
template <int EPI, int TAPS = 0, typename T = BF16>
__global__ __launch_bounds__(512) void gemm288_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                      const EpiArgs ep, uint16_t* __restrict__ C, int M, int N, int K,
                                                      int64_t lda, int64_t ldw, int64_t ldc, int tiles_t, int tiles_c,
                                                      const Taps tp) {
  constexpr int BM = 256, BN = 288, TM = 4, NT = 9, N1 = 4, N2 = 5;
  constexpr int A_STAGE = BM * 128, W1_BASE = 2 * A_STAGE, W1_STAGE = 32 * N1 * 128, W2_BASE = W1_BASE + 2 * W1_STAGE,
                W2_STAGE = 32 * N2 * 128;
  constexpr int Q1 = 2, Q2 = 3;  // load instructions (8 rows) of the weight parts per wave; of the second waves 4-7 have one less
  // epilogue: 16 rows of a wave at a time through its corner of LDS, rows padded by 16 bytes (conflict-free both ways)
  constexpr int PPR = 2 * NT, NS = (16 * PPR + 63) / 64, PITCH = 32 * NT + 16, CORNER = 16 * PITCH;
  constexpr int OUT_BASE = W2_BASE + W2_STAGE, ROW_BASE = OUT_BASE + 8 * CORNER;  // bias and gate rows, of this tile and the next
  constexpr bool HAS_BIAS = EPI != SANA_EPI_NONE, GATED = EPI == SANA_EPI_GATE_RES;
  constexpr int SMEM = ROW_BASE + (GATED ? 4096 : 2048);
  static_assert(ROW_BASE >= W2_BASE + 2 * W2_STAGE && SMEM <= 160 * 1024, "LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[SMEM];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave >> 2, wm = wave & 3;
  // The lane index, hidden from the optimiser: what is derived from it per tile (load offsets, epilogue addresses) would
  // otherwise be hoisted out of the tile loop and occupy registers across the main loop.
  auto lane_id = [&]() {
    int l = threadIdx.x & 63;
    asm volatile("" : "+v"(l));
    return l;
  };

  const int KT = (K + 63) >> 6;
  // k pieces past K (K % 64 != 0) and k-tiles past the last one are loaded from outside the resource, i.e. as zeros
  constexpr uint32_t kOut = 0x80000000u;
  const int tap_b = TAPS ? (int)(tp.stride * lda * 2) : 0;
  const int last_tap = TAPS ? K / tp.kc - 1 : 0;

  // per tile
  int m0 = 0, n0 = 0, row_sel = 0;
  const uint16_t *base_a = A, *base_w = W;          // buffer resources of the operands: first row, bytes
  int bytes_a = 0, bytes_w = 0;
  uint32_t va[TM], vw1[Q1], vw2[Q2];  // vector offsets; rows past M / N lie outside the resource: zeros
  uint32_t tail_mask = 0;
  int a_kin = 0, a_tapk = 0, a_tap = 0;             // TAPS: its column inside the tap, byte offset of (tap, column), tap
  uint32_t zlast[TM] = {0, 0, 0, 0};                // TAPS == 2: rows whose last tap reads zeros

  // One load instruction into LDS offset lds + 1024 * wave.  (The k offset is uniform, which a compiler short of scalar
  // registers forgets: the load becomes a loop over its lanes' values; and the sum is formed at each use, held ones took the
  // scalar registers.)
  auto load1 = [&](const uint16_t* base, int bytes, uint32_t v, int lds, int kl) {
    int at = wave * 1024;
    asm volatile("" : "+s"(at));
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(smem + (lds + at)), 16, (int)v,
                                             __builtin_amdgcn_readfirstlane(kl * 128), 0, 0);
  };
  constexpr int P2 = TM + Q1;            // loads of phase 2: A and the first weight part, two k-tiles on
  auto load_p2 = [&](int q, int st, int kl) {
    if (q < TM) load1(base_a, bytes_a, TAPS ? va[q] + (uint32_t)a_tapk : va[q], st * A_STAGE + 8192 * q, TAPS ? 0 : kl);
    else load1(base_w, bytes_w, vw1[q - TM], W1_BASE + st * W1_STAGE + 8192 * (q - TM), kl);
  };
  auto load_p1 = [&](int q, int st, int kl) {  // phase 1: the second weight part, one k-tile on (20 loads)
    if (q < 2 || wave < 4) load1(base_w, bytes_w, vw2[q], W2_BASE + st * W2_STAGE + 8192 * q, kl);
  };
  auto advance1 = [&](int kl) {  // the loads of phase 1 go on to k-tile kl
    if (kl >= KT - 1) {
      const uint32_t x = kl >= KT ? kOut : tail_mask;
#pragma unroll
      for (int q = 0; q < Q2; ++q) vw2[q] |= x;
    }
  };
  auto advance2 = [&](int kl) {
    if (TAPS && kl) {
      a_kin += 64;
      a_tapk += 128;
      if (a_kin >= tp.kc) {
        a_kin = 0;
        a_tapk += tap_b - tp.kc * 2;
        ++a_tap;
        if (TAPS == 2 && a_tap == last_tap) {
#pragma unroll
          for (int q = 0; q < TM; ++q) va[q] |= zlast[q];
        }
      }
    }
    if (kl >= KT - 1) {
      const uint32_t x = kl >= KT ? kOut : tail_mask;
#pragma unroll
      for (int q = 0; q < TM; ++q) va[q] |= x;
#pragma unroll
      for (int q = 0; q < Q1; ++q) vw1[q] |= x;
    }
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
    // bias and gate row of the tile's first token: older than every load that is waited for by number
    row_sel ^= 1024;
    auto load_row = [&](const uint16_t* p, int64_t at, int lds) {  // (null: zeros)
      const __amdgpu_buffer_rsrc_t rsrc =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p ? p + at : A), 0, p ? (w_last + 1) * 2 : 0, 0x00020000);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(smem + (lds + row_sel)), 16,
                                               lane * 16, 0, 0, 0);
    };
    if (HAS_BIAS && wave == 0) load_row(ep.bias, n0, ROW_BASE);
    if (GATED && wave == 1) load_row(ep.gate, (int64_t)(m0 / ep.rows_per_gate) * ep.gate_stride + n0, ROW_BASE + 2048);
    // A lane carries piece (lane % 8) of LDS row 8 * (wave + 8 q) + lane / 8 of a part
    const int piece = (lane & 7) ^ (4 * (wave & 1) + (lr >> 1));  // the global k piece of this lane's place in LDS
    tail_mask = 8 * piece >= K - (KT - 1) * 64 ? kOut : 0u;
    // LDS row l of a part's rows of a wave column is row l % 16 = 4 g + r of MFMA tile i and holds channel
    // 32 (i / 2) + 8 g + 4 (i % 2) + r of the column -- or 128 + 4 g + r for the ninth
    auto w_off = [&](int row, int n, int i0) -> uint32_t {
      const int col = row / (16 * n), l = row - col * 16 * n, i = i0 + (l >> 4), g = (l >> 2) & 3;
      const int chan = 32 * (i >> 1) + (i == NT - 1 ? 4 * g : 8 * g + 4 * (i & 1)) + (l & 3);
      return ((uint32_t)(col * 16 * NT + chan) * (uint32_t)ldw + 8 * piece) * 2;
    };
#pragma unroll
    for (int q = 0; q < TM; ++q) va[q] = ((uint32_t)(8 * wave + lr + 64 * q) * (uint32_t)lda + 8 * piece) * 2;
#pragma unroll
    for (int q = 0; q < Q1; ++q) vw1[q] = w_off(8 * wave + lr + 64 * q, N1, 0);
#pragma unroll
    for (int q = 0; q < Q2; ++q) vw2[q] = w_off(8 * wave + lr + 64 * q, N2, N1);
    a_kin = a_tapk = a_tap = 0;
    if (TAPS == 2 && tp.zero_last) {
#pragma unroll
      for (int q = 0; q < TM; ++q) {
        const int r = m0 + 64 * q + 8 * wave + lr;
        zlast[q] = r < M && tp.zero_last[r / tp.stride] ? kOut : 0u;
      }
    }
    advance2(0);  // (K <= 64)
#pragma unroll
    for (int q = 0; q < P2; ++q) load_p2(q, 0, 0);
    advance1(0);
#pragma unroll
    for (int q = 0; q < Q2; ++q) load_p1(q, 0, 0);
    advance2(1);
#pragma unroll
    for (int q = 0; q < P2; ++q) load_p2(q, 1, 1);
  };

  // ---- fragments and accumulators
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)smem;
  const int lane0 = threadIdx.x & 63, fr0 = lane0 & 15, key = (fr0 >> 1) & 7;
  uint32_t ra[2], rw1[2], rw2[2];  // LDS byte addresses of this lane's fragments, per k-step of 32; all else is an immediate
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int col = ((4 * ks + (lane0 >> 4)) ^ key) << 4;
    ra[ks] = lds0 + (16 * TM * wm + fr0) * 128 + col;
    rw1[ks] = lds0 + W1_BASE + (16 * N1 * wn + fr0) * 128 + col;
    rw2[ks] = lds0 + W2_BASE + (16 * N2 * wn + fr0) * 128 + col;
  }
  u32x4_t fa[2][TM], fb[2][N2];
  f32x4_t acc[NT][TM];

#define G288_PIN() __builtin_amdgcn_sched_barrier(0)
  // n fragments per k-step, 16 rows apart (asm reads: to the compiler an ordinary LDS read may alias the loads in flight)
  auto read_n = [&](auto& f, auto off_c, auto n_c, const uint32_t (&r)[2]) {
    constexpr int O = decltype(off_c)::value, n = decltype(n_c)::value;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      f[ks][0] = gemm_lds_read<O>(r[ks]);
      f[ks][1] = gemm_lds_read<O + 2048>(r[ks]);
      f[ks][2] = gemm_lds_read<O + 4096>(r[ks]);
      f[ks][3] = gemm_lds_read<O + 6144>(r[ks]);
      if constexpr (n > 4) f[ks][4] = gemm_lds_read<O + 8192>(r[ks]);
    }
  };
  auto wait_n = [&](auto& f, int n) {
#pragma unroll
    for (int i = 0; i < n; ++i) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0][i]), "+v"(f[1][i])::"memory");
  };
  // the MFMAs of a phase, with D load instructions (of `issue`) spread between them
  auto mfmas = [&](auto i0_c, auto n_c, auto d_c, auto issue) {
    constexpr int i0 = decltype(i0_c)::value, n = decltype(n_c)::value, D = decltype(d_c)::value, EVERY = 2 * n * TM / (D + 1);
    int m = 0;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < n; ++i)
#pragma unroll
        for (int jj = 0; jj < TM; ++jj) {
          const int j = ((ks * n + i) & 1) ? TM - 1 - jj : jj;  // every MFMA shares an operand with the one before
          gemm_mfma<T>(acc[i0 + i][j], fb[ks][i], fa[ks][j]);
          ++m;
          if (m % EVERY == 0 && m / EVERY <= D) {
            G288_PIN();
            issue(m / EVERY - 1);
            G288_PIN();
          }
        }
  };
  auto half_end = [&]() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    G288_PIN();
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;

  // Wait until at most a k-tile's loads less `left` are outstanding -- or, while `behind` (what is waited for was requested
  // in front of the previous tile's stores), those loads and the stores.
  constexpr int STORES = TM * NS, LOADS = P2 + Q2;
  auto wait_loads = [&](auto left_c, bool behind) {
    constexpr int LO = LOADS - decltype(left_c)::value, HI = LO - 1;
    if (wave >= 4) {
      if (behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(HI + STORES) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(HI) : "memory");
    } else {
      if (behind) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LO + STORES) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LO) : "memory");
    }
  };
  constexpr int D1 = 1, D2 = 3;  // loads of the phases that go out between their MFMAs
  auto ktile = [&](auto st_c, int kt) {  // LDS stage of this k-tile
    constexpr int ST = decltype(st_c)::value;
    // phase 1
    read_n(fa, std::integral_constant<int, ST * A_STAGE>{}, std::integral_constant<int, TM>{}, ra);
    read_n(fb, std::integral_constant<int, ST * W1_STAGE>{}, std::integral_constant<int, N1>{}, rw1);
    advance1(kt + 1);
#pragma unroll
    for (int q = D1; q < Q2; ++q) load_p1(q, ST ^ 1, kt + 1);
    wait_loads(std::integral_constant<int, D1>{}, ST == 0 && kt == 0);
    wait_n(fa, TM);
    wait_n(fb, N1);
    half_end();
    __builtin_amdgcn_s_setprio(1);
    mfmas(C0{}, std::integral_constant<int, N1>{}, std::integral_constant<int, D1>{}, [&](int i) { load_p1(i, ST ^ 1, kt + 1); });
    __builtin_amdgcn_s_setprio(0);
    half_end();
    // phase 2
    read_n(fb, std::integral_constant<int, ST * W2_STAGE>{}, std::integral_constant<int, N2>{}, rw2);
    advance2(kt + 2);
#pragma unroll
    for (int q = 0; q < P2 - D2; ++q) load_p2(q, ST, kt + 2);
    wait_loads(std::integral_constant<int, D2>{}, ST == 0 && kt == 0);
    wait_n(fb, N2);
    half_end();
    __builtin_amdgcn_s_setprio(1);
    mfmas(std::integral_constant<int, N1>{}, std::integral_constant<int, N2>{}, std::integral_constant<int, D2>{},
          [&](int i) { load_p2(P2 - D2 + i, ST, kt + 2); });
    __builtin_amdgcn_s_setprio(0);
    half_end();
  };

  int id = blockIdx.x;
  bool fresh = true;  // no stores behind this tile's first loads
  start_tile(id);
  for (;;) {
    const int m0t = m0, n0t = n0, rows_at = ROW_BASE + row_sel;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    // what the first phase reads (everything requested so far, if no stores lie in between)
    if (fresh) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else wait_loads(C0{}, true);
    half_end();
    // the MFMAs are asm statements: whatever wrote the accumulators last is done before the first of them
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(acc[i][j]));
    asm volatile("s_nop 7" ::: "memory");
    if (wn == 1) half_end();  // half a phase behind
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
    if (wn == 0) half_end();
    half_end();

    // ---- epilogue.  The accumulator layout has consecutive lanes in different rows, so the rows go through LDS: written as
    // the lane holds them, read back row by row, all of a row's channels together: memory gets whole segments.
    const int lane = lane_id(), fr = lane & 15, fg = lane >> 4;
    id += gridDim.x;
    const int rows = min(BM, M - m0t);
    const int wrows = min(16 * TM, rows - 16 * TM * wm);  // of this wave
    const int64_t row0 = m0t + 16 * TM * wm;
    const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
        C + row0 * ldc, 0, wrows > 0 ? (int)((((int64_t)wrows - 1) * ldc + N) * 2) : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_r = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(GATED ? ep.res + row0 * ep.ldr : nullptr), 0,
        GATED && wrows > 0 ? (int)((((int64_t)wrows - 1) * ep.ldr + N) * 2) : 0, 0x00020000);
    const uint32_t out0 = lds0 + OUT_BASE + wave * CORNER, wr = out0 + fr * PITCH + 16 * fg;
    const int nw = n0t + wn * 16 * NT;  // first channel of this wave
    constexpr int CEPI = GATED ? SANA_EPI_BIAS : EPI;
    // piece s of the lane in 16 rows: row and channel inside the wave's; formed anew for each 16 rows (registers)
    auto piece_of = [&](int s, int& row, int& ch) {
      const int idx = lane_id() + 64 * s;
      row = idx / PPR, ch = 8 * (idx - row * PPR);
      return idx < 16 * PPR && nw + ch < N;
    };
    u32x4_t res[GATED ? TM : 1][NS];
    // gate rows: one per rows_per_gate rows of C; the whole tile has one unless a batch boundary runs through it
    const bool one_gate = !GATED || !ep.gate || (int64_t)(m0t / ep.rows_per_gate + 1) * ep.rows_per_gate >= min(m0t + BM, M);
    auto fetch = [&](int j) {
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        int row, ch;
        const bool in = piece_of(s, row, ch);
        const int off = in ? ((row + 16 * j) * (int)ep.ldr + nw + ch) * 2 : (int)kOut;
        res[j][s] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, off, 0, 0));
      }
    };
    if constexpr (GATED) fetch(0), fetch(1);  // (the other two where the registers of finished rows are free)
    if (id < total) start_tile(id);
    fresh = false;
    auto finish = [&](auto j_c) {
      constexpr int j = decltype(j_c)::value;
      u32x2_t bpk[NT];
      if (HAS_BIAS) {
        const uint32_t at = lds0 + rows_at + 32 * NT * wn;
#pragma unroll
        for (int i = 0; i < NT; ++i) bpk[i] = g288_read2(at + 64 * (i >> 1) + (i == NT - 1 ? 8 * fg : 16 * fg + 8 * (i & 1)));
#pragma unroll
        for (int i = 0; i < NT; ++i) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(bpk[i])::"memory");
      }
      auto convert = [&](auto p_c) {  // MFMA tiles 2p and 2p + 1, or the ninth
        constexpr int p = decltype(p_c)::value, n = 2 * p + 1 < NT ? 2 : 1;
        float a8[8], bv[8];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int i = 2 * p + (e < n ? e : 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) a8[4 * e + r] = acc[i][j][r];
          bv[4 * e] = HAS_BIAS ? lo16<T>(bpk[i].x) : 0.f, bv[4 * e + 1] = HAS_BIAS ? hi16<T>(bpk[i].x) : 0.f;
          bv[4 * e + 2] = HAS_BIAS ? lo16<T>(bpk[i].y) : 0.f, bv[4 * e + 3] = HAS_BIAS ? hi16<T>(bpk[i].y) : 0.f;
        }
        const u32x4_t o = epi_pack8<CEPI, T>(a8, bv);
        if constexpr (n == 2) gemm_lds_write<64 * p>(wr, o);
        else gemm_lds_write<64 * p>(wr - 8 * fg, u32x2_t{o.x, o.y});
      };
      convert(C0{});
      convert(C1{});
      convert(C2{});
      convert(C3{});
      convert(std::integral_constant<int, 4>{});
      u32x4_t o[NS];
      int off[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {  // (a wave's LDS accesses are in order)
        int row, ch;
        const bool in = piece_of(s, row, ch);
        off[s] = in ? ((row + 16 * j) * (int)ldc + nw + ch) * 2 : (int)kOut;
        o[s] = gemm_lds_read<0>(out0 + (in ? row * PITCH + 2 * ch : 0));
      }
#pragma unroll
      for (int s = 0; s < NS; ++s) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(o[s])::"memory");
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        if constexpr (GATED) {
          const uint32_t one = is_f16<T> ? 0x3C003C00u : 0x3F803F80u;  // no gate: a plain residual add
          u32x4_t g8 = u32x4_t{one, one, one, one};
          if (ep.gate) {
            int row, ch;
            const bool in = piece_of(s, row, ch);
            if (one_gate) {
              g8 = gemm_lds_read<2048>(lds0 + rows_at + 2 * (wn * 16 * NT + ch));
              asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(g8)::"memory");
            } else if (in) {
              const int m = min((int)row0 + row + 16 * j, M - 1);
              g8 = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)(m / ep.rows_per_gate) * ep.gate_stride + nw + ch);
            }
          }
          o[s] = gate_res8v<T>(o[s], g8, res[j][s]);
        }
        // (cacheable: a wave column's 288 bytes end within a 64-byte sector, which the L2 puts together; with the non-temporal hint of gemm8_kernel /
        // without: a step of 16 x 1024 px 8276 / 8217 us, 4096 px 7993 / 7906, a streamed chunk 856 / 847)
        __builtin_amdgcn_raw_buffer_store_b128(o[s], rsrc_c, off[s], 0, 0);
      }
      if constexpr (GATED && j + 2 < TM) fetch(j + 2);
    };
    finish(C0{});
    finish(C1{});
    finish(C2{});
    finish(C3{});
    if (id >= total) return;
  }
#undef G288_PIN
}

}  // namespace
}  // namespace sana
