// The 16-bit GEMM for few tokens: small tiles, a ring of k-tiles in LDS filled by direct global -> LDS loads.
#pragma once
#include <type_traits>
#include <utility>

#include "gemm_common.h"

namespace sana {
namespace {

// N fragments, 2048 bytes (16 rows) apart
template <size_t N, size_t... I>
__device__ __forceinline__ void gr_read_n(u32x4_t (&f)[N], uint32_t addr, std::index_sequence<I...>) {
  ((f[I] = gemm_lds_read<2048 * (int)I>(addr)), ...);
}
// wait for the reads issued so far, tied to the registers they fill
template <size_t N>
__device__ __forceinline__ void gr_landed(u32x4_t (&f)[N]) {
  asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0])::"memory");
#pragma unroll
  for (size_t i = 1; i < N; ++i) asm volatile("" : "+v"(f[i])::"memory");
}
// Workgroup tile BM = 16 TM WM tokens x BN = 16 TN WN channels, WM x WN waves of TM x TN MFMA tiles of 16x16x32.
//
// LDS: ST stages of a k-tile of 64 ([A rows | W rows], 128 bytes a row, the 16-byte piece index XORed with (row / 2) % 8),
// filled by direct loads (1 KB = 8 rows per wave and instruction; swizzle and weight row order are applied to the global
// address).  A k-tile is two k-steps of 32: the fragments of one are read while the other's are multiplied, and the only
// barrier of a k-tile, between the two, says both that every wave has read the whole of stage kt -- so k-tile kt + ST is
// requested into it -- and that k-tile kt + 1 has landed.  Between ST - 2 and ST - 1 k-tiles are in flight all the time.
// Outputs sum their products in k order, as in all GEMMs of this library.
//
// What bounds it: operand bytes.  A compute unit takes about 107 bytes/ns from its L2, 50 when most of the chip fetches from
// behind it (some 16 KB of requests in flight against the latency of the slowest); a k-tile of 128 x 128 takes 0.32 us with
// 18 workgroups at work and 0.59 with 144, of which its MFMAs are 0.21.  More stages change nothing.  The kernels it replaced
// staged operands through registers, 0.8 - 1.1 us per k-tile, or cut K into ranges for them.  us, tokens x channels x k, before
// and now: 256 x 1152 x 1152 19.3 -> 6.5, 256 x 3456 x 1152 18.1 -> 8.0, 256 x 1152 x 2880 22.1 -> 11.6, 1024 x 2240 x 2240
// 29.0 -> 23.4, 2048 x 1152 x 1152 20.0 -> 11.9, 2048 x 2240 x 2240 35.0 -> 29.6, 4096 x 1152 x 2880 41.8 -> 35.4.
template <int WM, int WN, int TM, int TN, int ST, int EPI, typename T>
__global__ __launch_bounds__(64 * WM * WN) void gemm_ring_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                                 const EpiArgs ep, uint16_t* __restrict__ C, int M, int N,
                                                                 int K, int64_t lda, int64_t ldw, int64_t ldc, int tiles_t,
                                                                 int tiles_c, int group) {
  constexpr int NW = WM * WN, BM = 16 * TM * WM, BN = 16 * TN * WN;
  constexpr int STAGE = (BM + BN) * 128, W_OFF = BM * 128;
  constexpr int NA = BM / 8 / NW, NWP = BN / 8 / NW, LOADS = NA + NWP;  // load instructions per wave and k-tile
  static_assert(NA * 8 * NW == BM && NWP * 8 * NW == BN && NW % 2 == 0 && TN % 2 == 0 && ST >= 3, "tile shape");
  constexpr int PITCH = 32 * TN + 16, OUT_BYTES = 16 * PITCH;           // epilogue: 16 finished rows of a wave
  static_assert(NW * OUT_BYTES <= ST * STAGE, "the epilogue's rows fit in the ring");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[ST * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int fr = lane & 15, fg = lane >> 4, lr = lane >> 3;

  int m0, n0;
  gemm_tile_of(blockIdx.x, tiles_t, tiles_c, group, BM, BN, m0, n0);

  // ---- direct loads: rows past M / N, k pieces past K and k-tiles past the last one lie outside the resource: zeros
  constexpr uint32_t kOut = 0x80000000u;
  const int KT = (K + 63) >> 6;
  const int a_last = min(BM, M - m0) - 1, w_last = min(BN, N - n0) - 1;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(A + (int64_t)m0 * lda), 0, (int)(((int64_t)a_last * lda + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(W + (int64_t)n0 * ldw), 0, (int)(((int64_t)w_last * ldw + K) * 2), 0x00020000);
  const int piece = (lane & 7) ^ (4 * (wave & 1) + (lr >> 1));  // the global k piece of this lane's place in LDS
  const uint32_t tail_mask = 8 * piece >= K - (KT - 1) * 64 ? kOut : 0u;
  uint32_t va[NA], vw[NWP];
#pragma unroll
  for (int j = 0; j < NA; ++j) va[j] = ((uint32_t)(8 * (wave + NW * j) + lr) * (uint32_t)lda + 8 * piece) * 2;
#pragma unroll
  for (int j = 0; j < NWP; ++j) {
    // LDS row l of a wave column's 16*TN weight rows is row l % 16 = 4 g + r of MFMA tile i = l / 16 and holds channel
    // 32 (i / 2) + 8 g + 4 (i % 2) + r of the column: a lane ends with 8 contiguous channels per pair of MFMA tiles
    const int row = 8 * (wave + NW * j) + lr, l = row % (16 * TN), i = l >> 4, g = (l >> 2) & 3;
    const int chan = 32 * (i >> 1) + 8 * g + 4 * (i & 1) + (l & 3);
    vw[j] = ((uint32_t)(row - l + chan) * (uint32_t)ldw + 8 * piece) * 2;
  }
  auto past_end = [&](int kl) {  // in front of the loads of k-tile kl (uniform; idempotent)
    if (kl >= KT - 1) {
      const uint32_t x = kl >= KT ? kOut : tail_mask;
#pragma unroll
      for (int j = 0; j < NA; ++j) va[j] |= x;
#pragma unroll
      for (int j = 0; j < NWP; ++j) vw[j] |= x;
    }
  };
  auto load1 = [&](int j, int st, int kl) {  // load instruction j of a k-tile
    unsigned char* dst = smem + st * STAGE + wave * 1024 + NW * 1024 * j;
    if (j < NA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)dst, 16, (int)va[j], kl * 128, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (__attribute__((address_space(3))) void*)dst, 16, (int)vw[j - NA], kl * 128, 0, 0);
  };
  constexpr int L1 = (LOADS + 1) / 2;  // a k-tile's loads go out in two parts, one per k-step
#pragma unroll
  for (int s = 0; s < ST; ++s) {
    past_end(s);
#pragma unroll
    for (int j = 0; j < (s + 1 < ST ? LOADS : L1); ++j) load1(j, s, s);
  }

  // the lane's bias values, packed (8 channels per pair of MFMA tiles); waited for with the first k-tiles
  constexpr bool HAS_BIAS = EPI != SANA_EPI_NONE, GATED = EPI == SANA_EPI_GATE_RES;
  u32x4_t bpk[TN / 2];
#pragma unroll
  for (int c = 0; c < TN / 2; ++c) {
    const int n = n0 + wn * 16 * TN + 32 * c + 8 * fg;  // N % 8 == 0: eight channels are in or out together
    bpk[c] = u32x4_t{0u, 0u, 0u, 0u};
    if (HAS_BIAS && ep.bias && n < N) bpk[c] = *reinterpret_cast<const u32x4_t*>(ep.bias + n);
  }

  // ---- fragments (asm reads: to the compiler an ordinary LDS read may alias the loads in flight) and accumulators
  const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)smem;
  const int key = (fr >> 1) & 7;
  uint32_t ra[2], rw[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    const int col = ((4 * ks + fg) ^ key) << 4;
    ra[ks] = lds0 + (16 * TM * wm + fr) * 128 + col;
    rw[ks] = lds0 + W_OFF + (16 * TN * wn + fr) * 128 + col;
  }
  u32x4_t fa[2][TM], fb[2][TN];
  f32x4_t acc[TN][TM];
  // One k-step: the MFMAs of fragment set KS with, between them, the reads of the other set from stage st and the loads
  // j0 .. j1 - 1 of k-tile kl.  A memory instruction waits at issue while its pipe is busy, and what stands behind it in
  // the wave waits with it; one or two per MFMA keep all three pipes going.
  constexpr int NM = TM * TN, NR = TM + TN;
  auto kstep = [&](auto ks_c, int st, auto j0_c, auto j1_c, int stl, int kl) {
    constexpr int KS = decltype(ks_c)::value, J0 = decltype(j0_c)::value, J1 = decltype(j1_c)::value;
    constexpr int RPM = (2 * NR + NM - 1) / NM > 2 ? (2 * NR + NM - 1) / NM : 2;  // reads per MFMA: done in the first half
    constexpr int RSLOTS = (NR + RPM - 1) / RPM, LSLOTS = NM > RSLOTS ? NM - RSLOTS : 1;
    const uint32_t oa = ra[KS ^ 1] + st * STAGE, ob = rw[KS ^ 1] + st * STAGE;
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      const int i = m / TM, j = (i & 1) ? TM - 1 - m % TM : m % TM;  // every MFMA shares an operand with the one before
      gemm_mfma<T>(acc[i][j], fb[KS][i], fa[KS][j]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = RPM * m; r < RPM * (m + 1) && r < NR; ++r) {
        if (r < TM) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[KS ^ 1][r]) : "v"(oa), "n"(2048 * r));
        else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[KS ^ 1][r - TM]) : "v"(ob), "n"(2048 * (r - TM)));
      }
#pragma unroll
      for (int q = J0; q < J1; ++q)
        if ((NM > RSLOTS ? RSLOTS + (q - J0) * LSLOTS / (J1 - J0) : NM - 1) == m) load1(q, stl, kl);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
#define GR_PIN() __builtin_amdgcn_sched_barrier(0)
#define GR_BARRIER() do { asm volatile("" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); GR_PIN(); } while (0)

#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // (the bias loads are younger than the ring's: all but k-tile 0 may be outstanding, and fewer is safe)
  using J0 = std::integral_constant<int, 0>;
  using J1 = std::integral_constant<int, L1>;
  using J2 = std::integral_constant<int, LOADS>;
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * LOADS + L1) : "memory");
  GR_BARRIER();
  gr_read_n(fa[0], ra[0], std::make_index_sequence<TM>{});
  gr_read_n(fb[0], rw[0], std::make_index_sequence<TN>{});
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(acc[i][j]));
  asm volatile("s_nop 7" ::: "memory");  // the MFMAs are asm statements: the zeroing is done before the first of them
  gr_landed(fa[0]);
  gr_landed(fb[0]);
  int st = 0, last = ST - 1;  // stage of k-tile kt; of kt - 1, being refilled with k-tile kt + ST - 1
#pragma clang loop unroll(disable)
  for (int kt = 0; kt < KT; ++kt) {
    kstep(C0{}, st, J1{}, J2{}, last, kt + ST - 1);
    gr_landed(fa[1]);
    gr_landed(fb[1]);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * LOADS) : "memory");  // k-tile kt + 1 (this wave's part of it)
    GR_BARRIER();
    const int nxt = st + 1 == ST ? 0 : st + 1;
    past_end(kt + ST);
    kstep(C1{}, nxt, J0{}, J1{}, st, kt + ST);
    gr_landed(fa[0]);
    gr_landed(fb[0]);
    last = st;
    st = nxt;
  }
  // results of the last asm MFMAs; the zero-filling loads past the last k-tile
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_waitcnt vmcnt(0)" ::: "memory");
  GR_BARRIER();
#undef GR_PIN
#undef GR_BARRIER

  // ---- epilogue: 16 tokens at a time through the wave's own corner of LDS (rows padded by 16 bytes: conflict-free both
  // ways), so that a store instruction writes whole row segments.
  constexpr int PPR = 2 * TN, NS = TN / 2;  // 16-byte pieces of a row; store instructions per 16 rows
  const int rows = min(BM, M - m0);
  const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
      C + (int64_t)m0 * ldc, 0, (int)((((int64_t)rows - 1) * ldc + N) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(GATED ? ep.res + (int64_t)m0 * ep.ldr : nullptr), 0,
      GATED ? (int)((((int64_t)rows - 1) * ep.ldr + N) * 2) : 0, 0x00020000);
  const uint32_t out0 = lds0 + wave * OUT_BYTES, wr = out0 + fr * PITCH + 16 * fg;
  uint32_t rd[NS];
  int row_s[NS], n_s[NS], coff[NS], roff[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int idx = lane + 64 * s, row = idx / PPR, pc = idx % PPR;
    rd[s] = out0 + row * PITCH + 16 * pc;
    row_s[s] = 16 * TM * wm + row;
    n_s[s] = n0 + wn * 16 * TN + 8 * pc;
    coff[s] = n_s[s] < N ? (row_s[s] * (int)ldc + n_s[s]) * 2 : (int)kOut;
    roff[s] = n_s[s] < N ? (row_s[s] * (int)ep.ldr + n_s[s]) * 2 : (int)kOut;
  }
  u32x4_t res[GATED ? TM : 1][NS], gate[NS];
  bool one_gate = true;
  if (GATED) {
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int s = 0; s < NS; ++s)
        res[j][s] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, roff[s] + 32 * j * (int)ep.ldr, 0, 0));
    // gate rows: one per rows_per_gate rows of C; the whole tile has one unless a batch boundary runs through it
    const int g_first = m0 / ep.rows_per_gate;
    one_gate = (int64_t)(g_first + 1) * ep.rows_per_gate >= min(m0 + BM, M);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      gate[s] = u32x4_t{0u, 0u, 0u, 0u};
      if (one_gate && n_s[s] < N)
        gate[s] = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)g_first * ep.gate_stride + n_s[s]);
    }
  }
  float bv[TN / 2][8];
#pragma unroll
  for (int c = 0; c < TN / 2; ++c)
#pragma unroll
    for (int e = 0; e < 4; ++e) bv[c][2 * e] = lo16<T>(bpk[c][e]), bv[c][2 * e + 1] = hi16<T>(bpk[c][e]);
#pragma unroll
  for (int j = 0; j < TM; ++j) {
#pragma unroll
    for (int c = 0; c < TN / 2; ++c) {
      float a8[8];
#pragma unroll
      for (int r = 0; r < 4; ++r) a8[r] = acc[2 * c][j][r], a8[4 + r] = acc[2 * c + 1][j][r];
      gemm_lds_write<0>(wr + 64 * c, epi_pack8<GATED ? SANA_EPI_BIAS : EPI, T>(a8, bv[c]));
    }
    u32x4_t o[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) o[s] = gemm_lds_read<0>(rd[s]);  // (a wave's LDS accesses are in order)
#pragma unroll
    for (int s = 0; s < NS; ++s) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(o[s])::"memory");
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      if (GATED) {
        u32x4_t g8 = gate[s];
        if (!one_gate && n_s[s] < N) {
          const int m = min(m0 + row_s[s] + 16 * j, M - 1);
          g8 = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)(m / ep.rows_per_gate) * ep.gate_stride + n_s[s]);
        }
        o[s] = gate_res8v<T>(o[s], g8, res[j][s]);
      }
      // (cacheable: with the non-temporal hint of the many-token kernel a 512 px step takes 866 us instead of 845, 1024 - 2048
      // tokens 0.5 % less)
      __builtin_amdgcn_raw_buffer_store_b128(o[s], rsrc_c, coff[s] + 32 * j * (int)ldc, 0, 0);
    }
  }
}

}  // namespace
}  // namespace sana
