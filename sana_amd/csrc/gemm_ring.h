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
// behind a wait: the registers that the reads before it filled
template <size_t N>
__device__ __forceinline__ void gr_tie(u32x4_t (&f)[N]) {
#pragma unroll
  for (size_t i = 0; i < N; ++i) asm volatile("" : "+v"(f[i])::"memory");
}
// x is computed before this point, not later
__device__ __forceinline__ void gr_here(uint32_t& x) { asm volatile("" : "+v"(x)); }
template <typename F, int... I>
__device__ __forceinline__ void gr_each(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// RANGES: sums over ranges of k (KRanges in gemm_common.h), added up here.
// Workgroup tile BM = 16 TM WM tokens x BN = 16 TN WN channels, WM x WN waves of TM x TN MFMA tiles of 16x16x32.
//
// LDS: ST stages of a k-tile of 64 ([A rows | W rows], 128 bytes a row, the 16-byte piece index XORed with (row / 2) % 8),
// filled by direct loads (1 KB = 8 rows per wave and instruction; swizzle and weight row order are applied to the global
// address).  Between ST - 2 and ST - 1 k-tiles are in flight all the time.  Outputs sum their products in k order, as in all
// GEMMs of this library.  Two loops (which of them runs: gemm_ring.hip):
//  * WHOLE: a wave holds the fragments of two whole k-tiles: a pass multiplies one, reads the next and requests k-tile kt + ST
//    into the stage that the pass before has emptied; the one barrier at its end says both that every wave has read stage
//    kt + 1 and that k-tile kt + 2 has landed.
//  * else: of two k-steps of 32; those of one are read while the other's are multiplied, the barrier between the two says
//    that every wave has read the whole of stage kt -- so k-tile kt + ST is requested into it -- and that k-tile kt + 1 has landed.
//
// What bounds it.  Few workgroups: latency -- 1.0 - 1.5 us to the first k-tile, then the loop's waits: a k-tile of 128 x 128 takes
// 512 cycles of MFMAs, 512 of direct loads (64 bytes a cycle into LDS; LDS reads run at 254) and 660 in rounds of the ring,
// where the half-k-tile loop needs 753.  Weights that come from HBM double the time of a k-tile without the prefetch where several
// token tiles read them (2048 x 1152 x 2880 in 128 x 128: 27.4 us, with it 21.9, from the caches 19.9); on weights that the caches
// hold it costs 0.5 us.  From about 200 workgroups on the clock gives way (2.4 GHz -> 1.8 - 2.1) and a denser loop gains little.
// A branch in front of the first load costs a launch 0.3 us: a row is compared with BN only where rows are padded.  us, weights
// cold, the kernels before the whole k-tiles / now: 256 x 1152 x 2880 15.3 / 10.4 (halved tiles, gemm_ring.hip), 1024 x 2240 x 2240
// 23.7 / 18.5, 2048 x 1152 x 2880 28.7 / 21.8, 200 x 3456 x 1152 6.8 / 6.9; slower: 288 x 6720 x 2240 19.5 / 20.6, 150 x 11200 x 2240
// 21.0 / 22.2 (96 x 128 instead of 128 x 128: a last token tile of few rows, which the plan's tile times do not know), 1260 x 5760 x
// 1152 21.1 / 21.9 (256 x 128).
template <int WM, int WN, int TM, int TN, int ST, bool WHOLE, bool RANGES, int EPI, typename T>
__global__ __launch_bounds__(64 * WM * WN) void gemm_ring_kernel(const uint16_t* __restrict__ A, const uint16_t* __restrict__ W,
                                                                 const EpiArgs ep, uint16_t* __restrict__ C, int M, int N,
                                                                 int K, int64_t lda, int64_t ldw, int64_t ldc, int tiles_t,
                                                                 int tiles_c, int group, uint32_t prefetch, const KRanges kr) {
  constexpr int NW = WM * WN, BM = 16 * TM * WM, BN = 16 * TN * WN;
  // load instructions per wave and k-tile (rows past the tile's, where its rows are no whole number of them, read as zeros)
  constexpr int NA = (BM / 8 + NW - 1) / NW, NWP = (BN / 8 + NW - 1) / NW, LOADS = NA + NWP;
  constexpr int W_OFF = NA * NW * 1024, STAGE = W_OFF + NWP * NW * 1024;
  static_assert(NW % 2 == 0 && TN % 2 == 0 && ST >= 3 && ST * STAGE <= 163840, "tile shape");
  constexpr int PITCH = 32 * TN + 16, OUT_BYTES = 16 * PITCH;           // epilogue: 16 finished rows of a wave
  static_assert(NW * OUT_BYTES <= ST * STAGE, "the epilogue's rows fit in the ring");
  constexpr int PF = WHOLE ? 4 : 0;  // prefetch loads a thread
  constexpr int L1 = (LOADS + 1) / 2;  // (!WHOLE: a k-tile's loads go out in two parts, one per k-step)
  __shared__ __attribute__((aligned(1024))) unsigned char smem[ST * STAGE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int fr = lane & 15, fg = lane >> 4, lr = lane >> 3;

  int m0, n0;
  if (!WHOLE) asm volatile("" ::"s"(A), "s"(W), "s"(lda), "s"(ldw), "s"(M), "s"(N), "s"(K), "s"(tiles_t), "s"(tiles_c), "s"(group));  // (the arguments in one wait)
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
  // LDS row l of a wave column's 16*TN weight rows is row l % 16 = 4 g + r of MFMA tile i = l / 16 and holds channel
  // 32 (i / 2) + 8 g + 4 (i % 2) + r of the column: a lane ends with 8 contiguous channels per pair of MFMA tiles
#pragma unroll
  for (int j = 0; j < NWP; ++j) {
    const int row = 8 * (wave + NW * j) + lr, l = row % (16 * TN), i = l >> 4, g = (l >> 2) & 3;
    const int chan = 32 * (i >> 1) + 8 * g + 4 * (i & 1) + (l & 3);
    vw[j] = BN % (8 * NW) == 0 || row < BN ? ((uint32_t)(row - l + chan) * (uint32_t)ldw + 8 * piece) * 2 : kOut;
  }
  auto past_end = [&](int kl) {  // in front of the loads of k-tile kl (idempotent)
    if (!WHOLE && __builtin_expect(kl < KT - 1, 1)) return;
    const uint32_t x = kl >= KT ? kOut : kl == KT - 1 ? tail_mask : 0u;
#pragma unroll
    for (int j = 0; j < NA; ++j) va[j] |= x;
#pragma unroll
    for (int j = 0; j < NWP; ++j) vw[j] |= x;
  };
  auto load1 = [&](int j, int st, int kl) {  // load instruction j of k-tile kl into stage st
    unsigned char* dst = smem + st * STAGE + wave * 1024 + NW * 1024 * j;  // (W's rows stand behind A's NA * 8 * NW)
    if (j < NA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_a, (__attribute__((address_space(3))) void*)dst, 16, (int)va[j], kl * 128, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc_w, (__attribute__((address_space(3))) void*)dst, 16, (int)vw[j - NA], kl * 128, 0, 0);
  };
#pragma unroll
  for (int s = 0; s < ST; ++s) {
    past_end(s);
#pragma unroll
    for (int j = 0; j < (WHOLE || s + 1 < ST ? LOADS : L1); ++j) load1(j, s, s);
    if (!WHOLE) {  // the next stages' offsets are computed behind these loads (all of them in front: 1 us a launch)
#pragma unroll
      for (int j = 0; j < NA; ++j) asm volatile("" : "+v"(va[j])::"memory");
#pragma unroll
      for (int j = 0; j < NWP; ++j) asm volatile("" : "+v"(vw[j])::"memory");
    }
  }
  if (WHOLE) past_end(ST);
  // W's first `prefetch` bytes (dense: all of it; or none) towards the caches, an equal run of 128-byte lines per workgroup: k-tile by
  // k-tile it comes from HBM in pieces of one line a row, each with a row access of its own and a latency that ST - 1 k-tiles do
  // not cover.
  uint32_t pf[WHOLE ? PF : 1];
  if (WHOLE) {
    // (the waits count these loads as younger than the ring's: none of them moves in front of one)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t run = (((prefetch + 127) >> 7) + gridDim.x - 1) / gridDim.x;
    const __amdgpu_buffer_rsrc_t rsrc_all = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(W), 0, (int)prefetch, 0x00020000);
#pragma unroll
    for (int p = 0; p < PF; ++p) {
      const uint32_t i = p * 64 * NW + threadIdx.x;
      pf[p] = __builtin_amdgcn_raw_buffer_load_b32(rsrc_all, i < run ? (int)((blockIdx.x * run + i) * 128u) : (int)kOut, 0, 0);
    }
  }

  // the lane's bias values, packed (8 channels per pair of MFMA tiles)
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
  uint32_t ra[ST][2], rw[ST][2];  // per stage and k-step
#pragma unroll
  for (int s = 0; s < ST; ++s)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int col = ((4 * ks + fg) ^ key) << 4;
      ra[s][ks] = lds0 + s * STAGE + (16 * TM * wm + fr) * 128 + col;
      rw[s][ks] = lds0 + s * STAGE + W_OFF + (16 * TN * wn + fr) * 128 + col;
      if (WHOLE) gr_here(ra[s][ks]), gr_here(rw[s][ks]);
    }
  constexpr int KS = WHOLE ? 2 : 1;    // k-steps of a fragment set
  u32x4_t fa[2][KS][TM], fb[2][KS][TN];
  f32x4_t acc[TN][TM];
  auto landed = [&](auto b_c) {
    constexpr int B = decltype(b_c)::value;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      gr_tie(fa[B][ks]);
      gr_tie(fb[B][ks]);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
#define GR_BARRIER() do { asm volatile("" ::: "memory"); __builtin_amdgcn_s_barrier(); asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); } while (0)
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(WHOLE ? (ST - 1) * LOADS + PF : (ST - 2) * LOADS + L1) : "memory");  // (a bias in flight: stricter)
  GR_BARRIER();
#pragma unroll
  for (int ks = 0; ks < KS; ++ks) {
    gr_read_n(fa[0][ks], ra[0][ks], std::make_index_sequence<TM>{});
    gr_read_n(fb[0][ks], rw[0][ks], std::make_index_sequence<TN>{});
  }
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(acc[i][j]));
  asm volatile("s_nop 7" ::: "memory");  // the MFMAs are asm statements: the zeroing is done before the first of them
  landed(C0{});
  // what the epilogue reads, requested in front of the last passes
  constexpr int PPR = 2 * TN, NS = TN / 2;  // 16-byte pieces of a row; store instructions per 16 rows
  const int rows = min(BM, M - m0);
  const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
      C + (int64_t)m0 * ldc, 0, (int)((((int64_t)rows - 1) * ldc + N) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(GATED ? ep.res + (int64_t)m0 * ep.ldr : nullptr), 0,
      GATED ? (int)((((int64_t)rows - 1) * ep.ldr + N) * 2) : 0, 0x00020000);
  u32x4_t res[GATED ? TM : 1][NS], gate[NS];
  bool one_gate = true;
  auto request = [&]() {
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int idx = lane + 64 * s, row = 16 * TM * wm + idx / PPR, n = n0 + wn * 16 * TN + 8 * (idx % PPR);
      const int off = n < N ? (row * (int)ep.ldr + n) * 2 : (int)kOut;
#pragma unroll
      for (int j = 0; j < TM; ++j)
        res[j][s] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, off + 32 * j * (int)ep.ldr, 0, 0));
    }
    // gate rows: one per rows_per_gate rows of C; the whole tile has one unless a batch boundary runs through it
    const int g_first = m0 / ep.rows_per_gate;
    one_gate = (int64_t)(g_first + 1) * ep.rows_per_gate >= min(m0 + BM, M);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int n = n0 + wn * 16 * TN + 8 * ((lane + 64 * s) % PPR);
      gate[s] = u32x4_t{0u, 0u, 0u, 0u};
      if (one_gate && n < N) gate[s] = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)g_first * ep.gate_stride + n);
    }
  };
  constexpr bool EARLY = WHOLE && TN <= 4 && !(RANGES && TM * TN > 8);  // (registers)

  // RANGES: behind the last k-tile of a range of k (but the last one) its sum is added to those before it.
  f32x4_t sum[RANGES ? TN : 1][RANGES ? TM : 1];
  int range = 1, range_end = kr.tiles + (kr.rem > 0);
  if constexpr (RANGES) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) sum[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  auto end_range = [&](int done) {  // done: k-tiles multiplied so far
    if constexpr (RANGES) {
      if (done != range_end || range >= kr.ranges) return;
      asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");  // results of the last asm MFMAs
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          asm volatile("" : "+v"(acc[i][j]));
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
      for (int i = 0; i < TN; ++i)
#pragma unroll
        for (int j = 0; j < TM; ++j) asm volatile("" : "+v"(acc[i][j]));
      asm volatile("s_nop 7" ::: "memory");
      range_end += kr.tiles + (range < kr.rem);
      ++range;
    }
  };

  int kt = 0;
  if constexpr (WHOLE) {
    // The MFMAs of k-tile kt from fragment set B with, between them, the reads of k-tile kt + 1 into the other set and the loads of
    // k-tile kl = kt + ST into the stage of kt.  A memory instruction waits at issue while its pipe is busy, and what stands
    // behind it in the wave waits with it: they are spread over the MFMAs, the reads, which are waited for at the end, in front.
    // ROUND: st is a constant and kl not past the last whole k-tile.
    constexpr int NM = 2 * TM * TN, NR = 2 * (TM + TN), RPM = (NR + NM - 1) / NM;
    static_assert((LOADS - 1) * NM / LOADS <= NM - 2, "loads of a k-tile in front of the next one's offsets");
    auto ktile = [&](auto b_c, auto round_c, int st, int kl) {
      constexpr int B = decltype(b_c)::value;
      constexpr bool ROUND = decltype(round_c)::value;
      const int nxt = st + 1 == ST ? 0 : st + 1;
      uint32_t oa[2], ob[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        if (ROUND) oa[x] = ra[nxt][x], ob[x] = rw[nxt][x];
        else oa[x] = ra[0][x] + nxt * STAGE, ob[x] = rw[0][x] + nxt * STAGE;
      }
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const int ks = m / (TM * TN), i = m % (TM * TN) / TM, jj = m % TM, j = ((ks * TN + i) & 1) ? TM - 1 - jj : jj;
        gemm_mfma<T>(acc[i][j], fb[B][ks][i], fa[B][ks][j]);  // (every MFMA shares an operand with the one before)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = RPM * m; r < RPM * (m + 1) && r < NR; ++r) {
          const int rk = r / (TM + TN), q = r % (TM + TN);
          if (q < TM) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[B ^ 1][rk][q]) : "v"(oa[rk]), "n"(2048 * q));
          else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[B ^ 1][rk][q - TM]) : "v"(ob[rk]), "n"(2048 * (q - TM)));
        }
#pragma unroll
        for (int q = 0; q < LOADS; ++q)
          if (q * NM / LOADS == m) load1(q, st, kl);
        if (!ROUND && m == NM - 2 && __builtin_expect(kl + 1 >= KT - 1, 0)) past_end(kl + 1);  // (the pass's last load is out)
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    using Cpf = std::integral_constant<int, PF>;
    // A pass, to the point where its successor's fragments and (this wave's part of) k-tile kt + 2 have landed.  young: loads in
    // flight behind those of the ring's first ST k-tiles.  The fragments land before any branch: nothing is moved while in flight.
    auto pass = [&](auto b_c, auto round_c, auto young_c, int st, int kt) {
      constexpr int B = decltype(b_c)::value;
      ktile(b_c, round_c, st, kt + ST);
      landed(std::integral_constant<int, B ^ 1>{});
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * LOADS + decltype(young_c)::value) : "memory");
      GR_BARRIER();
    };
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * LOADS + PF) : "memory");
    GR_BARRIER();
    constexpr int HEAD = (ST - 2) & ~1;  // passes that wait for k-tiles requested in front of the prefetch
    gr_each([&](auto i_c) { constexpr int I = decltype(i_c)::value;
                            pass(std::integral_constant<int, I & 1>{}, C0{}, Cpf{}, I, I); },
            std::make_integer_sequence<int, HEAD>{});  // (past K: products of zeros)
    kt = HEAD;
    // Whole rounds of the ring with the end of K out of sight.  Nothing but an MFMA stands behind a barrier then, and no address is
    // computed: a taken branch and the address arithmetic there cost 100 - 150 cycles a k-tile.
    constexpr int UN = ST % 2 ? 2 * ST : ST;
    const int whole = K >> 6;
#pragma clang loop unroll(disable)
    for (; kt + UN + ST <= whole; kt += UN)
      gr_each([&](auto i_c) { constexpr int I = decltype(i_c)::value;
                              pass(std::integral_constant<int, I & 1>{}, C1{}, C0{}, (HEAD + I) % ST, kt + I);
                              end_range(kt + I + 1); },
              std::make_integer_sequence<int, UN>{});
    if (GATED && EARLY) request();
    int st = HEAD;  // (rounds of the ring end where they began)
    past_end(kt + ST);
#pragma clang loop unroll(disable)
    for (; kt < KT; kt += 2) {  // (an odd number of them: one pass of zeros)
      pass(C0{}, C0{}, C0{}, st, kt);
      end_range(kt + 1);
      st = st + 1 == ST ? 0 : st + 1;
      pass(C1{}, C0{}, C0{}, st, kt + 1);
      end_range(kt + 2);
      st = st + 1 == ST ? 0 : st + 1;
    }
#pragma unroll
    for (int p = 0; p < PF; ++p) asm volatile("" ::"v"(pf[p]));
  } else {
    // One k-step: the MFMAs of fragment set S with, between them, the reads of the other set from stage st and the loads
    // j0 .. j1 - 1 of k-tile kl (see WHOLE for the order).
    constexpr int NM = TM * TN, NR = TM + TN;
    auto kstep = [&](auto s_c, int st, auto j0_c, auto j1_c, int stl, int kl) {
      constexpr int S = decltype(s_c)::value, J0 = decltype(j0_c)::value, J1 = decltype(j1_c)::value;
      constexpr int RPM = (2 * NR + NM - 1) / NM > 2 ? (2 * NR + NM - 1) / NM : 2;  // reads per MFMA: done in the first half
      constexpr int RSLOTS = (NR + RPM - 1) / RPM, LSLOTS = NM > RSLOTS ? NM - RSLOTS : 1;
      const uint32_t oa = ra[0][S ^ 1] + st * STAGE, ob = rw[0][S ^ 1] + st * STAGE;
#pragma unroll
      for (int m = 0; m < NM; ++m) {
        const int i = m / TM, j = (i & 1) ? TM - 1 - m % TM : m % TM;
        gemm_mfma<T>(acc[i][j], fb[S][0][i], fa[S][0][j]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = RPM * m; r < RPM * (m + 1) && r < NR; ++r) {
          if (r < TM) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fa[S ^ 1][0][r]) : "v"(oa), "n"(2048 * r));
          else asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(fb[S ^ 1][0][r - TM]) : "v"(ob), "n"(2048 * (r - TM)));
        }
#pragma unroll
        for (int q = J0; q < J1; ++q)
          if ((NM > RSLOTS ? RSLOTS + (q - J0) * LSLOTS / (J1 - J0) : NM - 1) == m) load1(q, stl, kl);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    using J1 = std::integral_constant<int, L1>;
    using J2 = std::integral_constant<int, LOADS>;
    int st = 0, last = ST - 1;  // stage of k-tile kt; of kt - 1, being refilled with k-tile kt + ST - 1
#pragma clang loop unroll(disable)
    for (; kt < KT; ++kt) {
      kstep(C0{}, st, J1{}, J2{}, last, kt + ST - 1);
      landed(C1{});
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((ST - 2) * LOADS) : "memory");  // k-tile kt + 1 (this wave's part of it)
      GR_BARRIER();
      const int nxt = st + 1 == ST ? 0 : st + 1;
      past_end(kt + ST);
      kstep(C1{}, nxt, C0{}, J1{}, st, kt + ST);
      landed(C0{});
      end_range(kt + 1);
      last = st;
      st = nxt;
    }
  }
  // results of the last asm MFMAs; the zero-filling loads past the last k-tile
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_waitcnt vmcnt(0)" ::: "memory");
  GR_BARRIER();
#undef GR_BARRIER
  if constexpr (RANGES) {
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) acc[i][j] += sum[i][j];
  }

  // ---- epilogue: 16 tokens at a time through the wave's own corner of LDS (rows padded by 16 bytes: conflict-free both
  // ways), so that a store instruction writes whole row segments.
  if (GATED && !EARLY) request();
  const uint32_t out0 = lds0 + wave * OUT_BYTES, wr = out0 + fr * PITCH + 16 * fg;
  uint32_t rd[NS];
  int row_s[NS], n_s[NS], coff[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const int idx = lane + 64 * s, row = idx / PPR, pc = idx % PPR;
    rd[s] = out0 + row * PITCH + 16 * pc;
    row_s[s] = 16 * TM * wm + row;
    n_s[s] = n0 + wn * 16 * TN + 8 * pc;
    coff[s] = n_s[s] < N ? (row_s[s] * (int)ldc + n_s[s]) * 2 : (int)kOut;
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
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    gr_tie(o);
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
