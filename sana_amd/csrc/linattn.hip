// ReLU linear attention for gfx950: phase 1 (state = [V|1]^T relu(K) per head),
// split reduction + chunk prefix scan, phase 2 (apply to relu(Q), divide).
//
// Data layout: q, k, v and out are token-major [B][N][h*32] views (channel
// stride 1).  The state is fp32 [B][h][n_chunks][33][32]; row 32 holds
// sum_n relu(k_n).
//
// 16-bit io (bf16 / f16)
//   phase 1  one workgroup = (batch, pair of heads, chunk, token split); its four
//            waves take interleaved 32-token tiles.  A tile is loaded with
//            16-byte coalesced loads, written to wave-private LDS and read back
//            transposed (token-contiguous per channel) as MFMA 32x32x16
//            operands: S += V^T K; the ones-row (ksum) is a packed dot2 against (1, 1)
//            on the K operand registers.  Waves are summed in LDS.
//   phase 2  one wave = (pair of heads, token range); the fp32 state is split
//            into three bf16 terms (hi + mid + lo = all 24 mantissa bits) and
//            applied with MFMA 16x16x32; rows 32..47 of the A operand all carry
//            ksum so every lane gets its token's denominator in-lane.
// fp32 io uses MFMA 32x32x2 f32 directly from global memory.
#include <atomic>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "linattn_common.h"

// tuning knobs of the bf16 apply kernel: tokens per workgroup, 16-token steps in flight per wave
#ifndef SANA_LA_APPLY_MINWG
#define SANA_LA_APPLY_MINWG 256  // halve the tokens of a workgroup (to no less than 32) until the launch has this many
#endif
#ifndef SANA_LA_APPLY_TOKENS
#define SANA_LA_APPLY_TOKENS 128
#endif
#ifndef SANA_LA_NT_STORE
#define SANA_LA_NT_STORE 0
#endif
#ifndef SANA_LA_APPLY_U
#define SANA_LA_APPLY_U 4
#endif

namespace sana {
namespace {

constexpr int D = 32;
constexpr int STATE_ELEMS = (D + 1) * D;  // 1056
constexpr int TILE = 32;                  // tokens per phase-1 tile

template <int OFF>
__device__ __forceinline__ u32x2_t lds_read_tr16(uint32_t addr) {  // 4 tokens x 16 channels -> this lane's channel, 4 tokens
  u32x2_t v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}

// ----------------------------------------------------------------------------
// phase 1, 16-bit io
// grid: x = nsplit, y = n_chunks, z = B * pairs;  block 256
// dst: when nsplit == 1 the final state, else partial[(bh*n_chunks + c)*nsplit + split][1056]
// At a few thousand tokens bound by latency: a split is one or two tiles a wave.  Loads without a branch and a 64-bit product each, and 16
// transposing reads a tile where 64 two-byte ones were packed in pairs (same bits).  us with the reduction, before / now: 1600 tokens x 20 heads
// 7.8 / 7.1, 2048 x 36 8.7 / 8.1, 4096 x 70 14.4 / 13.7, with the norm 16.2 / 15.5, with the rotation 15.8 / 15.3, 16384 x 70 35.7 / 34.9.
// ----------------------------------------------------------------------------
// PRE: on-load transforms as compile-time bits (1 = q/k RMSNorm, 2 = rotary embedding, 4 = the rotation comes before
// the ReLU and ksum is taken from the rotated values: QkPre::rope_first)
template <typename T, int PRE>
__global__ __launch_bounds__(256) void linattn_state16_kernel(
    const uint16_t* __restrict__ K, const uint16_t* __restrict__ V, float* __restrict__ dst,
    const int32_t* __restrict__ chunk_starts, int N, int h, int n_chunks, int nsplit, int split_tokens,
    int64_t stride_b, int64_t stride_n, const QkPre pre) {
  // staging: per wave K tile [32 tok][64 ch] + V tile, 16-bit, rows of ROW bytes -> 10 KB per wave (four workgroups per CU).
  // reduction: per wave 2 heads x 1056 fp32 -> 8448 B per wave.  The two uses
  // never overlap in time, so they share one buffer.
  constexpr int ROW = 160;  // 40 banks: the eight rows of a transposing read meet every bank twice
  static_assert(2 * TILE * ROW >= 2 * STATE_ELEMS * 4, "the reduction fits in the stages");
  __shared__ __attribute__((aligned(16))) unsigned char smem[4 * 2 * TILE * ROW];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int pairs = (h + 1) >> 1;
  const int b = blockIdx.z / pairs, p = blockIdx.z % pairs;
  const int c = blockIdx.y, split = blockIdx.x;
  const int C = h * D;
  const ChunkRange cr = chunk_range(chunk_starts, c, N);
  const int t0 = cr.begin + split * split_tokens;
  const int t1 = min(cr.end, t0 + split_tokens);

  unsigned char* lds_k = smem + wave * (2 * TILE * ROW);
  unsigned char* lds_v = lds_k + TILE * ROW;

  // load mapping: lane -> token (lane/8 + 8*i), 16-byte channel chunk lane%8
  const int ld_tok = lane >> 3;
  const int ld_ch = p * 64 + (lane & 7) * 8;
  const bool ch_ok = ld_ch < C;
  const uint16_t* kbase = K + (int64_t)b * stride_b + ld_ch;
  const uint16_t* vbase = V + (int64_t)b * stride_b + ld_ch;

  f32x16_t accS[2];
  float accK[2] = {0.f, 0.f};  // sum over this lane's tokens of relu(K)[tok][j]
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    accS[0][i] = 0.f;
    accS[1][i] = 0.f;
  }
  const u32x4_t zero4 = {0u, 0u, 0u, 0u};

  constexpr bool has_norm = (PRE & 1) != 0, has_rope = (PRE & 2) != 0, rope_first = (PRE & 4) != 0;
  u32x4_t kreg[4], vreg[4];
  // PRE: per-token 1/rms and this lane's four (cos, sin) pairs travel with the tile; the norm weight
  // of the lane's 8 channels is loop-invariant; ksum is accumulated here, per lane and channel,
  // from the unrotated values (the MFMA operands in LDS are rotated).
  float rin[has_norm ? 4 : 1];
  f32x4_t cs[has_rope ? 4 : 1][2];
  u32x4_t kw = zero4;
  float ks8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (has_norm && ch_ok) kw = *reinterpret_cast<const u32x4_t*>(pre.weight + ld_ch);
  // Loads without a branch each: tokens from t1 on and channels past C lie outside the resources, zeros.
  const bool near = (int64_t)(t1 - t0 + TILE) * stride_n < (1 << 29);  // 32-bit offsets
  constexpr uint32_t kOut = 0x80000000u;
  auto issue_loads = [&](int tile) {
    if (near) {
      const int span = ((t1 - t0 - 1) * (int)stride_n + min(64, C - p * 64)) * 2;
      const int64_t at = (int64_t)b * stride_b + (int64_t)t0 * stride_n + p * 64;
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(K + at), 0, span, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(V + at), 0, span, 0x00020000);
      const __amdgpu_buffer_rsrc_t rn = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(has_norm ? pre.rinv + (int64_t)b * N + t0 : nullptr), 0, has_norm ? (t1 - t0) * 4 : 0, 0x00020000);
      const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<float*>(has_rope ? pre.rope + (int64_t)t0 * 32 : nullptr), 0, has_rope ? (t1 - t0) * 128 : 0, 0x00020000);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tok = tile - t0 + ld_tok + 8 * i, o = ch_ok ? (tok * (int)stride_n + (lane & 7) * 8) * 2 : (int)kOut;
        kreg[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, o, 0, 0));
        vreg[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, o, 0, 0));
        if (has_norm) rin[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rn, tok * 4, 0, 0));
        if (has_rope) {
          const int ro = tok * 128 + (lane & 3) * 32;
          cs[i][0] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rr, ro, 0, 0));
          cs[i][1] = __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rr, ro + 16, 0, 0));
        }
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int tok = tile + ld_tok + 8 * i;
      if (ch_ok && tok < t1) {
        kreg[i] = *reinterpret_cast<const u32x4_t*>(kbase + (int64_t)tok * stride_n);
        vreg[i] = *reinterpret_cast<const u32x4_t*>(vbase + (int64_t)tok * stride_n);
        if (has_norm) rin[i] = pre.rinv[(int64_t)b * N + tok];
        if (has_rope) {
          const float* rp = pre.rope + ((int64_t)tok * 16 + (lane & 3) * 4) * 2;
          cs[i][0] = *reinterpret_cast<const f32x4_t*>(rp);
          cs[i][1] = *reinterpret_cast<const f32x4_t*>(rp + 4);
        }
      } else {
        kreg[i] = zero4;
        vreg[i] = zero4;
        if (has_norm) rin[i] = 0.f;
        if (has_rope) {
          cs[i][0] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          cs[i][1] = cs[i][0];
        }
      }
    }
  };

  int tile = t0 + wave * TILE;
  if (tile < t1) issue_loads(tile);
  // operand read mapping: lane -> channel j = lane%32 (of head hh), k-group g = lane/32;
  // element r of k-step s is token 16*s + 2*r + g of the tile (any bijection works as
  // long as both operands use the same one: the MFMA contracts over tokens).
  const int j = lane & 31, g = lane >> 5;
  // A transposing read hands the 16 lanes of a group four rows, row i addressed by lanes 4 i .. 4 i + 3: two tokens apart here.
  const uint32_t k_at = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)lds_k +
                        (2 * ((lane >> 2) & 3) + g) * ROW + ((lane >> 4) & 1) * 32 + (lane & 3) * 8, v_at = k_at + TILE * ROW;
  for (; tile < t1; tile += 4 * TILE) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      u32x4_t kk = kreg[i];
      if (PRE) {
        if (has_norm) kk = rms_scale8(kk, rin[i], kw);
        if (rope_first) kk = rope8(kk, cs[i][0], cs[i][1]);
        kk = relu_pk16(kk);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          ks8[2 * e] += bf16_lo(kk[e]);
          ks8[2 * e + 1] += bf16_hi(kk[e]);
        }
        if (has_rope && !rope_first) kk = rope8(kk, cs[i][0], cs[i][1]);
      } else {
        kk = relu_pk16(kk);
      }
      *reinterpret_cast<u32x4_t*>(lds_k + (ld_tok + 8 * i) * ROW + (lane & 7) * 16) = kk;
      *reinterpret_cast<u32x4_t*>(lds_v + (ld_tok + 8 * i) * ROW + (lane & 7) * 16) = vreg[i];
    }
    if (tile + 4 * TILE < t1) issue_loads(tile + 4 * TILE);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private LDS: in-order, no barrier needed
    u32x2_t kf[2][2][2], vf[2][2][2];  // [head][k-step][elements 4 i ..]
    auto read = [&](auto hh_c) {
      constexpr int hh = decltype(hh_c)::value;
      kf[hh][0][0] = lds_read_tr16<64 * hh>(k_at), kf[hh][0][1] = lds_read_tr16<64 * hh + 8 * ROW>(k_at);
      vf[hh][0][0] = lds_read_tr16<64 * hh>(v_at), vf[hh][0][1] = lds_read_tr16<64 * hh + 8 * ROW>(v_at);
      kf[hh][1][0] = lds_read_tr16<64 * hh + 16 * ROW>(k_at), kf[hh][1][1] = lds_read_tr16<64 * hh + 24 * ROW>(k_at);
      vf[hh][1][0] = lds_read_tr16<64 * hh + 16 * ROW>(v_at), vf[hh][1][1] = lds_read_tr16<64 * hh + 24 * ROW>(v_at);
    };
    read(std::integral_constant<int, 0>{});
    if (!has_rope) read(std::integral_constant<int, 1>{});  // (with the rotation: later, for the registers of a third workgroup)
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      if (hh == 1 && has_rope) read(std::integral_constant<int, 1>{});
      if (hh == 0 && has_rope)
        asm volatile("s_waitcnt lgkmcnt(0)"
                     : "+v"(kf[0][0][0]), "+v"(kf[0][0][1]), "+v"(kf[0][1][0]), "+v"(kf[0][1][1]), "+v"(vf[0][0][0]), "+v"(vf[0][0][1]),
                       "+v"(vf[0][1][0]), "+v"(vf[0][1][1])::"memory");
      else if (hh == 0)  // (the reads come in order: the second head's eight are behind)
        asm volatile("s_waitcnt lgkmcnt(8)"
                     : "+v"(kf[0][0][0]), "+v"(kf[0][0][1]), "+v"(kf[0][1][0]), "+v"(kf[0][1][1]), "+v"(vf[0][0][0]), "+v"(vf[0][0][1]),
                       "+v"(vf[0][1][0]), "+v"(vf[0][1][1])::"memory");
      else
        asm volatile("s_waitcnt lgkmcnt(0)"  // (and before the next tile overwrites)
                     : "+v"(kf[1][0][0]), "+v"(kf[1][0][1]), "+v"(kf[1][1][0]), "+v"(kf[1][1][1]), "+v"(vf[1][0][0]), "+v"(vf[1][0][1]),
                       "+v"(vf[1][1][0]), "+v"(vf[1][1][1])::"memory");
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4_t fk = {kf[hh][s][0].x, kf[hh][s][0].y, kf[hh][s][1].x, kf[hh][s][1].y};
        accS[hh] = mfma_32x32x16<T>(u32x4_t{vf[hh][s][0].x, vf[hh][s][0].y, vf[hh][s][1].x, vf[hh][s][1].y}, fk,
                                    accS[hh]);  // S[i][j] += sum_tok V[tok][i] K[tok][j]
        if (!PRE) {
#pragma unroll
          for (int r2 = 0; r2 < 4; ++r2) accK[hh] = add_pk16<T>(fk[r2], accK[hh]);  // the "1" row of [V|1]
        }
      }
    }
  }

  // cross-wave reduction in LDS.  D layout of 32x32 MFMA: lane -> column j = lane%32,
  // register r -> row 8*(r/4) + 4*(lane/32) + r%4.
  __syncthreads();
  float* red = reinterpret_cast<float*>(smem) + wave * (2 * STATE_ELEMS);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int row = 8 * (r >> 2) + 4 * g + (r & 3);
      red[hh * STATE_ELEMS + row * D + j] = accS[hh][r];
    }
    if (!PRE) {
      const float ks = accK[hh] + __shfl_xor(accK[hh], 32, 64);  // the two token halves of channel j
      if (g == 0) red[hh * STATE_ELEMS + D * D + j] = ks;
    }
  }
  if (PRE) {  // lanes with the same channel chunk (lane % 8) hold different tokens: fold them
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float x = ks8[e];
      x += __shfl_xor(x, 8, 64);
      x += __shfl_xor(x, 16, 64);
      x += __shfl_xor(x, 32, 64);
      if (lane < 8) red[(lane >> 2) * STATE_ELEMS + D * D + (lane & 3) * 8 + e] = x;
    }
  }
  __syncthreads();
  const float* all = reinterpret_cast<const float*>(smem);
  for (int e = tid; e < 2 * STATE_ELEMS; e += 256) {
    const int hh = e / STATE_ELEMS, idx = e - hh * STATE_ELEMS;
    const int head = 2 * p + hh;
    if (head >= h) continue;
    const float sum = ((all[e] + all[2 * STATE_ELEMS + e]) + all[4 * STATE_ELEMS + e]) + all[6 * STATE_ELEMS + e];
    const int64_t slot = ((int64_t)(b * h + head) * n_chunks + c) * nsplit + split;
    dst[slot * STATE_ELEMS + idx] = sum;
  }
}

// ----------------------------------------------------------------------------
// phase 1, fp32 io: MFMA 32x32x2 f32 straight from global memory.
// grid: x = nsplit, y = n_chunks, z = B * ceil(h/4); block 256, wave = one head.
// Bound by load latency: 64 tokens in flight without a branch around a load (it was 16 behind branches); the key sum is
// adds, not a second MFMA chain.  Tokens x heads, us with the reduction: 1024 x 36 12.1 -> 7.6, 16384 x 70 136 -> 82.
// ----------------------------------------------------------------------------
// LINEAR: one chunk, the grid in one dimension of nsplit * B * ceil(h/4), an eighth of it in a row on each XCD: the phase 2 that
// reads the partial states (linattn_apply32_partials_kernel) runs its heads there too.
__device__ __forceinline__ int xcd_eighths(int id, int total) {  // workgroup -> its place in the order whose eighths are an XCD's
  const int xcd = id & 7, base = total >> 3, rem = total & 7;
  return xcd * base + min(xcd, rem) + (id >> 3);
}
// Short splits are one round trip behind what comes in front of their loads: with a 64-bit product and a clamp each, 64 loads went
// out over more than a microsecond.  us, whole calls, before (the phase 2 on partial states with its divisions first) / now, inputs from
// HBM: 1024 x 36 17.7 / 15.1 (from the caches 14.9 / 13.4), 400 x 70 14.0 / 12.5, 2 x 1024 x 36 22.4 / 19.8, 4 x 1737 x 36 46.4 / 45.7, 3 x 3000 x 36 68 / 58,
// 16384 x 36 99 / 89, 4 x 5000 x 70 224 / 207.
// FAR: rows too far apart for 32-bit offsets, an instance of its own: both ways in one kernel take the registers of a fourth workgroup per compute
// unit, of which plan_state's 1000 or so of a few thousand tokens need all (4 x 1500 x 36 45.5, so 42.5).
template <bool LINEAR, bool FAR>
__global__ __launch_bounds__(256) void linattn_state32_kernel(
    const float* __restrict__ K, const float* __restrict__ V, float* __restrict__ dst,
    const int32_t* __restrict__ chunk_starts, int N, int h, int n_chunks, int nsplit, int split_tokens,
    int64_t stride_b, int64_t stride_n) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int groups = (h + 3) >> 2;
  const int at = LINEAR ? xcd_eighths(blockIdx.x, gridDim.x) : 0;
  const int z = LINEAR ? at / nsplit : blockIdx.z, split = LINEAR ? at % nsplit : blockIdx.x;
  const int b = z / groups, head = (z % groups) * 4 + wave;
  if (head >= h) return;  // no barriers below
  const int c = LINEAR ? 0 : blockIdx.y;
  const ChunkRange cr = chunk_range(chunk_starts, c, N);
  const int t0 = cr.begin + split * split_tokens;
  const int t1 = min(cr.end, t0 + split_tokens);
  const int j = lane & 31, g = lane >> 5;
  const float* kp = K + (int64_t)b * stride_b + (int64_t)t0 * stride_n + head * D;
  const float* vp = V + (int64_t)b * stride_b + (int64_t)t0 * stride_n + head * D;
  f32x16_t accS;
  float accK = 0.f;  // the "1" row of [V|1]: this lane's half of the tokens
#pragma unroll
  for (int i = 0; i < 16; ++i) accS[i] = 0.f;
  const int n = t1 - t0;
  auto add = [&](auto& kk, auto& vv, auto u_c) {
#pragma unroll
    for (int u = 0; u < decltype(u_c)::value; ++u) {
      kk[u] = fmaxf(kk[u], 0.f);
      accS = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[u], kk[u], accS, 0, 0, 0);
      accK += kk[u];
    }
  };
  using U32 = std::integral_constant<int, 32>;  // 64 tokens in flight per wave: a small input is one round trip
  if constexpr (!FAR) {  // 32-bit offsets; rows past t1 lie outside the resources: zeros
    const int ld = (int)stride_n * 4, span = n > 0 ? (n - 1) * ld + 4 * D : 0;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(kp), 0, span, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(vp), 0, span, 0x00020000);
    auto pass = [&](int t, auto u_c) {
      constexpr int U = decltype(u_c)::value;
      float kk[U], vv[U];
      int at = (t + g) * ld + 4 * j;
#pragma unroll
      for (int u = 0; u < U; ++u, at += 2 * ld) {
        kk[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rk, at, 0, 0));
        vv[u] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, at, 0, 0));
      }
      add(kk, vv, u_c);
    };
    int t = 0;
#pragma unroll 1
    for (; t + 64 <= n; t += 64) pass(t, U32{});
    // (a load outside the resource takes its time all the same)
    if (n - t > 32) pass(t, U32{});
    else if (n - t > 16) pass(t, std::integral_constant<int, 16>{});
    else if (n - t > 0) pass(t, std::integral_constant<int, 8>{});
  } else {
    constexpr int U = U32::value;
    for (int t = 0; t < n; t += 2 * U) {
      float kk[U], vv[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int64_t at = (int64_t)min(t + 2 * u + g, n - 1) * stride_n + j;  // (no branch around a load)
        kk[u] = kp[at], vv[u] = vp[at];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool ok = t + 2 * u + g < n;
        kk[u] = ok ? kk[u] : 0.f, vv[u] = ok ? vv[u] : 0.f;
      }
      add(kk, vv, U32{});
    }
  }
  const int64_t slot = ((int64_t)(b * h + head) * n_chunks + c) * nsplit + split;
  float* o = dst + slot * STATE_ELEMS;
#pragma unroll
  for (int r = 0; r < 16; ++r) o[(8 * (r >> 2) + 4 * g + (r & 3)) * D + j] = accS[r];
  accK += __shfl_xor(accK, 32, 64);
  if (g == 0) o[D * D + j] = accK;
}

// ----------------------------------------------------------------------------
// split reduction (+ inclusive prefix over chunks when causal).
// One thread per (b*h, element); fixed summation order.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void linattn_reduce_scan_kernel(const float* __restrict__ partial,
                                                                  float* __restrict__ state, int BH,
                                                                  int n_chunks, int nsplit, int causal) {
  const int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (gid >= (int64_t)BH * STATE_ELEMS) return;
  const int64_t bh = gid / STATE_ELEMS;
  const int e = (int)(gid - bh * STATE_ELEMS);
  float run = 0.f;
  for (int c = 0; c < n_chunks; ++c) {
    const float* p0 = partial + ((bh * n_chunks + c) * nsplit) * STATE_ELEMS + e;
    // batches of sixteen independent loads (all in flight together), added in split order
    float s = 0.f;
    for (int sp0 = 0; sp0 < nsplit; sp0 += 16) {
      float v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = (sp0 + u < nsplit) ? p0[(int64_t)(sp0 + u) * STATE_ELEMS] : 0.f;
#pragma unroll
      for (int u = 0; u < 16; ++u) s += v[u];
    }
    if (causal) {
      run += s;
      s = run;
    }
    state[(bh * n_chunks + c) * STATE_ELEMS + e] = s;
  }
}

// ----------------------------------------------------------------------------
// phase 2, bf16 and f16 io.  grid: x = token ranges per chunk, y = n_chunks,
// z = B * ceil(pairs/4); block 256; wave = pair of heads.
// ----------------------------------------------------------------------------
struct SplitState {     // A operands of one head: 3 row blocks x 3 bf16 terms
  u32x4_t a[3][3];
};

__device__ __forceinline__ void split3(const float x[8], u32x4_t out[3]) {
  float r1[8], r2[8];
  uint32_t hi[8], mid[8], lo[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    hi[e] = f32_to_bf16_bits(x[e]);
    r1[e] = x[e] - bf16_bits_to_f32(hi[e]);
    mid[e] = f32_to_bf16_bits(r1[e]);
    r2[e] = r1[e] - bf16_bits_to_f32(mid[e]);
    lo[e] = f32_to_bf16_bits(r2[e]);
  }
#pragma unroll
  for (int e2 = 0; e2 < 4; ++e2) {
    out[0][e2] = hi[2 * e2] | (hi[2 * e2 + 1] << 16);
    out[1][e2] = mid[2 * e2] | (mid[2 * e2 + 1] << 16);
    out[2][e2] = lo[2 * e2] | (lo[2 * e2 + 1] << 16);
  }
}

// f16 queries go to the bf16 MFMA as the exact sum of two bf16 values (11 significant bits = 8 + 3): the state keeps its
// range and its 24 bits, which f16 terms would not.
__device__ __forceinline__ void f16_to_2bf16(u32x4_t q, u32x4_t& hi, u32x4_t& lo) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float a = lo16<F16>(q[e]), b = hi16<F16>(q[e]);
    hi[e] = pack_bf16(a, b);
    lo[e] = pack_bf16(a - bf16_lo(hi[e]), b - bf16_hi(hi[e]));
  }
}

// num / den for many numerators, rounded as the division is: the reciprocal with one Newton step, the product corrected by its
// residual (an exact fma), and the division's own handling of zeros, infinities and NaN.  f16 outputs need it: where the
// quotient lies halfway between two f16 values the error of num * rcp(den) decides the rounding.  Denominators beyond 2^126,
// whose reciprocal is not a normal number, do not occur (the operands are f16).  16384 x 70, us: num * rcp(den) 36, the
// compiler's division 48, this 39.
struct Quotient {
  float den, inv;
  __device__ __forceinline__ explicit Quotient(float d) : den(d) {
    inv = __builtin_amdgcn_rcpf(d);
    inv = fmaf(fmaf(-d, inv, 1.0f), inv, inv);
  }
  __device__ __forceinline__ float operator()(float num) const {
    const float q = num * inv;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-den, q, num), inv, q), den, num);
  }
};

// T = F16 replaces MFMAs in fp32 (32x32x2) and 2-byte loads and stores: tokens x heads, us: 2048 x 36
// 16.5 -> 7.2, 16384 x 70 125 -> 36.
// The state, then the first queries, are requested before anything is computed, later ones a pass ahead; the wave is uniform.  bf16, us,
// before / so, inputs from HBM: 16384 x 70 40.3 / 35.5, 16 x 1024 x 70 38.5 / 34.5, 4096 x 70 14.6 / 13.9, 2048 x 36 6.3 / 5.8, 4 x 1024 x 36 9.2 / 9.2.
template <typename T, bool OUT_F32, int PRE>
__global__ __launch_bounds__(256) void linattn_apply16_kernel(
    const uint16_t* __restrict__ Q, const float* __restrict__ state, void* __restrict__ out,
    const int32_t* __restrict__ chunk_starts, int N, int h, int n_chunks, int wg_tokens,
    int64_t q_stride_b, int64_t q_stride_n, int64_t o_stride_b, int64_t o_stride_n, float eps,
    const QkPre pre, int xranges, int ngroups) {
  asm volatile("" ::"s"(Q), "s"(state), "s"(chunk_starts), "s"(N), "s"(h), "s"(n_chunks), "s"(wg_tokens), "s"(q_stride_b), "s"(q_stride_n),
               "s"(xranges), "s"(ngroups));  // (the arguments in one wait)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int pairs = (h + 1) >> 1;
  const int pgroups = (pairs + 3) >> 2;
  // 3-D grid (token range, chunk, batch x head group), or -- with many (chunk, batch, head group)
  // combinations -- a 1-D grid dealt so that all token ranges of one combination run on the same XCD
  // (workgroup ids go round-robin to the 8 XCDs): their common state is then fetched into one L2 only.
  int bx = blockIdx.x, by = blockIdx.y, bz = blockIdx.z;
  if (ngroups > 0) {
    const uint32_t xcd = blockIdx.x & 7, idx = blockIdx.x >> 3, grp = xcd + 8 * (idx / (uint32_t)xranges);
    if (grp >= (uint32_t)ngroups) return;  // no barriers below
    bx = (int)(idx % (uint32_t)xranges), by = (int)(grp % (uint32_t)n_chunks), bz = (int)(grp / (uint32_t)n_chunks);
  }
  const int b = (int)((uint32_t)bz / (uint32_t)pgroups), p = (bz - b * pgroups) * 4 + wave;
  if (p >= pairs) return;  // no barriers below
  const int c = by;
  const ChunkRange cr = chunk_range(chunk_starts, c, N);
  const int t0 = cr.begin + bx * wg_tokens;
  const int t1 = min(cr.end, t0 + wg_tokens);
  if (t0 >= t1) return;
  const int n = lane & 15, g = lane >> 4;
  const int nheads = (2 * p + 1 < h) ? 2 : 1;

  // Global accesses are whole 128-byte lines: lane l fetches 16-byte chunk l%8 of token l/8 (both heads
  // of the pair), two instructions per 16-token step, and the step goes through wave-private LDS to
  // reach the MFMA layout (lane = token n, channel group g); results return the same way, so a store
  // instruction writes eight full lines.  (Fetching straight in MFMA layout touches every line twice
  // with 64-byte pieces and is bound by the L1 tag rate: 4.2 TB/s read side against 5.8 here.)
  // LDS slot of (token n of the step, chunk c): 16 * (8n + (c ^ (n/2) % 8)): conflict-free both ways.
  constexpr int U = PRE ? SANA_LA_APPLY_U / 2 : SANA_LA_APPLY_U;  // 16-token steps in flight
  __shared__ __attribute__((aligned(16))) unsigned char stage_all[4 * (SANA_LA_APPLY_U + 1) * 2048];
  unsigned char* stage = stage_all + wave * ((SANA_LA_APPLY_U + 1) * 2048);
  const int ld_tok = lane >> 3, ld_chunk = lane & 7;
  const bool ld_ok = nheads == 2 || ld_chunk < 4;   // the second head of the last pair may not exist
  const uint16_t* qrow = Q + (int64_t)b * q_stride_b + p * 64 + 8 * (ld_ok ? ld_chunk : ld_chunk - 4);
  int slot_w[2], slot_r[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int tl = 8 * j + ld_tok;
    slot_w[j] = 16 * (8 * tl + (ld_chunk ^ ((tl >> 1) & 7)));
  }
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) slot_r[hh] = 16 * (8 * n + ((4 * hh + g) ^ ((n >> 1) & 7)));
  // The queries of a pass are requested a pass ahead, the first ones behind the state's loads and in front of its split: it was one memory
  // latency after the other.  Past the range its last token once more (not stored), for the head that does not exist the one that does: no
  // branch around a load.
  u32x4_t raw[U][2];
  auto fetch = [&](int t) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j)
        raw[u][j] = *reinterpret_cast<const u32x4_t*>(qrow + (int64_t)min(t + 16 * u + 8 * j + ld_tok, t1 - 1) * q_stride_n);
  };

  // A operands.  MFMA 16x16x32: A lane -> row lane%16, k = 8*(lane/16)+e.  Output
  // lane (token n, g') register s of row block rb is row 4*g'+s; we place channel
  // 8*(r/4) + 4*rb + r%4 in row r so that a lane ends up with 8 contiguous channels.
  SplitState st[2];
  f32x4_t x[2][3][2];
#pragma unroll
  for (int hh = 0; hh < 2; ++hh) {
    const int head = min(2 * p + hh, h - 1);
    const float* sp = state + ((int64_t)(b * h + head) * n_chunks + c) * STATE_ELEMS;
#pragma unroll
    for (int rb = 0; rb < 3; ++rb) {
      const int row = (rb < 2) ? (8 * (n >> 2) + 4 * rb + (n & 3)) : D;
#pragma unroll
      for (int e = 0; e < 2; ++e) x[hh][rb][e] = *reinterpret_cast<const f32x4_t*>(sp + row * D + 8 * g + 4 * e);
    }
  }
  fetch(t0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int hh = 0; hh < 2; ++hh)
#pragma unroll
    for (int rb = 0; rb < 3; ++rb) {
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = x[hh][rb][e >> 2][e & 3];
      split3(v, st[hh].a[rb]);
    }

  constexpr bool has_norm = (PRE & 1) != 0, has_rope = (PRE & 2) != 0, rope_first = (PRE & 4) != 0;
  u32x4_t qw[2] = {{0u, 0u, 0u, 0u}, {0u, 0u, 0u, 0u}};
  if (has_norm) {
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
      if (hh < nheads) qw[hh] = *reinterpret_cast<const u32x4_t*>(pre.weight + p * 64 + hh * D + 8 * g);
  }
  for (int t = t0; t < t1; t += 16 * U) {
    float rin[has_norm ? U : 1];
    f32x4_t cs[has_rope ? U : 1][2];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int tok = t + 16 * u + n;
      if (has_norm) rin[u] = tok < t1 ? pre.rinv[(int64_t)b * N + tok] : 0.f;
      if (has_rope) {
        const float* rp = pre.rope + ((int64_t)min(tok, t1 - 1) * 16 + g * 4) * 2;
        cs[u][0] = *reinterpret_cast<const f32x4_t*>(rp);
        cs[u][1] = *reinterpret_cast<const f32x4_t*>(rp + 4);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) *reinterpret_cast<u32x4_t*>(stage + u * 2048 + slot_w[j]) = raw[u][j];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private LDS: in-order, no barrier needed
    if (t + 16 * U < t1) fetch(t + 16 * U);  // uniform
    unsigned char* ostage = stage + SANA_LA_APPLY_U * 2048;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (t + 16 * u >= t1) break;  // uniform
      const int tok = t + 16 * u + n;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        u32x4_t qd = *reinterpret_cast<const u32x4_t*>(stage + u * 2048 + slot_r[hh]);
        if (has_norm) qd = rms_scale8(qd, rin[u], qw[hh]);
        if (rope_first) qd = rope8(qd, cs[u][0], cs[u][1]);              // rotated first: both operands
        qd = relu_pk16(qd);                                              // denominator operand
        const u32x4_t qb = (has_rope && !rope_first) ? rope8(qd, cs[u][0], cs[u][1]) : qd;  // numerator operand
        u32x4_t q_hi, q_lo;
        if constexpr (is_f16<T>) f16_to_2bf16(qd, q_hi, q_lo);
        f32x4_t acc[3];
#pragma unroll
        for (int rb = 0; rb < 3; ++rb) {
          [[maybe_unused]] const u32x4_t bop = rb < 2 ? qb : qd;
          f32x4_t a = {0.f, 0.f, 0.f, 0.f};
          if constexpr (is_f16<T>) {  // (no PRE: bop is qd)
            a = mfma_16x16x32_bf16(st[hh].a[rb][2], q_lo, a);  // smallest terms first
            a = mfma_16x16x32_bf16(st[hh].a[rb][2], q_hi, a);
            a = mfma_16x16x32_bf16(st[hh].a[rb][1], q_lo, a);
            a = mfma_16x16x32_bf16(st[hh].a[rb][1], q_hi, a);
            a = mfma_16x16x32_bf16(st[hh].a[rb][0], q_lo, a);
            a = mfma_16x16x32_bf16(st[hh].a[rb][0], q_hi, a);
          } else {
            a = mfma_16x16x32_bf16(st[hh].a[rb][2], bop, a);  // smallest term first
            a = mfma_16x16x32_bf16(st[hh].a[rb][1], bop, a);
            a = mfma_16x16x32_bf16(st[hh].a[rb][0], bop, a);
          }
          acc[rb] = a;
        }
        const float den = acc[2][0] + eps;
        if (OUT_F32) {
          if (tok < t1 && hh < nheads) {
            const int64_t o_off = (int64_t)b * o_stride_b + (int64_t)tok * o_stride_n + p * 64 + hh * D + 8 * g;
            f32x4_t o0, o1;
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              o0[s] = acc[0][s] / den;
              o1[s] = acc[1][s] / den;
            }
            float* op = reinterpret_cast<float*>(out) + o_off;
            store_stream<SANA_LA_NT_STORE != 0>(o0, reinterpret_cast<f32x4_t*>(op));
            store_stream<SANA_LA_NT_STORE != 0>(o1, reinterpret_cast<f32x4_t*>(op + 4));
          }
        } else {
          u32x4_t o;
          if constexpr (is_f16<T>) {
            const Quotient by(den);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = pk16<T>(by(acc[e >> 1][2 * (e & 1)]), by(acc[e >> 1][2 * (e & 1) + 1]));
          } else {
            const float inv = __builtin_amdgcn_rcpf(den);
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = pk16<T>(acc[e >> 1][2 * (e & 1)] * inv, acc[e >> 1][2 * (e & 1) + 1] * inv);
          }
          *reinterpret_cast<u32x4_t*>(ostage + slot_r[hh]) = o;
        }
      }
      if (!OUT_F32) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int tok_s = t + 16 * u + 8 * j + ld_tok;
          const u32x4_t o = *reinterpret_cast<const u32x4_t*>(ostage + slot_w[j]);
          if (tok_s < t1 && ld_ok)
            store_stream<SANA_LA_NT_STORE != 0>(o, reinterpret_cast<u32x4_t*>(reinterpret_cast<uint16_t*>(out) + (int64_t)b * o_stride_b +
                                                       (int64_t)tok_s * o_stride_n + p * 64 + 8 * ld_chunk));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the reads are done before the next step overwrites
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// ----------------------------------------------------------------------------
// phase 2, fp32 io: MFMA 32x32x2 f32.  grid as above but wave = one head,
// z = B * ceil(h/4).  A lane -> state row lane%32, contraction index 16*(lane/32)+s;
// B lane -> token lane%32, same contraction index.  The denominator is 16 fused multiply-adds per lane and one exchange
// with the lane that holds the token's other half.  Tokens x heads, us, against a second
// MFMA chain for the denominator and scalar loads: 1024 x 36 9.2 -> 5.4, 16384 x 70 167 -> 88.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void linattn_apply32_kernel(
    const float* __restrict__ Q, const float* __restrict__ state, float* __restrict__ out,
    const int32_t* __restrict__ chunk_starts, int N, int h, int n_chunks, int wg_tokens,
    int64_t q_stride_b, int64_t q_stride_n, int64_t o_stride_b, int64_t o_stride_n, float eps) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int groups = (h + 3) >> 2;
  const int b = blockIdx.z / groups, head = (blockIdx.z % groups) * 4 + wave;
  if (head >= h) return;
  const int c = blockIdx.y;
  const ChunkRange cr = chunk_range(chunk_starts, c, N);
  const int t0 = cr.begin + blockIdx.x * wg_tokens;
  const int t1 = min(cr.end, t0 + wg_tokens);
  if (t0 >= t1) return;
  const int n = lane & 31, g = lane >> 5;
  const float* sp = state + ((int64_t)(b * h + head) * n_chunks + c) * STATE_ELEMS;
  f32x4_t qn[4];  // (rows start at multiples of 16 bytes)
  auto load_q = [&](int t) {
    const float* qp = Q + (int64_t)b * q_stride_b + (int64_t)min(t + n, t1 - 1) * q_stride_n + head * D + 16 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) qn[i] = *reinterpret_cast<const f32x4_t*>(qp + 4 * i);
  };
  load_q(t0);
  f32x4_t a_num[4], a_den[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a_num[i] = *reinterpret_cast<const f32x4_t*>(sp + n * D + 16 * g + 4 * i);
    a_den[i] = *reinterpret_cast<const f32x4_t*>(sp + D * D + 16 * g + 4 * i);
  }
  for (int t = t0; t < t1; t += 32) {
    const int tok = t + n;
    const bool ok = tok < t1;
    float qv[16], den = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) qv[s] = ok ? fmaxf(qn[s >> 2][s & 3], 0.f) : 0.f;
    if (t + 32 < t1) load_q(t + 32);
    f32x16_t num;
#pragma unroll
    for (int i = 0; i < 16; ++i) num[i] = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) num = __builtin_amdgcn_mfma_f32_32x32x2f32(a_num[s >> 2][s & 3], qv[s], num, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 16; ++s) den = fmaf(a_den[s >> 2][s & 3], qv[s], den);
    den += __shfl_xor(den, 32, 64);
    if (ok) {
      // D layout: lane -> token (column) lane%32; register r -> channel 8*(r/4)+4*g+r%4
      const float dd = den + eps;
      float* op = out + (int64_t)b * o_stride_b + (int64_t)tok * o_stride_n + head * D;
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<f32x4_t*>(op + 2 * r + 4 * g) = f32x4_t{num[r] / dd, num[r + 1] / dd, num[r + 2] / dd, num[r + 3] / dd};
    }
  }
}

// ----------------------------------------------------------------------------
// phase 2, fp32 io, on the partial states of one head (one chunk): the sum over the splits is formed here, in the order of
// linattn_reduce_scan_kernel, so that a short sequence needs two launches.  grid: B * h * 128-token ranges (per_range: 2^16 / ranges,
// rounded up: exact for fewer than 2^13 workgroups); block 320: waves 0 .. 3
// 32 tokens each, the fifth takes the state's 33rd row, so that the sums are one round of loads.  The partial states are requested first;
// a workgroup then reads nsplit x 4.2 KB of partial states, four times what its queries are at 16 splits, and that takes less than
// the third launch: bound by the latency of the two loads.  us, issued eagerly on three sets of inputs in turn, three launches / two:
// 1024 tokens x 36 heads 15.5 / 14.2, 400 x 70 14.2 / 13.8, 2 x 1024 x 36 20.6 / 17.7.  Both launches keep a head on one XCD: with its
// partial states read by all eight, phase 1 of the next call takes 9.1 us instead of 5.9 to write them again.  Beyond 1024 tokens, and
// beyond the heads that sana_hip_linattn takes it for, the partial states that are read again outweigh the launch.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(320) void linattn_apply32_partials_kernel(
    const float* __restrict__ Q, const float* __restrict__ partial, float* __restrict__ out, int N, int h, int nsplit,
    uint32_t per_range, int64_t q_stride_b, int64_t q_stride_n, int64_t o_stride_b, int64_t o_stride_n, float eps) {
  constexpr int ROW = D + 4;  // floats of a state row in LDS (conflict-free 16-byte reads down a column)
  __shared__ __attribute__((aligned(16))) float st[(D + 1) * ROW];
  asm volatile("" ::"s"(Q), "s"(partial), "s"(N), "s"(h), "s"(nsplit), "s"(per_range), "s"(q_stride_b), "s"(q_stride_n));  // (in one wait)
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ranges = (N + 127) >> 7, at = xcd_eighths(blockIdx.x, gridDim.x), bh = (int)((uint32_t)at * per_range >> 16);
  // the partial states first: their sum is the longer way
  const int e = min((int)threadIdx.x, STATE_ELEMS / 4 - 1);
  const float* p0 = partial + (int64_t)bh * nsplit * STATE_ELEMS;
  f32x4_t v[16];
#pragma unroll
  for (int u = 0; u < 16; ++u) v[u] = *reinterpret_cast<const f32x4_t*>(p0 + min(u, nsplit - 1) * STATE_ELEMS + 4 * e);
  const int b = (int)((uint32_t)bh / (uint32_t)h), head = bh - b * h;
  const int n = lane & 31, g = lane >> 5, tok = (at - bh * ranges) * 128 + wave * 32 + n;
  const bool ok = tok < N && wave < 4;
  f32x4_t q[4];
  const float* qp = Q + (int64_t)b * q_stride_b + (int64_t)min(tok, N - 1) * q_stride_n + head * D + 16 * g;
#pragma unroll
  for (int i = 0; i < 4; ++i) q[i] = *reinterpret_cast<const f32x4_t*>(qp + 4 * i);
  f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < 16; ++u)
    if (u < nsplit) s += v[u];
  if (threadIdx.x < STATE_ELEMS / 4) *reinterpret_cast<f32x4_t*>(st + (e >> 3) * ROW + 4 * (e & 7)) = s;
  __syncthreads();
  if (wave == 4) return;
  float qv[16], den = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) qv[i] = ok ? fmaxf(q[i >> 2][i & 3], 0.f) : 0.f;
  f32x16_t num;
#pragma unroll
  for (int i = 0; i < 16; ++i) num[i] = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(st + n * ROW + 16 * g + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) num = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], qv[4 * i + e], num, 0, 0, 0);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(st + D * ROW + 16 * g + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) den = fmaf(a[e], qv[4 * i + e], den);
  }
  den += __shfl_xor(den, 32, 64);
  if (ok) {  // (layouts: linattn_apply32_kernel)
    const float dd = den + eps;
    float* op = out + (int64_t)b * o_stride_b + (int64_t)tok * o_stride_n + head * D;
#pragma unroll
    for (int r = 0; r < 16; r += 4)
      *reinterpret_cast<f32x4_t*>(op + 2 * r + 4 * g) = f32x4_t{num[r] / dd, num[r + 1] / dd, num[r + 2] / dd, num[r + 3] / dd};
  }
}

// ----------------------------------------------------------------------------
// Both phases in one launch, for short sequences: one workgroup = one head of one batch entry (16-bit io, few heads: its state and
// a share of its queries), the state never leaves LDS.
// Three launches (phase 1, reduction, phase 2) are 3 - 6 us of work each with a gap in front; here everything a head needs
// for 1024 tokens is requested at once and the rest is one memory round trip, the transposes and the matrix products of one
// compute unit.  That is also the bound: a head's keys and values are one compute unit's work.  us, two calls / this, replayed from a
// graph on one set of inputs (on 16 in turn): bf16, 36 heads x 256 tokens 9.8 / 5.2 (10.5 / 6.0), 36 x 1024 12.1 / 8.8 (13.3 /
// 11.5), 140 x 1024 18.9 / 15.4 (22.2 / 17.0); fp16 36 x 256 10.5 / 5.8 (11.2 / 6.6); fp32 256 x 1024 35.9 / 26.7 (45.6 / 38.4).
// (Adding the state up in the two calls' order costs 0.4 us at 1024 tokens: sixteen partial states in LDS, not eight.)
// Two 16-bit heads share the 128-byte lines of their tokens: neighbours run on one XCD and meet in its L2 (workgroup ids alternate over
// the XCDs: 210 heads x 972 tokens 19.0 -> 16.8 us behind the GEMM that wrote them, 70 x 1024 12.0 -> 11.8).
// ----------------------------------------------------------------------------
constexpr int WHOLE_TOKENS = 1024;  // the most that one round of loads covers

// 16-bit io.  grid: B * h * R; block 512: R workgroups form the state of a head each for itself and share its queries.  The state is formed by the sums of linattn_state16_kernel and its reduction, in their
// order (at most 256 heads: always splits of 256 tokens), so that the result is that of the two calls bit for bit: "chain" c is
// what wave c % 4 of split c / 4 adds up there, the 32-token tiles 256 (c / 4) + 32 (c % 4) + {0, 128}.  Wave w takes chains w and
// w + 8 through its own LDS (rows of 96 bytes: conflict-free transposing reads).  Phase 2 as linattn_apply16_kernel, on the
// 16-token steps R w + part, R (w + 8) + part, ..
template <typename T, int R>
__global__ __launch_bounds__(512) void linattn_whole16_kernel(
    const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K, const uint16_t* __restrict__ V, uint16_t* __restrict__ out,
    int N, int h, int64_t q_stride_b, int64_t q_stride_n, int64_t stride_b, int64_t stride_n, int64_t o_stride_b,
    int64_t o_stride_n, float eps) {
  constexpr int WAVES = 8, ROW = 96, SPLIT = 256, CHAINS = 4 * WHOLE_TOKENS / SPLIT, U1 = CHAINS / WAVES,
                U2 = (WHOLE_TOKENS / 16 + WAVES * R - 1) / (WAVES * R);
  constexpr int STATE_AT = CHAINS * STATE_ELEMS * 4;
  static_assert(STATE_AT >= WAVES * 2 * TILE * ROW && STATE_AT >= WAVES * U2 * 1024, "the state lies behind the stages");
  __shared__ __attribute__((aligned(16))) unsigned char smem[STATE_AT + STATE_ELEMS * 4];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int at = xcd_eighths(blockIdx.x, gridDim.x), bh = at / R, part = at % R, b = bh / h, head = bh - b * h;
  const int ld_tok = lane >> 2, ld_chunk = lane & 3;  // a load instruction: 16 tokens x 64 bytes
  const uint16_t* kbase = K + (int64_t)b * stride_b + head * D;
  const uint16_t* vbase = V + (int64_t)b * stride_b + head * D;
  const uint16_t* qbase = Q + (int64_t)b * q_stride_b + head * D;
  uint16_t* obase = out + (int64_t)b * o_stride_b + head * D;

  // ---- phase 1
  auto tile_of = [&](int u, int t) {
    const int c = wave + WAVES * u;
    return SPLIT * (c >> 2) + TILE * (c & 3) + 128 * t;
  };
  auto query_of = [&](int u) { return ((wave + u * WAVES) * R + part) * 16; };  // phase 2, step u of this wave: its first token
  u32x4_t kreg[U1][2][2], vreg[U1][2][2], raw[U2];
  // Every load goes out without a branch: rows past N lie outside the resource (zeros).
  const bool near = max(max(q_stride_n, stride_n), o_stride_n) < (1 << 20);  // 32-bit offsets over 1024 rows
  auto resource = [&](const uint16_t* base, int64_t stride) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), 0, (N - 1) * (int)stride * 2 + 2 * D, 0x00020000);
  };
  auto offset = [&](int tok0, int64_t stride) { return (tok0 + ld_tok) * (int)stride * 2 + 16 * ld_chunk; };
  if (near) {
    const __amdgpu_buffer_rsrc_t rk = resource(kbase, stride_n), rv = resource(vbase, stride_n), rq = resource(qbase, q_stride_n);
#pragma unroll
    for (int u = 0; u < U1; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        if (tile_of(u, t) >= N) break;  // uniform (and not read below)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int o = offset(tile_of(u, t) + 16 * i, stride_n);
          kreg[u][t][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rk, o, 0, 0));
          vreg[u][t][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rv, o, 0, 0));
        }
      }
#pragma unroll
    for (int u = 0; u < U2; ++u) {
      if (query_of(u) >= N) break;  // uniform
      raw[u] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rq, offset(query_of(u), q_stride_n), 0, 0));
    }
  } else {
    auto row = [&](const uint16_t* base, int tok, int64_t stride) {
      return tok < N ? *reinterpret_cast<const u32x4_t*>(base + (int64_t)tok * stride + 8 * ld_chunk) : u32x4_t{0u, 0u, 0u, 0u};
    };
#pragma unroll
    for (int u = 0; u < U1; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int tok = tile_of(u, t) + 16 * i + ld_tok;
          kreg[u][t][i] = row(kbase, tok, stride_n), vreg[u][t][i] = row(vbase, tok, stride_n);
        }
#pragma unroll
    for (int u = 0; u < U2; ++u) raw[u] = row(qbase, query_of(u) + ld_tok, q_stride_n);
  }
  // MFMA 32x32x16: lane -> channel lane % 32, element r of k-step s is token 16 s + 2 r + lane / 32 of the tile.  A transposing
  // read hands the 16 lanes of a group four rows, row i addressed by lanes 4 i .. 4 i + 3: two tokens apart here.
  unsigned char* stage = smem + wave * (2 * TILE * ROW);
  const uint32_t stage_addr = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)stage;
  const uint32_t k_at = stage_addr + (2 * ((lane >> 2) & 3) + (lane >> 5)) * ROW + ((lane >> 4) & 1) * 32 + (lane & 3) * 8,
                 v_at = k_at + TILE * ROW;
  f32x16_t S[U1];
  float ks[U1];
#pragma unroll
  for (int u = 0; u < U1; ++u) {
#pragma unroll
    for (int i = 0; i < 16; ++i) S[u][i] = 0.f;
    ks[u] = 0.f;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if (tile_of(u, t) >= N) break;  // uniform
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        *reinterpret_cast<u32x4_t*>(stage + (16 * i + ld_tok) * ROW + 16 * ld_chunk) = relu_pk16(kreg[u][t][i]);
        *reinterpret_cast<u32x4_t*>(stage + TILE * ROW + (16 * i + ld_tok) * ROW + 16 * ld_chunk) = vreg[u][t][i];
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // wave-private LDS: in-order, no barrier needed
      u32x2_t kf[2][2], vf[2][2];  // [k-step][elements 4 i ..]
      kf[0][0] = lds_read_tr16<0>(k_at), kf[0][1] = lds_read_tr16<8 * ROW>(k_at);
      kf[1][0] = lds_read_tr16<16 * ROW>(k_at), kf[1][1] = lds_read_tr16<24 * ROW>(k_at);
      vf[0][0] = lds_read_tr16<0>(v_at), vf[0][1] = lds_read_tr16<8 * ROW>(v_at);
      vf[1][0] = lds_read_tr16<16 * ROW>(v_at), vf[1][1] = lds_read_tr16<24 * ROW>(v_at);
      asm volatile("s_waitcnt lgkmcnt(0)"
                   : "+v"(kf[0][0]), "+v"(kf[0][1]), "+v"(kf[1][0]), "+v"(kf[1][1]), "+v"(vf[0][0]), "+v"(vf[0][1]),
                     "+v"(vf[1][0]), "+v"(vf[1][1])::"memory");
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const u32x4_t kk = {kf[s][0].x, kf[s][0].y, kf[s][1].x, kf[s][1].y};
        S[u] = mfma_32x32x16<T>(u32x4_t{vf[s][0].x, vf[s][0].y, vf[s][1].x, vf[s][1].y}, kk, S[u]);
#pragma unroll
        for (int e = 0; e < 4; ++e) ks[u] = add_pk16<T>(kk[e], ks[u]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < U1; ++u) {
    const int c = wave + WAVES * u;
    if (SPLIT * (c >> 2) >= N) break;  // uniform: no such split
    float* red = reinterpret_cast<float*>(smem) + c * STATE_ELEMS;
    const int j = lane & 31, g2 = lane >> 5;
#pragma unroll
    for (int r = 0; r < 16; ++r) red[(8 * (r >> 2) + 4 * g2 + (r & 3)) * D + j] = S[u][r];
    const float both = ks[u] + __shfl_xor(ks[u], 32, 64);
    if (g2 == 0) red[D * D + j] = both;
  }
  __syncthreads();
  float* state = reinterpret_cast<float*>(smem + STATE_AT);
  if (tid < STATE_ELEMS / 4) {  // the waves of a split, then the splits
    const f32x4_t* p = reinterpret_cast<const f32x4_t*>(smem) + tid;
    constexpr int STEP = STATE_ELEMS / 4;
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sp = 0; sp < CHAINS / 4; ++sp) {
      if (SPLIT * sp >= N) break;  // uniform
      s += ((p[(4 * sp) * STEP] + p[(4 * sp + 1) * STEP]) + p[(4 * sp + 2) * STEP]) + p[(4 * sp + 3) * STEP];
    }
    reinterpret_cast<f32x4_t*>(state)[tid] = s;
  }
  __syncthreads();

  // ---- phase 2 (operand layout: linattn_apply16_kernel)
  const int n = lane & 15, g = lane >> 4;
  u32x4_t st[3][3];
#pragma unroll
  for (int rb = 0; rb < 3; ++rb) {
    const float* sp = state + (rb < 2 ? 8 * (n >> 2) + 4 * rb + (n & 3) : D) * D + 8 * g;
    const f32x4_t x0 = *reinterpret_cast<const f32x4_t*>(sp), x1 = *reinterpret_cast<const f32x4_t*>(sp + 4);
    const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
    split3(x, st[rb]);
  }
  unsigned char* qstage = smem + wave * (U2 * 1024);
  const int slot_w = 16 * (4 * ld_tok + (ld_chunk ^ ((ld_tok >> 1) & 3)));
  const int slot_r = 16 * (4 * n + (g ^ ((n >> 1) & 3)));
#pragma unroll
  for (int u = 0; u < U2; ++u) {
    if (query_of(u) >= N) break;  // uniform
    *reinterpret_cast<u32x4_t*>(qstage + u * 1024 + slot_w) = relu_pk16(raw[u]);
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int u = 0; u < U2; ++u) {
    if (query_of(u) >= N) break;  // uniform
    unsigned char* slot = qstage + u * 1024 + slot_r;
    const u32x4_t qd = *reinterpret_cast<const u32x4_t*>(slot);
    u32x4_t q_hi, q_lo;
    if constexpr (is_f16<T>) f16_to_2bf16(qd, q_hi, q_lo);
    f32x4_t acc[3];
#pragma unroll
    for (int rb = 0; rb < 3; ++rb) {
      f32x4_t a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int term = 2; term >= 0; --term) {  // smallest terms first
        if constexpr (is_f16<T>) {
          a = mfma_16x16x32_bf16(st[rb][term], q_lo, a);
          a = mfma_16x16x32_bf16(st[rb][term], q_hi, a);
        } else {
          a = mfma_16x16x32_bf16(st[rb][term], qd, a);
        }
      }
      acc[rb] = a;
    }
    const float den = acc[2][0] + eps;
    u32x4_t o;
    if constexpr (is_f16<T>) {
      const Quotient by(den);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pk16<T>(by(acc[e >> 1][2 * (e & 1)]), by(acc[e >> 1][2 * (e & 1) + 1]));
    } else {
      const float inv = __builtin_amdgcn_rcpf(den);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = pk16<T>(acc[e >> 1][2 * (e & 1)] * inv, acc[e >> 1][2 * (e & 1) + 1] * inv);
    }
    *reinterpret_cast<u32x4_t*>(slot) = o;  // in the place of this lane's queries
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (near) {
    const __amdgpu_buffer_rsrc_t ro = resource(obase, o_stride_n);
#pragma unroll
    for (int u = 0; u < U2; ++u) {
      if (query_of(u) >= N) break;  // uniform
      __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4_t*>(qstage + u * 1024 + slot_w), ro,
                                             offset(query_of(u), o_stride_n), 0, 0);
    }
  } else {
#pragma unroll
    for (int u = 0; u < U2; ++u) {
      const int tok = query_of(u) + ld_tok;
      const u32x4_t o = *reinterpret_cast<const u32x4_t*>(qstage + u * 1024 + slot_w);
      if (tok < N) *reinterpret_cast<u32x4_t*>(obase + (int64_t)tok * o_stride_n + 8 * ld_chunk) = o;
    }
  }
}

// fp32 io.  grid: B * h; block 1024.  Phase 1 as linattn_state32_kernel with the waves as its splits (split_tokens as planned for
// it, at most 16 splits) and their sums added in its order: the two calls' result bit for bit.  Phase 2 as
// linattn_apply32_kernel on the 32-token tiles w, w + 16, ..
__global__ __launch_bounds__(1024) void linattn_whole32_kernel(
    const float* __restrict__ Q, const float* __restrict__ K, const float* __restrict__ V, float* __restrict__ out, int N, int h,
    int split_tokens, int64_t q_stride_b, int64_t q_stride_n, int64_t stride_b, int64_t stride_n, int64_t o_stride_b,
    int64_t o_stride_n, float eps) {
  constexpr int WAVES = WHOLE_TOKENS / 64, U = 16;
  __shared__ __attribute__((aligned(16))) float smem[(WAVES + 1) * STATE_ELEMS];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int b = blockIdx.x / h, head = blockIdx.x - b * h;
  const int j = lane & 31, g = lane >> 5;
  const float* kp = K + (int64_t)b * stride_b + head * D + j;
  const float* vp = V + (int64_t)b * stride_b + head * D + j;
  f32x16_t accS;
  float accK = 0.f;
#pragma unroll
  for (int i = 0; i < 16; ++i) accS[i] = 0.f;
  const int t1 = min((wave + 1) * split_tokens, N);
#pragma unroll 1
  for (int t = wave * split_tokens; t < t1; t += 2 * U) {  // (64 tokens at once need more registers than there are)
    float kk[U], vv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int64_t at = (int64_t)min(t + 2 * u + g, t1 - 1) * stride_n;  // (no branch around a load)
      kk[u] = kp[at], vv[u] = vp[at];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool ok = t + 2 * u + g < t1;
      kk[u] = ok ? fmaxf(kk[u], 0.f) : 0.f;
      vv[u] = ok ? vv[u] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      accS = __builtin_amdgcn_mfma_f32_32x32x2f32(vv[u], kk[u], accS, 0, 0, 0);
      accK += kk[u];
    }
  }
  f32x4_t qn[4];
  auto load_q = [&](int t) {
    const float* qp = Q + (int64_t)b * q_stride_b + (int64_t)min(t + j, N - 1) * q_stride_n + head * D + 16 * g;
#pragma unroll
    for (int i = 0; i < 4; ++i) qn[i] = *reinterpret_cast<const f32x4_t*>(qp + 4 * i);
  };
  load_q(wave * 32);  // (a wave without a tile: the last token)
  float* red = smem + wave * STATE_ELEMS;
#pragma unroll
  for (int r = 0; r < 16; ++r) red[(8 * (r >> 2) + 4 * g + (r & 3)) * D + j] = accS[r];
  accK += __shfl_xor(accK, 32, 64);
  if (g == 0) red[D * D + j] = accK;
  __syncthreads();
  float* state = smem + WAVES * STATE_ELEMS;
  for (int e = threadIdx.x; e < STATE_ELEMS; e += 64 * WAVES) {
    float s = smem[e];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) s += smem[w * STATE_ELEMS + e];
    state[e] = s;
  }
  __syncthreads();
  f32x4_t a_num[4], a_den[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a_num[i] = *reinterpret_cast<const f32x4_t*>(state + j * D + 16 * g + 4 * i);
    a_den[i] = *reinterpret_cast<const f32x4_t*>(state + D * D + 16 * g + 4 * i);
  }
  for (int t = wave * 32; t < N; t += WAVES * 32) {
    const int tok = t + j;
    const bool ok = tok < N;
    float qv[16], den = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) qv[s] = ok ? fmaxf(qn[s >> 2][s & 3], 0.f) : 0.f;
    if (t + WAVES * 32 < N) load_q(t + WAVES * 32);
    f32x16_t num;
#pragma unroll
    for (int i = 0; i < 16; ++i) num[i] = 0.f;
#pragma unroll
    for (int s = 0; s < 16; ++s) num = __builtin_amdgcn_mfma_f32_32x32x2f32(a_num[s >> 2][s & 3], qv[s], num, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 16; ++s) den = fmaf(a_den[s >> 2][s & 3], qv[s], den);
    den += __shfl_xor(den, 32, 64);
    if (ok) {
      const float dd = den + eps;
      float* op = out + (int64_t)b * o_stride_b + (int64_t)tok * o_stride_n + head * D;
#pragma unroll
      for (int r = 0; r < 16; r += 4)
        *reinterpret_cast<f32x4_t*>(op + 2 * r + 4 * g) = f32x4_t{num[r] / dd, num[r + 1] / dd, num[r + 2] / dd, num[r + 3] / dd};
    }
  }
}

// ----------------------------------------------------------------------------
// Per-token 1/rms of q and of k over all C channels (the statistic of the reference's
// RMSNorm before the head split): rinv = rsqrt(mean(x^2) + eps).  One wave per (token, tensor).
// grid: x = ceil(B*N/4), y = 2 (q, k); block 256.
// ----------------------------------------------------------------------------
__global__ __launch_bounds__(256) void qk_rms_kernel(const uint16_t* __restrict__ Q, const uint16_t* __restrict__ K,
                                                     float* __restrict__ rq, float* __restrict__ rk, int64_t BN,
                                                     int N, int C, int64_t stride_b, int64_t stride_n, float eps) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + wave;
  if (row >= BN) return;
  const uint16_t* x = (blockIdx.y == 0 ? Q : K) + (row / N) * stride_b + (row % N) * stride_n;
  float acc = 0.f;
  for (int c0 = lane * 8; c0 < C; c0 += 512) {
    const u32x4_t v = *reinterpret_cast<const u32x4_t*>(x + c0);  // cacheable: the attention kernels read q and k next
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float a = bf16_lo(v[e]), b2 = bf16_hi(v[e]);
      acc = fmaf(a, a, acc);
      acc = fmaf(b2, b2, acc);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (lane == 0) (blockIdx.y == 0 ? rq : rk)[row] = rsqrtf(acc / (float)C + eps);
}

// ---------------------------------------------------------------------------- host side

int pick_nsplit(int items, int max_chunk_tokens, int min_tokens) {
  // aim for >= 1024 workgroups (four per CU), but keep >= min_tokens tokens per split
  int ns = (1024 + items - 1) / items;
  const int cap = (max_chunk_tokens + min_tokens - 1) / min_tokens;
  if (ns > cap) ns = cap;
  if (ns < 1) ns = 1;
  if (ns > 64) ns = 64;
  return ns;
}
int split_len(int max_chunk_tokens, int nsplit, int granule) {
  int len = (max_chunk_tokens + nsplit - 1) / nsplit;
  return (len + granule - 1) / granule * granule;
}

struct StatePlan {
  int items;   // workgroups before splitting
  int nsplit;
  int split_tokens;
};
StatePlan plan_state(int B, int h, int n_chunks, int max_chunk_tokens, int io_dtype) {
  StatePlan pl;
  const int per_b = (io_dtype == SANA_DT_F32) ? (h + 3) / 4 : (h + 1) / 2;
  pl.items = B * per_b * n_chunks;
  // 16-bit: four waves x 32-token tiles per round; fp32: 16 tokens per wave iteration
  const bool f32 = io_dtype == SANA_DT_F32;
  pl.nsplit = pick_nsplit(pl.items, max_chunk_tokens, f32 ? 64 : 256);
  pl.split_tokens = split_len(max_chunk_tokens, pl.nsplit, f32 ? 16 : 128);
  // drop splits that would be empty after rounding the length up
  pl.nsplit = (max_chunk_tokens + pl.split_tokens - 1) / pl.split_tokens;
  if (pl.nsplit < 1) pl.nsplit = 1;
  return pl;
}

}  // namespace
}  // namespace sana

using namespace sana;

extern "C" __attribute__((visibility("default"))) size_t sana_hip_linattn_workspace_bytes(int B, int h, int d,
                                                                                          int n_chunks,
                                                                                          int max_chunk_tokens,
                                                                                          int io_dtype) {
  if (B <= 0 || h <= 0 || (d != D && d != 112) || n_chunks <= 0 || max_chunk_tokens <= 0) return 0;
  if (d == 112) return io_dtype == SANA_DT_F32 ? 0 : workspace_bytes112(B, h, n_chunks, max_chunk_tokens);
  const StatePlan pl = plan_state(B, h, n_chunks, max_chunk_tokens, io_dtype);
  return pl.nsplit > 1 ? (size_t)B * h * n_chunks * pl.nsplit * STATE_ELEMS * sizeof(float) : 0;
}

static int check_pre(const QkPre& pre, int io_dtype) {
  if (!pre.rinv && !pre.rope) return SANA_OK;
  if (io_dtype != SANA_DT_BF16) return SANA_ERR_DTYPE;
  if (pre.rinv && !pre.weight) return SANA_ERR_ARG;
  if (pre.rope_first && !pre.rope) return SANA_ERR_ARG;
  if ((pre.weight && !aligned16(pre.weight)) || (pre.rope && !aligned16(pre.rope))) return SANA_ERR_ALIGN;
  return SANA_OK;
}

static int state_impl(const void* k, const void* v, float* state, void* workspace, size_t workspace_bytes, int B,
                      int N, int h, int d, int64_t stride_b, int64_t stride_n, const int32_t* chunk_starts,
                      int n_chunks, int max_chunk_tokens, int causal, int io_dtype, const QkPre pre, void* stream) {
  if (!k || !v || !state || B <= 0 || N <= 0 || h <= 0 || n_chunks <= 0) return SANA_ERR_ARG;
  {
    const int rc = check_pre(pre, io_dtype);
    if (rc != SANA_OK) return rc;
  }
  if (d != D && d != 112) return SANA_ERR_SHAPE;
  if (n_chunks > 1 && !chunk_starts) return SANA_ERR_ARG;
  if (n_chunks == 1 && !chunk_starts) max_chunk_tokens = N;
  if (max_chunk_tokens <= 0 || max_chunk_tokens > N) return SANA_ERR_ARG;
  if (io_dtype != SANA_DT_F32 && io_dtype != SANA_DT_BF16 && io_dtype != SANA_DT_F16) return SANA_ERR_DTYPE;
  if (stride_n < (int64_t)h * d || stride_b < 0) return SANA_ERR_ARG;
  if ((int64_t)B * h > (1 << 22) || n_chunks > 65535) return SANA_ERR_SHAPE;
  const int esz = io_dtype == SANA_DT_F32 ? 4 : 2;
  if (!aligned16(k) || !aligned16(v) || !aligned16(state) || (stride_n * esz) % 16 || (stride_b * esz) % 16)
    return SANA_ERR_ALIGN;
  if (d == 112 && pre.rope_first) return SANA_ERR_SHAPE;  // the rotate-first order exists for head_dim 32 only
  if (d == 112)
    return launch_state112(k, v, state, workspace, workspace_bytes, B, N, h, stride_b, stride_n, chunk_starts, n_chunks,
                           max_chunk_tokens, causal, io_dtype, pre, static_cast<hipStream_t>(stream));
  const StatePlan pl = plan_state(B, h, n_chunks, max_chunk_tokens, io_dtype);
  float* dst = state;
  if (pl.nsplit > 1) {
    const size_t need = (size_t)B * h * n_chunks * pl.nsplit * STATE_ELEMS * sizeof(float);
    if (!workspace || workspace_bytes < need) return SANA_ERR_WORKSPACE;
    if (!aligned16(workspace)) return SANA_ERR_ALIGN;
    dst = static_cast<float*>(workspace);
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (io_dtype == SANA_DT_F32) {
    dim3 grid(pl.nsplit, n_chunks, B * ((h + 3) / 4));
    const bool far = (int64_t)(pl.split_tokens + 64) * stride_n >= (1 << 29);  // beyond the 32-bit offsets
    hipLaunchKernelGGL((far ? linattn_state32_kernel<false, true> : linattn_state32_kernel<false, false>), grid, dim3(256), 0, s, static_cast<const float*>(k),
                       static_cast<const float*>(v), dst, chunk_starts, N, h, n_chunks, pl.nsplit,
                       pl.split_tokens, stride_b, stride_n);
  } else {
    dim3 grid(pl.nsplit, n_chunks, B * ((h + 1) / 2));
    const int mode = (pre.rinv ? 1 : 0) | (pre.rope ? 2 : 0) | (pre.rope_first ? 4 : 0);
#define SANA_STATE16(T, PRE)                                                                                  \
  hipLaunchKernelGGL((linattn_state16_kernel<T, PRE>), grid, dim3(256), 0, s, static_cast<const uint16_t*>(k), \
                     static_cast<const uint16_t*>(v), dst, chunk_starts, N, h, n_chunks, pl.nsplit,           \
                     pl.split_tokens, stride_b, stride_n, pre)
    if (io_dtype == SANA_DT_F16) SANA_STATE16(F16, 0);
    else if (mode == 7) SANA_STATE16(BF16, 7);
    else if (mode == 6) SANA_STATE16(BF16, 6);
    else if (mode == 3) SANA_STATE16(BF16, 3);
    else if (mode == 2) SANA_STATE16(BF16, 2);
    else if (mode == 1) SANA_STATE16(BF16, 1);
    else SANA_STATE16(BF16, 0);
#undef SANA_STATE16
  }
  if (hipGetLastError() != hipSuccess) return SANA_ERR_LAUNCH;
  const bool scan = causal && n_chunks > 1;
  if (pl.nsplit > 1 || scan) {
    const int64_t threads = (int64_t)B * h * STATE_ELEMS;
    hipLaunchKernelGGL(linattn_reduce_scan_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, dst,
                       state, B * h, n_chunks, pl.nsplit, scan ? 1 : 0);
    if (hipGetLastError() != hipSuccess) return SANA_ERR_LAUNCH;
  }
  return SANA_OK;
}

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn_state(
    const void* k, const void* v, float* state, void* workspace, size_t workspace_bytes, int B, int N, int h, int d,
    int64_t stride_b, int64_t stride_n, const int32_t* chunk_starts, int n_chunks, int max_chunk_tokens, int causal,
    int io_dtype, void* stream) {
  const QkPre none = {nullptr, nullptr, nullptr, 0};
  return state_impl(k, v, state, workspace, workspace_bytes, B, N, h, d, stride_b, stride_n, chunk_starts, n_chunks,
                    max_chunk_tokens, causal, io_dtype, none, stream);
}

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn_state_pre(
    const void* k, const void* v, float* state, void* workspace, size_t workspace_bytes, int B, int N, int h, int d,
    int64_t stride_b, int64_t stride_n, const int32_t* chunk_starts, int n_chunks, int max_chunk_tokens, int causal,
    int io_dtype, const float* k_rinv, const void* k_weight, const float* rope, void* stream) {
  const QkPre pre = {k_rinv, static_cast<const uint16_t*>(k_weight), rope, 0};
  return state_impl(k, v, state, workspace, workspace_bytes, B, N, h, d, stride_b, stride_n, chunk_starts, n_chunks,
                    max_chunk_tokens, causal, io_dtype, pre, stream);
}

extern "C" __attribute__((visibility("default"))) int sana_hip_litela_state(
    const void* k, const void* v, float* state, void* workspace, size_t workspace_bytes, int B, int N, int h, int d,
    int64_t stride_b, int64_t stride_n, int io_dtype, const float* k_rinv, const void* k_weight, const float* rope,
    void* stream) {
  const QkPre pre = {k_rinv, static_cast<const uint16_t*>(k_weight), rope, rope ? 1 : 0};
  return state_impl(k, v, state, workspace, workspace_bytes, B, N, h, d, stride_b, stride_n, nullptr, 1, N, 0, io_dtype,
                    pre, stream);
}

// ---------------------------------------------------------------------------- phase 1 without a workspace argument
// For callers that cannot allocate (code under HIP graph capture, serving loops, harnesses that forbid it): the
// per-split partial states go to a fixed array in device memory instead of a caller-provided workspace.  Each GPU
// the library runs on holds its own copy of the array, at its own address, until the process ends.  `scratch` is a
// host-side stand-in for that symbol, not a device address: host code uses the address hipGetSymbolAddress returns
// for the current device and never the array's name.
static __device__ __align__(256) unsigned char scratch[SANA_HIP_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_addr[kMaxDevices];  // device address of `scratch` per GPU, looked up once per device
std::mutex g_scratch_mutex;

// The current device's copy of the array, or null when the runtime refuses the lookup.
void* scratch_of_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  void* p = g_scratch_addr[dev].load(std::memory_order_acquire);
  if (p) return p;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  p = g_scratch_addr[dev].load(std::memory_order_relaxed);
  if (!p) {
    void* addr = nullptr;
    if (hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)) != hipSuccess || !addr) return nullptr;
    g_scratch_addr[dev].store(addr, std::memory_order_release);
    p = addr;
  }
  return p;
}
}  // namespace

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn_state_noalloc(
    const void* k, const void* v, float* state, int B, int N, int h, int d, int64_t stride_b, int64_t stride_n,
    const int32_t* chunk_starts, int n_chunks, int max_chunk_tokens, int causal, int io_dtype, const float* k_rinv,
    const void* k_weight, const float* rope, void* stream) {
  if (B <= 0 || N <= 0 || h <= 0 || n_chunks <= 0) return SANA_ERR_ARG;
  const int longest = (n_chunks == 1 && !chunk_starts) ? N : max_chunk_tokens;
  const size_t need = sana_hip_linattn_workspace_bytes(B, h, d, n_chunks, longest, io_dtype);
  if (need > (size_t)SANA_HIP_NOALLOC_SCRATCH_BYTES) return SANA_ERR_SCRATCH_LIMIT;
  void* ws = scratch_of_current_device();
  if (!ws) return SANA_ERR_RUNTIME;
  // every partial state the reduction reads is written by the launch before it (empty splits write zeros), so the
  // array's old contents never reach a result and nothing has to be cleared
  const QkPre pre = {k_rinv, static_cast<const uint16_t*>(k_weight), rope, 0};
  return state_impl(k, v, state, ws, (size_t)SANA_HIP_NOALLOC_SCRATCH_BYTES, B, N, h, d, stride_b, stride_n,
                    chunk_starts, n_chunks, max_chunk_tokens, causal, io_dtype, pre, stream);
}

extern "C" __attribute__((visibility("default"))) int sana_hip_qk_rms(const void* q, const void* k, float* q_rinv,
                                                                      float* k_rinv, int B, int N, int C,
                                                                      int64_t stride_b, int64_t stride_n, float eps,
                                                                      int io_dtype, void* stream) {
  if (!q || !k || !q_rinv || !k_rinv || B <= 0 || N <= 0 || C <= 0) return SANA_ERR_ARG;
  if (io_dtype != SANA_DT_BF16) return SANA_ERR_DTYPE;
  if (C % 8) return SANA_ERR_SHAPE;
  if (stride_n < C || stride_b < 0) return SANA_ERR_ARG;
  if (!aligned16(q) || !aligned16(k) || (stride_n * 2) % 16 || (stride_b * 2) % 16) return SANA_ERR_ALIGN;
  const int64_t BN = (int64_t)B * N;
  if ((BN + 3) / 4 > 0x7fffffff) return SANA_ERR_SHAPE;
  hipLaunchKernelGGL(qk_rms_kernel, dim3((unsigned)((BN + 3) / 4), 2), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint16_t*>(q), static_cast<const uint16_t*>(k), q_rinv, k_rinv, BN, N, C,
                     stride_b, stride_n, eps);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn_chunk_scan(float* state, int B, int h, int d, int n_chunks, void* stream) {
  if (!state || B <= 0 || h <= 0 || n_chunks <= 0) return SANA_ERR_ARG;
  if (d != D && d != 112) return SANA_ERR_SHAPE;
  if (n_chunks == 1) return SANA_OK;
  if (d == 112) return launch_scan112(state, B, h, n_chunks, static_cast<hipStream_t>(stream));
  const int64_t threads = (int64_t)B * h * STATE_ELEMS;
  hipLaunchKernelGGL(linattn_reduce_scan_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), state, state, B * h, n_chunks, 1, 1);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

static int apply_impl(const void* q, const float* state, void* out, int B, int N, int h, int d, int64_t q_stride_b,
                      int64_t q_stride_n, int64_t o_stride_b, int64_t o_stride_n, const int32_t* chunk_starts,
                      int n_chunks, int max_chunk_tokens, float eps, int io_dtype, int out_dtype, const QkPre pre,
                      void* stream) {
  if (!q || !state || !out || B <= 0 || N <= 0 || h <= 0 || n_chunks <= 0) return SANA_ERR_ARG;
  {
    const int rc = check_pre(pre, io_dtype);
    if (rc != SANA_OK) return rc;
  }
  if (d != D && d != 112) return SANA_ERR_SHAPE;
  if (n_chunks > 1 && !chunk_starts) return SANA_ERR_ARG;
  if (n_chunks == 1 && !chunk_starts) max_chunk_tokens = N;
  if (max_chunk_tokens <= 0 || max_chunk_tokens > N) return SANA_ERR_ARG;
  if (io_dtype != SANA_DT_F32 && io_dtype != SANA_DT_BF16 && io_dtype != SANA_DT_F16) return SANA_ERR_DTYPE;
  if (out_dtype != io_dtype && out_dtype != SANA_DT_F32) return SANA_ERR_DTYPE;
  if (q_stride_n < (int64_t)h * d || o_stride_n < (int64_t)h * d || q_stride_b < 0 || o_stride_b < 0)
    return SANA_ERR_ARG;
  if ((int64_t)B * h > (1 << 22) || n_chunks > 65535) return SANA_ERR_SHAPE;
  const int qsz = io_dtype == SANA_DT_F32 ? 4 : 2, osz = out_dtype == SANA_DT_F32 ? 4 : 2;
  if (!aligned16(q) || !aligned16(state) || !aligned16(out) || (q_stride_n * qsz) % 16 || (q_stride_b * qsz) % 16 ||
      (o_stride_n * osz) % 16 || (o_stride_b * osz) % 16)
    return SANA_ERR_ALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (d == 112 && pre.rope_first) return SANA_ERR_SHAPE;
  if (d == 112)
    return launch_apply112(q, state, out, B, N, h, q_stride_b, q_stride_n, o_stride_b, o_stride_n, chunk_starts,
                           n_chunks, max_chunk_tokens, eps, io_dtype, out_dtype, pre, s);
  // tokens per workgroup: enough to share the state's preparation, fewer where the grid would not fill the chip (bf16,
  // tokens x heads, us: 256 x 36 7.1 -> 4.2, 1024 x 36 7.3 -> 4.5, 1024 x 70 7.6 -> 5.9; with 512 workgroups as the
  // target 2916 x 70 would go from 9.4 to 12.4, with 256 it is 8.9)
  const int64_t combos = (int64_t)n_chunks * B * (io_dtype == SANA_DT_F32 ? (h + 3) / 4 : ((h + 1) / 2 + 3) / 4);
  int wg_tokens = io_dtype == SANA_DT_F32 ? 64 : SANA_LA_APPLY_TOKENS;
  while (wg_tokens > 32 && combos * ((max_chunk_tokens + wg_tokens - 1) / wg_tokens) < SANA_LA_APPLY_MINWG) wg_tokens /= 2;
  const unsigned gx = (unsigned)((max_chunk_tokens + wg_tokens - 1) / wg_tokens);
  if (io_dtype != SANA_DT_F32) {
    const int pairs = (h + 1) / 2;
    dim3 grid(gx, n_chunks, B * ((pairs + 3) / 4));
    // many distinct states (chunk-causal video shapes): keep the readers of one state on one XCD
    int ngroups = n_chunks * B * ((pairs + 3) / 4);
    if (ngroups >= 64 && (int64_t)((ngroups + 7) / 8) * 8 * gx < 0x7fffffff)
      grid = dim3((unsigned)((ngroups + 7) / 8 * 8) * gx, 1, 1);
    else
      ngroups = 0;
#define SANA_APPLY(T, F32, PRE)                                                                                \
  hipLaunchKernelGGL((linattn_apply16_kernel<T, F32, PRE>), grid, dim3(256), 0, s, static_cast<const uint16_t*>(q), \
                     state, out, chunk_starts, N, h, n_chunks, wg_tokens, q_stride_b, q_stride_n, o_stride_b,     \
                     o_stride_n, eps, pre, (int)gx, ngroups)
    const int mode = (pre.rinv ? 1 : 0) | (pre.rope ? 2 : 0) | (pre.rope_first ? 4 : 0);
    if (io_dtype == SANA_DT_F16) {  // (check_pre: no norm or rotation on load)
      if (out_dtype == SANA_DT_F32) SANA_APPLY(F16, true, 0);
      else SANA_APPLY(F16, false, 0);
    } else if (out_dtype == SANA_DT_F32) {
      if (mode == 7) SANA_APPLY(BF16, true, 7);
      else if (mode == 6) SANA_APPLY(BF16, true, 6);
      else if (mode == 3) SANA_APPLY(BF16, true, 3);
      else if (mode == 2) SANA_APPLY(BF16, true, 2);
      else if (mode == 1) SANA_APPLY(BF16, true, 1);
      else SANA_APPLY(BF16, true, 0);
    } else {
      if (mode == 7) SANA_APPLY(BF16, false, 7);
      else if (mode == 6) SANA_APPLY(BF16, false, 6);
      else if (mode == 3) SANA_APPLY(BF16, false, 3);
      else if (mode == 2) SANA_APPLY(BF16, false, 2);
      else if (mode == 1) SANA_APPLY(BF16, false, 1);
      else SANA_APPLY(BF16, false, 0);
    }
#undef SANA_APPLY
  } else {
    dim3 grid(gx, n_chunks, B * ((h + 3) / 4));
    hipLaunchKernelGGL(linattn_apply32_kernel, grid, dim3(256), 0, s, static_cast<const float*>(q), state,
                       static_cast<float*>(out), chunk_starts, N, h, n_chunks, wg_tokens, q_stride_b, q_stride_n, o_stride_b,
                       o_stride_n, eps);
  }
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn_apply(
    const void* q, const float* state, void* out, int B, int N, int h, int d, int64_t q_stride_b, int64_t q_stride_n,
    int64_t o_stride_b, int64_t o_stride_n, const int32_t* chunk_starts, int n_chunks, int max_chunk_tokens,
    float eps, int io_dtype, int out_dtype, void* stream) {
  const QkPre none = {nullptr, nullptr, nullptr, 0};
  return apply_impl(q, state, out, B, N, h, d, q_stride_b, q_stride_n, o_stride_b, o_stride_n, chunk_starts,
                    n_chunks, max_chunk_tokens, eps, io_dtype, out_dtype, none, stream);
}

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn_apply_pre(
    const void* q, const float* state, void* out, int B, int N, int h, int d, int64_t q_stride_b, int64_t q_stride_n,
    int64_t o_stride_b, int64_t o_stride_n, const int32_t* chunk_starts, int n_chunks, int max_chunk_tokens,
    float eps, int io_dtype, int out_dtype, const float* q_rinv, const void* q_weight, const float* rope,
    void* stream) {
  const QkPre pre = {q_rinv, static_cast<const uint16_t*>(q_weight), rope, 0};
  return apply_impl(q, state, out, B, N, h, d, q_stride_b, q_stride_n, o_stride_b, o_stride_n, chunk_starts,
                    n_chunks, max_chunk_tokens, eps, io_dtype, out_dtype, pre, stream);
}

extern "C" __attribute__((visibility("default"))) int sana_hip_litela_apply(
    const void* q, const float* state, void* out, int B, int N, int h, int d, int64_t q_stride_b, int64_t q_stride_n,
    int64_t o_stride_b, int64_t o_stride_n, float eps, int io_dtype, int out_dtype, const float* q_rinv,
    const void* q_weight, const float* rope, void* stream) {
  const QkPre pre = {q_rinv, static_cast<const uint16_t*>(q_weight), rope, rope ? 1 : 0};
  return apply_impl(q, state, out, B, N, h, d, q_stride_b, q_stride_n, o_stride_b, o_stride_n, nullptr, 1, N, eps,
                    io_dtype, out_dtype, pre, stream);
}

// One launch while a head is a short piece of work and every head has a compute unit.  us, the launches of the two calls / one,
// from a graph on 16 sets of inputs in turn (what another kernel has just written is not in the reading XCD's L2 either):
// bf16 36 x 1024 13.3 / 11.5, 256 x 1024 27.6 / 25.1, but 280 x 1024 32.2 / 38.4 (a second round); f16 36 x 1024 14.0 / 14.0, 256 x
// 1024 29.5 / 27.2.  fp32 moves twice the bytes and has the slower matrix instruction, so that beyond 256 tokens a head is too much
// for one compute unit while others idle: 70 x 512 18.6 / 22.9, 108 x 768 25.0 / 27.6, 140 x 768 26.3 / 28.2, and 180 x 512 25.5 /
// 25.5, 180 x 768 33.0 / 29.2, 256 x 1024 45.6 / 38.4.  Up to 256 the spared launches decide, issued eagerly 15.7 / 14.3 for 36 x
// 256 (from the graph 13.3 / 14.5), 16.4 / 13.5 for 70 x 128 (13.3 / 13.5).
static bool one_launch(int B, int N, int h, int io_dtype) {
  const int64_t heads = (int64_t)B * h;
  if (N > WHOLE_TOKENS || heads > 256) return false;
  return io_dtype != SANA_DT_F32 || N <= 256 || heads >= 160;
}
static size_t state_bytes(int B, int h) { return ((size_t)B * h * STATE_ELEMS * sizeof(float) + 255) & ~(size_t)255; }

extern "C" __attribute__((visibility("default"))) size_t sana_hip_linattn_scratch_bytes(int B, int N, int h, int d, int io_dtype) {
  if (B <= 0 || N <= 0 || h <= 0 || d != D || one_launch(B, N, h, io_dtype)) return 0;
  return state_bytes(B, h) + sana_hip_linattn_workspace_bytes(B, h, d, 1, N, io_dtype);
}

extern "C" __attribute__((visibility("default"))) int sana_hip_linattn(
    const void* q, const void* k, const void* v, void* out, void* scratch, size_t scratch_bytes, int B, int N, int h, int d,
    int64_t q_stride_b, int64_t q_stride_n, int64_t stride_b, int64_t stride_n, int64_t o_stride_b, int64_t o_stride_n, float eps,
    int io_dtype, void* stream) {
  if (!q || !k || !v || !out || B <= 0 || N <= 0 || h <= 0) return SANA_ERR_ARG;
  if (d != D) return SANA_ERR_SHAPE;
  if (io_dtype != SANA_DT_F32 && io_dtype != SANA_DT_BF16 && io_dtype != SANA_DT_F16) return SANA_ERR_DTYPE;
  const int64_t C = (int64_t)h * d, heads = (int64_t)B * h, vec = io_dtype == SANA_DT_F32 ? 4 : 8;  // values in 16 bytes
  if (q_stride_n < C || stride_n < C || o_stride_n < C || q_stride_b < 0 || stride_b < 0 || o_stride_b < 0) return SANA_ERR_ARG;
  if (heads > (1 << 22)) return SANA_ERR_SHAPE;
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out)) return SANA_ERR_ALIGN;
  for (int64_t x : {q_stride_b, q_stride_n, stride_b, stride_n, o_stride_b, o_stride_n})
    if (x % vec) return SANA_ERR_ALIGN;
  if (!one_launch(B, N, h, io_dtype)) {
    const size_t at = state_bytes(B, h);
    if (!scratch || scratch_bytes < sana_hip_linattn_scratch_bytes(B, N, h, d, io_dtype)) return SANA_ERR_WORKSPACE;
    if (!aligned16(scratch)) return SANA_ERR_ALIGN;
    float* state = static_cast<float*>(scratch);
    const StatePlan pl = plan_state(B, h, 1, N, io_dtype);
    // Short sequences of few heads: what phase 2 reads again, N / 128 times the partial states, grows with both.  us, three launches
    // / two, three sets of inputs in turn, and in brackets sets that come from HBM: 2 x 1024 x 36 20.6 / 17.7 (23.5 / 21.5), 4 x 640 x 36 21.5 /
    // 18.2 (24.8 / 22.3), 4 x 512 x 36 21.1 / 17.5, 2 x 1024 x 70 26.9 / 26.2 (30.3 / 31.6), 4 x 1024 x 36 27.0 / 26.4 (30.8 / 32.0), beyond the line
    // 4 x 900 x 70 48.3 / 52.1, 8 x 1024 x 36 52.8 / 55.1, 8 x 400 x 70 43.9 / 47.5.  Below it 4 x 400 x 70 loses too, 22.9 / 23.5.
    if (io_dtype == SANA_DT_F32 && N <= WHOLE_TOKENS && pl.nsplit > 1 && pl.nsplit <= 16 && heads * N <= (144 << 10)) {
      float* partial = reinterpret_cast<float*>(static_cast<char*>(scratch) + at);
      hipStream_t st = static_cast<hipStream_t>(stream);
      const bool far = (int64_t)(pl.split_tokens + 64) * stride_n >= (1 << 29);  // beyond the 32-bit offsets
      hipLaunchKernelGGL((far ? linattn_state32_kernel<true, true> : linattn_state32_kernel<true, false>), dim3(pl.nsplit * B * ((h + 3) / 4)), dim3(256), 0, st, static_cast<const float*>(k),
                         static_cast<const float*>(v), partial, nullptr, N, h, 1, pl.nsplit, pl.split_tokens, stride_b, stride_n);
      if (hipGetLastError() != hipSuccess) return SANA_ERR_LAUNCH;
      hipLaunchKernelGGL(linattn_apply32_partials_kernel, dim3((N + 127) / 128 * (unsigned)heads), dim3(320), 0, st,
                         static_cast<const float*>(q), partial, static_cast<float*>(out), N, h, pl.nsplit,
                         (65536u + (N + 127) / 128 - 1) / ((N + 127) / 128), q_stride_b, q_stride_n, o_stride_b, o_stride_n, eps);
      return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
    }
    const int rc = sana_hip_linattn_state(k, v, state, static_cast<char*>(scratch) + at, scratch_bytes - at, B, N, h, d, stride_b,
                                          stride_n, nullptr, 1, N, 0, io_dtype, stream);
    return rc != SANA_OK ? rc
                         : sana_hip_linattn_apply(q, state, out, B, N, h, d, q_stride_b, q_stride_n, o_stride_b, o_stride_n,
                                                  nullptr, 1, N, eps, io_dtype, io_dtype, stream);
  }
  // 16-bit io: up to four workgroups a head while the chip has room for all of them at once.  us, one / so (two, three or four), behind
  // the launch that writes q, k and v: 36 heads x 256 tokens 5.6 / 4.8, 36 x 1024 11.3 / 8.7, 70 x 576 8.2 / 7.2, 70 x 1024 11.0 / 9.0,
  // fp16 72 x 1024 13.8 / 10.1, 128 x 1000 13.5 / 11.4; with more of them than compute units 140 x 1024 12.2 / 14.6, 210 x 972 13.8 / 15.1.
  // (Seven for 36 x 1024: 8.3.)
  const int parts = io_dtype == SANA_DT_F32 ? 1 : heads <= 64 ? 4 : heads <= 85 ? 3 : heads <= 128 ? 2 : 1;
  const dim3 grid((unsigned)(heads * parts));
  hipStream_t s = static_cast<hipStream_t>(stream);
#define SANA_WHOLE(kernel, threads, E, ...)                                                                            \
  hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, s, static_cast<const E*>(q), static_cast<const E*>(k),           \
                     static_cast<const E*>(v), static_cast<E*>(out), N, h, __VA_ARGS__, q_stride_n, stride_b, stride_n, \
                     o_stride_b, o_stride_n, eps)
#define SANA_WHOLE16(R)                                                                                       \
  do {                                                                                                        \
    if (io_dtype == SANA_DT_F16) SANA_WHOLE((linattn_whole16_kernel<F16, R>), 512, uint16_t, q_stride_b);      \
    else SANA_WHOLE((linattn_whole16_kernel<BF16, R>), 512, uint16_t, q_stride_b);                             \
  } while (0)
  if (io_dtype == SANA_DT_F32)
    SANA_WHOLE(linattn_whole32_kernel, WHOLE_TOKENS, float, plan_state(B, h, 1, N, io_dtype).split_tokens, q_stride_b);
  else if (parts == 1) SANA_WHOLE16(1);
  else if (parts == 2) SANA_WHOLE16(2);
  else if (parts == 3) SANA_WHOLE16(3);
  else SANA_WHOLE16(4);
#undef SANA_WHOLE16
#undef SANA_WHOLE
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}
