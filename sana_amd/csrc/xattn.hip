// Softmax attention of many queries over a SHORT key set (the block's cross-attention to the text tokens:
// 16384 image tokens x 300 text tokens x 20 heads of 112 at the 4096 px latent), bf16 or f16 in and out.
//
//   out[b, n, h*d + :] = softmax_m(q[b, n, h, :] . k[b, m, h, :] * scale + bias[b, m]) . v[b, m, h, :]
//
// q and out are token-major [B, N, H*d] (what the linear layers on either side read and write: no head
// transposes), k and v are the two halves of the kv projection [B, Nk, 2, H*d].
//
// The key set of one (batch, head) fits LDS whole (Nk <= 320: K as [key][d padded to 32*DK] and V as [key][112]: 151 KB at d = 112), so
// there is no online softmax: a wave takes 16*QT queries, multiplies them with
// all keys (v_mfma_f32_16x16x32_bf16, scores^T = K . Q^T: a lane owns one query and 4 keys of every 16-key tile),
// takes max / exp2 / sum in registers (two cross-lane steps over the four lane groups that share a query), and
// feeds the probabilities straight back as the column operand of out^T = V^T . P^T -- the k index of that
// product is permuted so that the 8 values a lane needs are the ones its own accumulators hold (keys
// 32s + 4g + {0..3} and 32s + 16 + 4g + {0..3} for lane group g), and V is read transposed in that key order (ds_read_b64_tr_b16).
// Few queries (one 512 px image: 64 workgroups of one item) are bound by the staging.  K and V go global -> LDS by direct loads: no
// staging registers, no branch per piece (rows past Nk and pieces past d lie outside the resource: zeros), no transposing writes.
// Through registers, each piece behind a branch of its own and V written transposed, the instructions in front of the last load alone
// took over a microsecond.  us, before / now: 256 queries x 300 keys x 16 heads of 72 9.6 / 8.3 (launch 1.7, staging 3.0, the rest the
// attention), 1024 9.9 / 8.5, 2 x 1024 12.6 / 11.8, 256 x 20 heads of 112 11.8 / 11.1, 1024 13.1 / 12.4, 4680 31.2 / 30.2, 16384 78 / 78; same bits.
// Workgroups are persistent over consecutive (batch, head, query block) items and restage K / V only when the
// (batch, head) changes.  Every K / V fragment read from LDS feeds QT MFMAs.
// Many queries: of an item of 128 queries (8 us at 112 channels) the matrix pipes take 2 us, the vector units 2.6 and the LDS reads, eight
// waves reading all of K and V, 2 - 4; the waves of a unit, in step, overlap little of it.  What a wave need not wait for is requested ahead:
// an item's queries behind the scores of the one before it, and a new head's V, which the scores do not need, behind its K.  us, all in front of
// the scores / so: 256 queries x 300 keys x 16 heads of 72 8.3 / 7.5, 2 x 1024 11.8 / 11.4, 16 x 1024 56 / 49, 1024 x 20 heads of 112 12.4 / 12.1, 4096
// 30.6 / 27.0, 16 x 1024 87 / 76, 16384 79 / 69, 32760 152 / 132.
#include <type_traits>

#include "common.h"

// Query tiles of 16 per wave and pass (every K / V fragment read feeds that many MFMAs).  One measured best: two need either one wave
// per SIMD (nothing hides the LDS latency: 112 us against 75 us at 16384 x 300 x 20 heads of 112) or, the keys in two groups, all
// registers and a few more (92 us against 80).
constexpr int XA_QT = 1;

namespace sana {
namespace {

constexpr int XA_NKP = 320;       // keys an LDS image holds (padded)
constexpr int XA_VCH = 14, XA_VPITCH = 16 * XA_VCH;  // 16-byte pieces / bytes of a V row: 112 channels, and 8 rows cover all banks

// 16-byte-slot swizzles that make 16 consecutive rows of one chunk hit 16 different bank groups
template <int DK>
__device__ __forceinline__ int xa_kkey(int row) {  // K rows of DK*64 bytes
  return DK == 4 ? (row & 15) : DK == 3 ? ((row >> 2) & 3) : DK == 2 ? ((row >> 1) & 7) : ((row >> 2) & 3);
}
// 4 keys x 16 channels of row-major V -> this lane's channel, 4 keys: row i of a group of 16 lanes is addressed by its lanes 4 i .. 4 i + 3
__device__ __forceinline__ u32x2_t xa_read_tr(uint32_t lds) {
  typedef short s16x4_t __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4_t*)(size_t)lds));
}

// n / by of n < 2^31 with magic = (2^32 - 1) / by, which is at most one too small
__device__ __forceinline__ int xa_div(int n, int by, uint32_t magic) {
  const int z = (int)__umulhi((uint32_t)n, magic);
  return n - z * by >= by ? z + 1 : z;
}
// What this wave wrote to LDS is there, and what it reads from there has come; loads from memory stay in flight.
__device__ __forceinline__ void xa_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename T, int DK, int DT, int QT, int NW, int NKT, bool FAR>
__global__ __launch_bounds__(64 * NW) void cross_attn_kernel(const uint16_t* __restrict__ q, const uint16_t* __restrict__ kv,
                                                         const float* __restrict__ bias, uint16_t* __restrict__ out, int B,
                                                         int N, int Nk, int H, int d, int64_t ldq, int64_t ldkv, int64_t ldo,
                                                         int64_t bias_stride, float scale_log2e, int qblocks, int items,
                                                         int items_per_wg, uint32_t qblocks_magic, uint32_t h_magic) {
  asm volatile("" ::"s"(q), "s"(kv), "s"(bias), "s"(B), "s"(N), "s"(Nk), "s"(H), "s"(d), "s"(ldq), "s"(ldkv), "s"(bias_stride), "s"(qblocks),
               "s"(items), "s"(items_per_wg), "s"(qblocks_magic), "s"(h_magic));  // (the arguments in one wait)
  constexpr int KPITCH = DK * 64, KCH = DK * 4;  // bytes / 16-byte chunks per K row
  constexpr int K_BYTES = XA_NKP * KPITCH, V_BYTES = XA_NKP * XA_VPITCH;
  __shared__ __attribute__((aligned(16))) unsigned char smem[K_BYTES + V_BYTES + XA_NKP * 4];
  unsigned char* sk = smem;
  unsigned char* sv = smem + K_BYTES;
  float* sb = reinterpret_cast<float*>(smem + K_BYTES + V_BYTES);  // per key: bias * log2(e), -inf past Nk
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int fr = lane & 15, fg = lane >> 4;

  // ---- Q fragments: column operand, lane -> query fr, k = 32*ks + 8*fg .. +7; requested an item ahead
  u32x4_t qn[QT][DK];
  int bh, b, h, q0;  // of the item requested last
  auto request = [&](int item) {
    bh = xa_div(item, qblocks, qblocks_magic), b = xa_div(bh, H, h_magic), h = bh - b * H;
    q0 = (item - bh * qblocks) * (NW * 16 * QT) + wave * (16 * QT);
    const uint16_t* qbase = q + ((int64_t)b * N) * ldq + (int64_t)h * d;
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const uint16_t* qrow = qbase + (int64_t)min(q0 + 16 * t + fr, N - 1) * ldq;  // (no branch around a load)
#pragma unroll
      for (int ks = 0; ks < DK; ++ks) qn[t][ks] = *reinterpret_cast<const u32x4_t*>(qrow + (32 * ks + 8 * fg < d ? 32 * ks + 8 * fg : 0));
    }
  };
  u32x4_t qf[QT][DK];
  auto take = [&]() {  // (here, not behind the stores or the branches that follow)
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
      for (int ks = 0; ks < DK; ++ks) {
        asm volatile("" : "+v"(qn[t][ks]));
#pragma unroll
        for (int e = 0; e < 4; ++e) qf[t][ks][e] = 32 * ks + 8 * fg < d ? qn[t][ks][e] : 0u;
        asm volatile("" : "+v"(qf[t][ks]));
      }
  };
  const uint32_t sk0 = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)sk + fr * KPITCH;
  uint32_t ka[DK];  // this lane's piece of K row fr, per k-step (rows 16 apart have the same swizzle)
#pragma unroll
  for (int ks = 0; ks < DK; ++ks) ka[ks] = sk0 + (((4 * ks + fg) ^ xa_kkey<DK>(fr)) << 4);

  const int item0 = blockIdx.x * items_per_wg, item1 = min(items, item0 + items_per_wg);
  auto stage = [&](bool first) {  // K and V of b, h
    // the biases first, and K in front of V: the scores are multiplied while V is on its way
    constexpr int NB = (16 * NKT + 64 * NW - 1) / (64 * NW);
    float key_bias[NB];
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(bias + (bias ? (int64_t)b * bias_stride : 0)), 0, bias ? 4 * Nk : 0, 0x00020000);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int m = tid + 64 * NW * i;
      key_bias[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, 4 * m, 0, 0));  // (past Nk, and without biases: 0)
    }
    __builtin_amdgcn_sched_barrier(0);
    auto older = [&]() {  // the biases and the first item's queries, which are older than K, have landed (the compiler, too, knows it in here)
#pragma unroll
      for (int i = 0; i < NB; ++i) asm volatile("" : "+v"(key_bias[i]));
      if (first) {
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
          for (int ks = 0; ks < DK; ++ks) asm volatile("" : "+v"(qn[t][ks]));
      }
    };
    const uint16_t* kbase = kv + (int64_t)b * Nk * ldkv + (int64_t)h * d;
    const uint16_t* vbase = kbase + (int64_t)H * d;
    // Rows past Nk and pieces past d lie outside the resources: zeros.  (key tiles past NKT are not read)
    constexpr int NT = 64 * NW, KEYS = 16 * NKT;
    constexpr uint32_t kOut = 0x80000000u;
    if constexpr (!FAR) {
      const uint32_t ld2 = 2 * (uint32_t)ldkv;
      const int span = (int)((uint32_t)(Nk - 1) * ld2 + 2 * d);
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(kbase), 0, span, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(vbase), 0, span, 0x00020000);
      auto load = [&](const __amdgpu_buffer_rsrc_t& r, unsigned char* dst, uint32_t off) {
        const int o = (int)off;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)dst, 16, o, 0, 0, 0);
      };
      // K: KI load instructions of 1 KB are 16 (12 pieces a row) or 4 rows (16 pieces); 16 rows and 4 waves repeat the swizzle
      constexpr int KI = KCH == 16 ? 1 : KCH / 4, KR = 64 * KI / KCH;
      static_assert(NW % 4 == 0 && (KR * NW) % 16 == 0 && KEYS % KR == 0, "");
      uint32_t ko[KI];
#pragma unroll
      for (int j = 0; j < KI; ++j) {
        const int l = 64 * j + lane, row = l / KCH, c = (l - row * KCH) ^ xa_kkey<DK>(KR * wave + row);
        ko[j] = 8 * c < d ? (uint32_t)(KR * wave + row) * ld2 + 16 * c : kOut;
      }
#pragma unroll
      for (int i = 0; i < (KEYS / KR + NW - 1) / NW; ++i) {
        const int g = i * NW + wave;
        if (i == KEYS / KR / NW && g >= KEYS / KR) break;  // uniform
#pragma unroll
        for (int j = 0; j < KI; ++j) load(rk, sk + (g * KI + j) * 1024, ko[j] + (uint32_t)(KR * NW * i) * ld2);
      }
      // V: 7 instructions are 32 rows
      uint32_t vo[7];
#pragma unroll
      for (int j = 0; j < 7; ++j) {
        const int l = 64 * j + lane, row = l / XA_VCH, c = l - row * XA_VCH;
        vo[j] = 8 * c < d ? (uint32_t)(32 * wave + row) * ld2 + 16 * c : kOut;
      }
#pragma unroll
      for (int i = 0; i < (KEYS / 32 + NW - 1) / NW; ++i) {
        const int g = i * NW + wave;
        if (i == KEYS / 32 / NW && g >= KEYS / 32) break;  // uniform
#pragma unroll
        for (int j = 0; j < 7; ++j) load(rv, sv + (g * 7 + j) * 1024, vo[j] + (uint32_t)(32 * NW * i) * ld2);
      }
      // K has landed (and what was requested before it); V is waited for behind the scores
      constexpr int VI = KEYS / 32 / NW * 7;
      if (wave < KEYS / 32 % NW) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VI + 7) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(VI) : "memory");
      older();
    } else {  // rows too far apart for 32-bit offsets
      older();
#pragma unroll 1
      for (int i = tid; i < KEYS * KCH; i += NT) {
        const int row = i / KCH, c = i - row * KCH;
        u32x4_t x = {0u, 0u, 0u, 0u};
        if (row < Nk && 8 * c < d) x = *reinterpret_cast<const u32x4_t*>(kbase + (int64_t)row * ldkv + 8 * c);
        *reinterpret_cast<u32x4_t*>(sk + row * KPITCH + ((c ^ xa_kkey<DK>(row)) << 4)) = x;
      }
#pragma unroll 1
      for (int i = tid; i < KEYS * XA_VCH; i += NT) {
        const int row = i / XA_VCH, c = i - row * XA_VCH;
        u32x4_t x = {0u, 0u, 0u, 0u};
        if (row < Nk && 8 * c < d) x = *reinterpret_cast<const u32x4_t*>(vbase + (int64_t)row * ldkv + 8 * c);
        *reinterpret_cast<u32x4_t*>(sv + 16 * i) = x;
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int m = tid + NT * i;
      if (m < KEYS) sb[m] = m < Nk ? key_bias[i] * 1.44269504088896341f : -INFINITY;
    }
    if (first) take();
    xa_barrier();
  };
  request(item0);
  stage(true);
  int staged = -1;
  for (int item = item0; item < item1; ++item) {
    const bool fresh = bh != staged;  // uniform
    if (fresh && item > item0) {
      xa_barrier();  // everyone is done with the previous head's K / V
      stage(false);
    }
    staged = bh;
    const int first_query = q0;
    uint16_t* obase = out + ((int64_t)b * N) * ldo + (int64_t)h * d;
    auto scores_done = [&]() {
      if (fresh) {  // V has landed, everyone's
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        xa_barrier();
      }
      request(min(item + 1, item1 - 1));
      __builtin_amdgcn_sched_barrier(0);
    };
    if (first_query >= N) {
      scores_done();
      take();
      continue;  // (no barrier below)
    }
    // Keys in NG groups, one after the other (scores, softmax, product; the first group's scores are gone before the second's come:
    // 0.1 - 0.7 us less than all scores first).  f16: two, each with a maximum of its own, combined in fp32 at the end, and the sum
    // is over the rounded probabilities.  A group's largest probability is 1 and has no rounding error; the stock fused kernels,
    // which keep a running maximum over blocks of keys, have that in every block.  Error against 64 bits, one maximum / two /
    // stock, e-4: 300 keys x 72 2.75 / 2.69 / 2.68, x 112 2.76 / 2.69 / 2.69, 10 keys 2.43 / 2.39 / 2.43.
    constexpr int NG = is_f16<T> ? 2 : 1, G0 = NG == 2 ? 2 * ((NKT + 3) / 4) : NKT;  // key tiles of the first group
    float mx[QT][NG], sum[QT][NG];
    f32x4_t oc[NG][QT][DT];
    auto group = [&](auto g_c) {
      constexpr int g = decltype(g_c)::value, k0 = g * G0, k1 = g + 1 < NG ? G0 : NKT;
      // ---- scores^T = K . Q^T: sc[t][kt][r] = query 16t + fr, key 16*(k0 + kt) + 4*fg + r
      f32x4_t sc[QT][G0];
#pragma unroll
      for (int kt = 0; kt < G0; ++kt)
#pragma unroll
        for (int t = 0; t < QT; ++t) sc[t][kt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      // key tiles in pairs (two independent accumulator chains), the next pair's fragments requested before this pair's MFMAs
      u32x4_t kf[2][2][DK];
      // (asm reads: to the compiler an ordinary one may alias the loads of V in flight)
      auto load_k = [&](int buf, int kt) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int ks = 0; ks < DK; ++ks) {
            const uint32_t at = ka[ks] + (kt + j < 10 ? 0 : 160 * KPITCH);  // (an offset has 16 bits)
            asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(kf[buf][j][ks]) : "v"(at), "n"((kt + j) % 10 * 16 * KPITCH));
          }
      };
      auto landed = [&](int buf, bool more) {
        if (more) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * DK) : "memory");
        else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int ks = 0; ks < DK; ++ks) asm volatile("" : "+v"(kf[buf][j][ks])::"memory");
      };
      load_k(0, k0);
#pragma unroll
      for (int kt = k0; kt < k1; kt += 2) {
        const int buf = (kt - k0) / 2 & 1;
        if (kt + 2 < k1) load_k(buf ^ 1, kt + 2);
        landed(buf, kt + 2 < k1);
#pragma unroll
        for (int ks = 0; ks < DK; ++ks)
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int t = 0; t < QT; ++t)
              sc[t][kt - k0 + j] = mfma_16x16x32<T>(kf[buf][j][ks], qf[t][ks], sc[t][kt - k0 + j]);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (g == 0) scores_done();
      // ---- softmax over the group's keys (log2 domain), probabilities packed to 16 bits
      u32x2_t pk[QT][G0];
#pragma unroll
      for (int t = 0; t < QT; ++t) {
        float m = -INFINITY, l = 0.f;
#pragma unroll
        for (int kt = k0; kt < k1; ++kt) {
          const f32x4_t kb = *reinterpret_cast<const f32x4_t*>(sb + 16 * kt + 4 * fg);
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            sc[t][kt - k0][r] = fmaf(sc[t][kt - k0][r], scale_log2e, kb[r]);
            m = fmaxf(m, sc[t][kt - k0][r]);
          }
        }
        m = fmaxf(m, __shfl_xor(m, 16));
        m = fmaxf(m, __shfl_xor(m, 32));
        if (NG == 2) m = fmaxf(m, -3.0e38f);  // a group without keys: -inf - -inf
#pragma unroll
        for (int kt = 0; kt < k1 - k0; ++kt) {
          float p[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            p[r] = __builtin_amdgcn_exp2f(sc[t][kt][r] - m);
            if constexpr (is_f16<T>) p[r] = (float)(_Float16)p[r];
            l += p[r];
          }
          pk[t][kt] = u32x2_t{pk16<T>(p[0], p[1]), pk16<T>(p[2], p[3])};
        }
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        mx[t][g] = m, sum[t][g] = l;
      }
      // ---- out^T = V^T . P^T: oc[t][dt][r] = query 16t + fr, channel 16*dt + 4*fg + r
#pragma unroll
      for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) oc[g][t][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      u32x4_t vf[2][DT];
      const uint32_t vrow = (uint32_t)(size_t)(__attribute__((address_space(3))) const unsigned char*)sv + (4 * fg + (fr >> 2)) * XA_VPITCH + 8 * (fr & 3);
      auto load_v = [&](int buf, int s) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const u32x2_t lo = xa_read_tr(vrow + 32 * s * XA_VPITCH + 32 * dt), hi = xa_read_tr(vrow + (32 * s + 16) * XA_VPITCH + 32 * dt);
          vf[buf][dt] = u32x4_t{lo.x, lo.y, hi.x, hi.y};
        }
      };
      load_v(0, k0 / 2);
#pragma unroll
      for (int s = 0; s < (k1 - k0) / 2; ++s) {
        if (s + 1 < (k1 - k0) / 2) load_v((s + 1) & 1, k0 / 2 + s + 1);
        u32x4_t pf[QT];
#pragma unroll
        for (int t = 0; t < QT; ++t)
          pf[t] = u32x4_t{pk[t][2 * s].x, pk[t][2 * s].y, pk[t][2 * s + 1].x, pk[t][2 * s + 1].y};
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int t = 0; t < QT; ++t) oc[g][t][dt] = mfma_16x16x32<T>(vf[s & 1][dt], pf[t], oc[g][t][dt]);
      }
    };
    group(std::integral_constant<int, 0>{});
    if constexpr (NG == 2) group(std::integral_constant<int, 1>{});
    float factor[QT][NG];
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      if constexpr (NG == 2) {
        const float m = fmaxf(mx[t][0], mx[t][1]);
        const float f0 = __builtin_amdgcn_exp2f(mx[t][0] - m), f1 = __builtin_amdgcn_exp2f(mx[t][1] - m);
        const float inv = 1.0f / fmaf(sum[t][0], f0, sum[t][1] * f1);
        factor[t][0] = f0 * inv, factor[t][1] = f1 * inv;
      } else {
        factor[t][0] = 1.0f / sum[t][0];
      }
    }
    take();  // (in front of the stores, which it need not wait for)
    // ---- normalise and store: a lane holds 4 consecutive channels of its query per channel tile
#pragma unroll
    for (int t = 0; t < QT; ++t) {
      const int qi = first_query + 16 * t + fr;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const int c0 = 16 * dt + 4 * fg;
        if (qi < N && c0 < d) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r)
            v[r] = NG == 2 ? fmaf(oc[NG - 1][t][dt][r], factor[t][NG - 1], oc[0][t][dt][r] * factor[t][0]) : oc[0][t][dt][r] * factor[t][0];
          const u32x2_t o = {pk16<T>(v[0], v[1]), pk16<T>(v[2], v[3])};
          *reinterpret_cast<u32x2_t*>(obase + (int64_t)qi * ldo + c0) = o;
        }
      }
    }
  }
}

template <typename T, int DK, int DT, int QT, int NW, int NKT, bool FAR = false>
int launch_xa(const uint16_t* q, const uint16_t* kv, const float* bias, uint16_t* out, int B, int N, int Nk, int H, int d,
              int64_t ldq, int64_t ldkv, int64_t ldo, int64_t bias_stride, float scale, hipStream_t s) {
  const int qblocks = (N + NW * 16 * QT - 1) / (NW * 16 * QT);
  const int64_t items64 = (int64_t)B * H * qblocks;
  if (items64 > 0x7fffffff) return SANA_ERR_SHAPE;
  const int items = (int)items64, cus = 256;
  const int ipw = (items + cus - 1) / cus;
  const int grid = (items + ipw - 1) / ipw;
  hipLaunchKernelGGL((cross_attn_kernel<T, DK, DT, QT, NW, NKT, FAR>), dim3((unsigned)grid), dim3(64 * NW), 0, s, q, kv, bias, out, B, N, Nk, H, d,
                     ldq, ldkv, ldo, bias_stride, scale * 1.44269504088896341f, qblocks, items, ipw, 0xffffffffu / (uint32_t)qblocks, 0xffffffffu / (uint32_t)H);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

template <typename T>
int cross_attention(const void* q, const void* kv, const float* key_bias, void* out, int B, int N, int Nk, int H, int d,
                    int64_t ldq, int64_t ldkv, int64_t ldo, int64_t bias_stride, float scale, void* stream) {
  if (!q || !kv || !out || B <= 0 || N <= 0 || Nk <= 0 || H <= 0 || d <= 0) return SANA_ERR_ARG;
  if (Nk > XA_NKP || d % 8 || d > 112 || d <= 64) return SANA_ERR_SHAPE;  // LDS: K + V^T of one head at d <= 112
  if (ldq < (int64_t)H * d || ldkv < 2 * (int64_t)H * d || ldo < (int64_t)H * d || (key_bias && bias_stride < Nk))
    return SANA_ERR_ARG;
  if (ldq % 8 || ldkv % 8 || ldo % 4 || !aligned16(q) || !aligned16(kv) || (reinterpret_cast<uintptr_t>(out) & 7u))
    return SANA_ERR_ALIGN;
  const uint16_t* qp = static_cast<const uint16_t*>(q);
  const uint16_t* kp = static_cast<const uint16_t*>(kv);
  uint16_t* op = static_cast<uint16_t*>(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define SANA_XA_GO(DK, DT, NW, NKT) \
  launch_xa<T, DK, DT, XA_QT, NW, NKT>(qp, kp, key_bias, op, B, N, Nk, H, d, ldq, ldkv, ldo, bias_stride, scale, s)
  // Waves per workgroup: eight, two per SIMD (up to 220 registers).  Four, half the queries, at up to 96 channels a head where these
  // workgroups have a compute unit each: a unit then reads K and V from LDS for four waves.  us, 8 / 4 waves: 300 keys, 150 queries x
  // 16 heads of 72 10.6 / 9.8, 512 11.5 / 10.1, 1024 11.7 / 10.5, f16 12.6 / 10.6, 77 keys 6.9 / 6.3; in two rounds 2 x 1024 13.8 / 16.2.
  // 112 channels a head: 600 x 20 heads 13.1 / 12.7, 2 x 300 13.6 / 14.0 (the staging is more of it).
  // Nor with the keys and values of 64 heads and more, each of which two workgroups then stage instead of one: 4 x 256 x 16 heads
  // 12.7 / 13.8, 160 keys 8.9 / 9.2, f16 13.5 / 14.0; but 77 keys 8.1 / 7.8.
  const bool restaged = (int64_t)B * H >= 64 && N > 64 * XA_QT && Nk > (is_f16<T> ? 256 : 128);
  const bool few = d <= 96 && !restaged && (int64_t)B * H * ((N + 64 * XA_QT - 1) / (64 * XA_QT)) <= 256;
  if (ldkv >= (1 << 21))  // rows of K and V too far apart for 32-bit offsets: staged through registers (the same bits)
    return Nk > 160 ? launch_xa<T, 4, 7, XA_QT, 8, 20, true>(qp, kp, key_bias, op, B, N, Nk, H, d, ldq, ldkv, ldo, bias_stride, scale, s)
                    : launch_xa<T, 4, 7, XA_QT, 8, 10, true>(qp, kp, key_bias, op, B, N, Nk, H, d, ldq, ldkv, ldo, bias_stride, scale, s);
  // key tiles of 16 that are multiplied: all 20, or 10 for up to 160 keys (tiles past Nk hold zeros and -inf)
  if (d > 96) return Nk > 160 ? SANA_XA_GO(4, 7, 8, 20) : SANA_XA_GO(4, 7, 8, 10);
  // (the product with V in tiles of 16 channels: five up to 80)
  if (few && d <= 80) return Nk > 160 ? SANA_XA_GO(3, 5, 4, 20) : SANA_XA_GO(3, 5, 4, 10);
  if (few) return Nk > 160 ? SANA_XA_GO(3, 6, 4, 20) : SANA_XA_GO(3, 6, 4, 10);
  if (d <= 80) return Nk > 160 ? SANA_XA_GO(3, 5, 8, 20) : SANA_XA_GO(3, 5, 8, 10);
  return Nk > 160 ? SANA_XA_GO(3, 6, 8, 20) : SANA_XA_GO(3, 6, 8, 10);
#undef SANA_XA_GO
}

// (1 - mask) * -10000, the additive key bias of a prompt mask.  Bound by its launch (a few hundred values); as three
// elementwise operators it was 18 us a block.
template <typename E>
__global__ __launch_bounds__(256) void key_bias_kernel(const E* __restrict__ mask, float* __restrict__ bias, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) bias[i] = (1.0f - (float)mask[i]) * -10000.0f;
}

}  // namespace
}  // namespace sana

using namespace sana;

#define SANA_API extern "C" __attribute__((visibility("default")))

SANA_API int sana_hip_cross_attention(const void* q, const void* kv, const float* key_bias, void* out, int B, int N, int Nk,
                                      int H, int d, int64_t ldq, int64_t ldkv, int64_t ldo, int64_t bias_stride,
                                      float scale, void* stream) {
  return cross_attention<BF16>(q, kv, key_bias, out, B, N, Nk, H, d, ldq, ldkv, ldo, bias_stride, scale, stream);
}

SANA_API int sana_hip_cross_attention_f16(const void* q, const void* kv, const float* key_bias, void* out, int B, int N,
                                          int Nk, int H, int d, int64_t ldq, int64_t ldkv, int64_t ldo,
                                          int64_t bias_stride, float scale, void* stream) {
  return cross_attention<F16>(q, kv, key_bias, out, B, N, Nk, H, d, ldq, ldkv, ldo, bias_stride, scale, stream);
}

SANA_API int sana_hip_key_bias(const void* mask, float* bias, int64_t n, int mask_type, void* stream) {
  if (!mask || !bias || n <= 0) return SANA_ERR_ARG;
  if ((n + 255) / 256 > 0x7fffffff) return SANA_ERR_SHAPE;
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
#define SANA_KB(E) hipLaunchKernelGGL(key_bias_kernel<E>, grid, block, 0, s, static_cast<const E*>(mask), bias, n)
  switch (mask_type) {
    case SANA_MASK_U8: SANA_KB(uint8_t); break;
    case SANA_MASK_I16: SANA_KB(int16_t); break;
    case SANA_MASK_I32: SANA_KB(int32_t); break;
    case SANA_MASK_I64: SANA_KB(int64_t); break;
    case SANA_MASK_F32: SANA_KB(float); break;
    case SANA_MASK_F16: SANA_KB(_Float16); break;
    case SANA_MASK_BF16: SANA_KB(__bf16); break;
    default: return SANA_ERR_DTYPE;
  }
#undef SANA_KB
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}
