// What the GEMM kernels share: the epilogue operands and the arithmetic of the epilogues.
#pragma once
#include "common.h"

// No implicit fused multiply-adds in the GEMMs: the epilogues reproduce the stock op chain's roundings (product
// rounded to the io dtype, THEN the sum), and for fp16 -- which has native arithmetic -- the compiler would otherwise
// contract "round(g * y) + r" into one v_fma_f16 and drop the product's rounding.  Wanted fmas are written as fmaf.
#pragma clang fp contract(off)

namespace sana {

// Epilogue operands.  SANA_EPI_GATE_RES: C = res + gate[row / rows_per_gate] * (acc + bias), i.e. the
// gated residual update of the block (x + gate * module(x)), with the reference's three roundings
// (linear output, gate product, residual sum) reproduced in registers.
struct EpiArgs {
  const uint16_t* bias;  // [N] or null
  const uint16_t* gate;  // [*, N] rows gate_stride apart, one row per rows_per_gate rows of C
  const uint16_t* res;   // [M, N] with row stride ldr
  int64_t ldr, gate_stride;
  int rows_per_gate;
  // SANA_EPI_QKV_STATE only: per-token-tile partial states, [B * heads][tiles_per_batch][33 * 32] fp32
  float* part;
  int q_cols, q_pad, heads, tiles_per_batch;  // q_cols = C (columns of the q region), q_pad = C rounded up to the tile
};
#define SANA_EPI_GATE_RES 3
// (not part of the C ABI's epilogue codes) qkv projection of the linear attention with the k / v column tiles
// contracted over their tokens in the epilogue instead of stored: see g8_state_tile
#define SANA_EPI_QKV_STATE 4
// (nor this) K split into ranges, one grid row each: the fp32 accumulators to plane blockIdx.y of C, [M][N] floats each
#define SANA_EPI_PLANES 5

// Virtual concatenation of the A operand along k: columns [t*kc, (t+1)*kc) of the GEMM's A are columns
// [0, kc) of the matrix whose row m is row m + t*stride of the buffer (a convolution over rows as one GEMM,
// without materialising its im2col matrix).  rows = rows of the buffer that exist, counted from A: reads
// past them return zero (the convolution's zero padding on that side).
struct Taps {
  int kc;          // columns per tap, a multiple of the k-tile
  int64_t stride;  // rows between taps
  int64_t rows;
  // split-k launches (SPLIT, never together with taps): grid row z works on k-tiles
  // [z*split_tiles + min(z, split_rem), ...) -- split_tiles of them, one more for z < split_rem
  int split_tiles, split_rem;
  // taps only, may be null: one byte per block of `stride` output rows; non-zero = the LAST tap reads zeros for
  // these rows (a chunk boundary behind the block: the convolution's zero padding inside the buffer)
  const unsigned char* zero_last;
};

// The many-token GEMM (gemm8.hip): C = epilogue(A . W^T) in 256-token x 64*nb-channel tiles, nb = 2, 3 or 4; operands
// 16-bit (f16 or bf16), K % 8 == 0; epilogue SANA_EPI_NONE .. SANA_EPI_GATE_RES, or SANA_EPI_QKV_STATE with nb = 4
// (bf16); taps (bf16, SANA_EPI_GATE_RES, nb = 3 or 4) or null.  Arguments are checked by the caller.
int gemm8_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                 int64_t ldw, int64_t ldc, int epilogue, bool f16, int nb, const Taps* taps, hipStream_t s);

// K split into `ranges` ranges of `tiles` k-tiles (one more in the first `rem`), tiles of 256 x 192: the fp32 sums of range z to plane z of
// `planes`, [M][N] each.  One workgroup a tile and range; M * N * 4 < 2^31.
int gemm8_planes_launch(const uint16_t* a, const uint16_t* w, float* planes, int M, int N, int K, int64_t lda, int64_t ldw, bool f16,
                        int tiles, int rem, int ranges, hipStream_t s);

// The same in tiles of 256 tokens x 288 channels (gemm288.hip); no SANA_EPI_QKV_STATE; rows of W less than 2^21 values apart,
// bias 16-byte aligned (or null).
int gemm288_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                   int64_t ldw, int64_t ldc, int epilogue, bool f16, const Taps* taps, hipStream_t s);

// The GEMM for few tokens (gemm_ring.hip): the same operands and epilogues up to SANA_EPI_GATE_RES (gate not null), in tiles
// of bm tokens x bn channels: 64 x 32, 64 x 64, 64 x 128, 96 x 128,
// 128 x 128, 128 x 160, 192 x 128 or 256 x 128.
// ranges > 1: each output is the sum, in order, of the sums over that many ranges of k-tiles, the bits of the GEMM split over k; `tiles`
// k-tiles each (8 or more), one more in the first `rem`.  64 x 32, 64 x 64, 96 x 128 and 192 x 128 only.
struct KRanges {
  int tiles, rem, ranges;
};
int gemm_ring_launch(const uint16_t* a, const uint16_t* w, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                     int64_t ldw, int64_t ldc, int epilogue, bool f16, int bm, int bn, const KRanges& kr, hipStream_t s);

namespace {

// A wave-uniform value into scalar registers, whatever the compiler thinks of it.
__device__ __forceinline__ int gemm_uniform(int x) {
  int r;
  asm volatile("s_mov_b32 %0, %1" : "=s"(r) : "s"(x));
  return r;
}
__device__ __forceinline__ const uint16_t* gemm_uniform(const uint16_t* x) {
  const uint16_t* r;
  asm volatile("s_mov_b64 %0, %1" : "=s"(r) : "s"(x));
  return r;
}
// LDS accesses and MFMAs of the tile kernels as asm statements: to the compiler an ordinary LDS access may alias the direct
// loads in flight.  The caller waits.
template <int OFF>
__device__ __forceinline__ u32x4_t gemm_lds_read(uint32_t addr) {
  u32x4_t v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
template <int OFF>
__device__ __forceinline__ void gemm_lds_write(uint32_t addr, u32x4_t v) {
  asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(v), "n"(OFF) : "memory");
}
template <int OFF>
__device__ __forceinline__ void gemm_lds_write(uint32_t addr, u32x2_t v) {
  asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(addr), "v"(v), "n"(OFF) : "memory");
}
template <typename T>
__device__ __forceinline__ void gemm_mfma(f32x4_t& c, u32x4_t a, u32x4_t b) {
  if constexpr (is_f16<T>) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
// Workgroup id -> first token and first channel of its tile of bm x bn: XCD x (ids x, x + 8, ..) takes the x-th contiguous
// eighth of the order in groups of `group` token tiles.
__device__ __forceinline__ void gemm_tile_of(int id, int tiles_t, int tiles_c, int group, int bm, int bn, int& m0, int& n0) {
  const int total = tiles_t * tiles_c, xcd = id & 7, local = id >> 3, base = total >> 3, rem = total & 7;
  const int pid = xcd * base + min(xcd, rem) + local;
  const int group_sz = group * tiles_c, gid = pid / group_sz, first_t = gid * group, gt = min(tiles_t - first_t, group);
  m0 = (first_t + (pid % group_sz) % gt) * bm, n0 = ((pid % group_sz) / gt) * bn;
}

// 8 outputs of one row: accumulator (+bias) -> io dtype, per the epilogue kind (everything except
// the gated residual, which needs the row's residual and gate and is applied at store time).
template <int EPI, typename T = BF16>
__device__ __forceinline__ u32x4_t epi_pack8(const float* a, const float* bv) {
  float v[8];
#pragma unroll
  for (int r = 0; r < 8; ++r) v[r] = EPI != SANA_EPI_NONE ? a[r] + bv[r] : a[r];
  u32x4_t o;
  o.x = pk16<T>(v[0], v[1]);
  o.y = pk16<T>(v[2], v[3]);
  o.z = pk16<T>(v[4], v[5]);
  o.w = pk16<T>(v[6], v[7]);
  if (EPI == SANA_EPI_BIAS_SILU) {
    // The reference rounds the linear output to bf16 before the activation.  x * rcp(1 + 2^(-x log2 e)),
    // written stage by stage over the eight values (and pinned that way): one value at a time is a
    // chain of dependent instructions with two slow transcendentals, which a lone wave per SIMD
    // cannot hide.
    float x[8], t[8];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      x[2 * p] = lo16<T>(o[p]);
      x[2 * p + 1] = hi16<T>(o[p]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) t[r] = -1.44269504088896341f * x[r];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) t[r] = __builtin_amdgcn_exp2f(t[r]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) t[r] = 1.0f + t[r];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) t[r] = __builtin_amdgcn_rcpf(t[r]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 8; ++r) x[r] *= t[r];
    __builtin_amdgcn_sched_barrier(0);
    o.x = pk16<T>(x[0], x[1]);
    o.y = pk16<T>(x[2], x[3]);
    o.z = pk16<T>(x[4], x[5]);
    o.w = pk16<T>(x[6], x[7]);
  }
  return o;
}
template <typename T = BF16>
__device__ __forceinline__ uint32_t gate_res2(uint32_t y, uint32_t g, uint32_t r) {
  const float t0 = rnd16<T>(lo16<T>(g) * lo16<T>(y)), t1 = rnd16<T>(hi16<T>(g) * hi16<T>(y));
  return pk16<T>(lo16<T>(r) + t0, hi16<T>(r) + t1);
}
// y: 8 linear outputs (already rounded to bf16), g / r: the gate and residual values of the same 8 columns
template <typename T = BF16>
__device__ __forceinline__ u32x4_t gate_res8v(u32x4_t y, u32x4_t g, u32x4_t r) {
  u32x4_t o;
  o.x = gate_res2<T>(y.x, g.x, r.x);
  o.y = gate_res2<T>(y.y, g.y, r.y);
  o.z = gate_res2<T>(y.z, g.z, r.z);
  o.w = gate_res2<T>(y.w, g.w, r.w);
  return o;
}
// the same with the gate values already unpacked (they are the same for every row a lane handles)
template <typename T = BF16>
__device__ __forceinline__ u32x4_t gate_res8f(u32x4_t y, const float* g, u32x4_t r) {
  u32x4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const uint32_t t = pk16<T>(g[2 * e] * lo16<T>(y[e]), g[2 * e + 1] * hi16<T>(y[e]));  // one convert rounds both
    o[e] = pk16<T>(lo16<T>(r[e]) + lo16<T>(t), hi16<T>(r[e]) + hi16<T>(t));
  }
  return o;
}
// y: 8 linear outputs (already rounded to bf16) of row m, columns n..n+7
template <typename T = BF16>
__device__ __forceinline__ u32x4_t gate_res8(u32x4_t y, const EpiArgs& e, int m, int n) {
  const u32x4_t g = *reinterpret_cast<const u32x4_t*>(e.gate + (int64_t)(m / e.rows_per_gate) * e.gate_stride + n);
  const u32x4_t r = *reinterpret_cast<const u32x4_t*>(e.res + (int64_t)m * e.ldr + n);
  u32x4_t o;
  o.x = gate_res2<T>(y.x, g.x, r.x);
  o.y = gate_res2<T>(y.y, g.y, r.y);
  o.z = gate_res2<T>(y.z, g.z, r.z);
  o.w = gate_res2<T>(y.w, g.w, r.w);
  return o;
}

}  // namespace
}  // namespace sana
