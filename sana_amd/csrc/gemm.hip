// bf16 MFMA GEMM for gfx950:  C[M][N] = epilogue(A[M][K] . W[N][K]^T), with an int8-weight (W8A16) variant
// dequantised on the way into LDS: the C entry points, the choice of a kernel by shape, and the kernels for int8
// weights, which the rest of this comment describes.  16-bit GEMMs run the kernels of gemm8.h and gemm288.h (many tokens, and k
// split into ranges) and gemm_ring.h (few).
//
// Both operands are K-contiguous, which is exactly the MFMA operand layout (a
// lane holds 8 consecutive k of one row), so nothing is transposed.  The MFMA
// "row" operand is the WEIGHT tile and the "column" operand the ACTIVATION
// tile: a lane of the accumulator then owns one token (column) and a few output
// channels (rows).  Weight rows are permuted on their way into LDS so that the
// channels a lane owns are contiguous in C (the pipelined kernel: 8*NI channels
// from 2*NI MFMA tiles of 16; the compiler-scheduled one: 16 channels per 32x32 tile).
//
// Workgroup tile 256 (tokens) x 256 (channels) x 64 (k), four waves in 2x2,
// each 128x128 (256 fp32 accumulators).  The pipelined kernel multiplies with
// v_mfma_f32_16x16x32_bf16: on this chip the matrix pipes are power-limited, and
// with random bf16 operands a loop of nothing but 32x32x16 MFMAs settles at 1.64 GHz
// (0.69 of the 2.5 PFLOP/s peak) where the same flops as 16x16x32 run at 1.9-2.0 GHz.
// LDS is double buffered (2 x 64 KB); 16-byte chunks are XOR-swizzled by (row / 2) % 8 so
// that ds_read_b128 / ds_write_b128 are bank-conflict free.  Workgroup ids are
// remapped so that each XCD (own L2) works on a compact group of tiles.
#include <algorithm>

#include "gemm_common.h"

namespace sana {
namespace {

constexpr int BT = 256;   // tokens (rows of A / C) per workgroup
constexpr int BK = 64;
constexpr int ROW_BYTES = BK * 2;            // 128
constexpr int TILE_BYTES = 256 * ROW_BYTES;  // 32 KB per operand per stage

// LDS reads of 16 bytes are served 16 lanes (256 bytes = all 64 banks) per clock, so 16 consecutive
// rows of one k chunk must land in 16 different 16-byte bank groups: rows alternate between the two
// halves of the bank space (128-byte rows), and the chunk index is XORed with (row / 2) % 8.
__device__ __forceinline__ int swz_key(int row) { return (row >> 1) & 7; }
__device__ __forceinline__ int swz(int row, int chunk) { return row * ROW_BYTES + ((chunk ^ swz_key(row)) << 4); }

// LDS row of weight row n (within the 256-row tile): permute inside each 32-row block
__device__ __forceinline__ int wrow_to_lds(int n) {
  const int blk = n & ~31, r = n & 31;
  return blk + 8 * ((r >> 2) & 3) + 4 * (r >> 4) + (r & 3);
}

// The GEMMs exist for the two 16-bit io dtypes, T = BF16 (also the int8-weight and the fused-state variants) or F16:
// same loops, the MFMA of the dtype, and the dtype's own conversions in the epilogues (one v_cvt_pk_bf16_f32 per pair
// for bf16; two conversions and a pack for f16, which has no packed round-to-nearest conversion).
// acc += W fragment (16 channels x 32 k) . A fragment (32 k x 16 tokens), as an asm statement so that the
// accumulator is one AGPR quad in and out: given the builtin, whose destination may differ from its addend, the
// register allocator rotates accumulators through other registers across the loop edge (dozens of copies and
// their wait states per k-tile in some instances).
template <typename T>
__device__ __forceinline__ void mfma_acc(f32x4_t& c, u32x4_t a, u32x4_t b) {
  if constexpr (is_f16<T>) asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
  else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

__device__ __forceinline__ uint32_t dequant2(uint32_t q4, int which, float s, float off) {
  // two int8 (bytes 2*which, 2*which+1 of q4, already biased by +128) -> packed bf16(q*s)
  // (the compiler turns these byte extracts into v_cvt_f32_ubyteN)
  const float f0 = (float)((q4 >> (16 * which)) & 0xffu);
  const float f1 = (float)((q4 >> (16 * which + 8)) & 0xffu);
  // (q+128)*s - 128*s == q*s exactly before the single fp32 rounding
  return pack_bf16(fmaf(f0, s, off), fmaf(f1, s, off));
}

// int8 weight [N][K] + per-row scale -> bf16 [N][K], with the rounding of dequant2: the expansion the GEMM's
// int8 path performs on its way to LDS, as a streaming kernel of its own.  A wave takes 512 values of a row, a lane 8 (a store instruction is
// 1 KB in a row): no division, whole sectors.  HBM bound; short rows by latency, for which a wave is to have one round trip: with a whole row a wave, six
// pieces a lane requested at once, it was the longer way for narrow weights.  us, 16 values a thread with a 64-bit division for its row / a row a wave / so:
// 504 x 2208 2.8 / 3.4 / 2.6, 1152 x 1152 2.9 / 3.2 / 2.7, 1152 x 2880 4.5 / 5.1 / 4.0, 2240 x 5600 11.2 / 11.9 / 10.0, 5760 x 1152 7.1 / 6.5 / 6.8, 6720 x 2240 12.9 /
// 11.2 / 11.2, 11200 x 2240 19.6 / 17.9 / 16.3.
// grid: ceil(K / 512), rows by four in y and, 2^15 of them each, z; block 256.
__global__ __launch_bounds__(256) void dequant_w8_kernel(const int8_t* __restrict__ wq, const float* __restrict__ scale,
                                                         uint16_t* __restrict__ out, int N, int K, int64_t ldw,
                                                         int64_t ldo) {
  const uint32_t n = (blockIdx.z << 15 | blockIdx.y) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t p = blockIdx.x * 64 + (threadIdx.x & 63);
  if (n >= (uint32_t)N || p >= (uint32_t)K >> 3) return;
  const u32x2_t q = *reinterpret_cast<const u32x2_t*>(wq + n * ldw + 8 * (int64_t)p);
  const float s = scale[n], off = -128.f * s;
  const uint32_t x = q.x ^ 0x80808080u, y = q.y ^ 0x80808080u;
  *reinterpret_cast<u32x4_t*>(out + n * ldo + 8 * (int64_t)p) =
      u32x4_t{dequant2(x, 0, s, off), dequant2(x, 1, s, off), dequant2(y, 0, s, off), dequant2(y, 1, s, off)};
}

// Compiler-scheduled kernel for int8 weights, any K % 16 == 0.  Workgroup tile 64*TT tokens x 64*TC channels,
// four waves in 2x2, each TT x TC MFMA tiles.  <4, 4>: the 256 x 256 tile of the pipelined kernel, for the K
// values that one does not take.  <2, 2>: 128 x 128 with 64 accumulators and 64 KB of LDS, two workgroups per
// CU -- a quarter of the work per k-tile, so a much shorter latency chain for shapes whose 256-wide grid would
// leave the chip mostly idle (a few hundred to a few thousand tokens); its k-tiles are requested three ahead
// (three register sets in rotation), because with so little math per k-tile the chain is otherwise one global
// load latency per k-tile.  Every output sums its k products in the same order in all of these kernels, so
// they agree bit for bit.
template <int EPI, int TT, int TC>
__global__ __launch_bounds__(256, (TT * TC <= 4 ? 2 : 1)) void gemm_w8_kernel(const uint16_t* __restrict__ A,
                                                   const int8_t* __restrict__ Wq, const float* __restrict__ scale,
                                                   const EpiArgs ep, uint16_t* __restrict__ C,
                                                   int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc,
                                                   int tiles_t, int tiles_c) {
  typedef BF16 T;
  constexpr int BT = 64 * TT, BC = 64 * TC;              // shadow the file-scope 256 x 256
  constexpr int A_BYTES = BT * ROW_BYTES, STAGE_BYTES = (BT + BC) * ROW_BYTES;
  __shared__ __attribute__((aligned(16))) unsigned char smem[2 * STAGE_BYTES];  // [stage][A | W]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;

  // ---- workgroup -> tile, XCD aware: ids are dealt round-robin to the 8 XCDs, so
  // give XCD x the x-th contiguous eighth of the (grouped) tile order.
  const int total = tiles_t * tiles_c;
  int pid = blockIdx.x;
  {
    const int xcd = pid & 7, local = pid >> 3;
    const int base = total >> 3, rem = total & 7;
    pid = xcd * base + min(xcd, rem) + local;  // ids with id%8 == x: base + (x < rem) of them
  }
  constexpr int GROUP = 8;  // token tiles per group
  const int group_sz = GROUP * tiles_c;
  const int gid = pid / group_sz;
  const int first_t = gid * GROUP;
  const int gt = min(tiles_t - first_t, GROUP);
  const int tile_t = first_t + (pid % group_sz) % gt;
  const int tile_c = (pid % group_sz) / gt;
  const int m0 = tile_t * BT, n0 = tile_c * BC;

  // ---- global -> register staging
  // A tile: BT rows x 8 chunks(16 B); thread -> chunk tid%8, rows tid/8 + 32*i
  const int a_chunk = tid & 7, a_row = tid >> 3;
  constexpr int NA = 2 * TT, NW = TC;
  constexpr int DEPTH = TT * TC <= 4 ? 3 : 1;  // k-tiles in flight in registers
  u32x4_t ra[DEPTH][NA];
  // W tile: BC rows x 4 chunks of 16 int8; thread -> chunk tid%4, rows tid/4 + 64*i
  u32x4_t rw[DEPTH][NW];
  const int w_chunk = tid & 3, w_row = tid >> 2;

  // Operand tiles are read with buffer loads, one resource per operand over the tile's valid rows (ending with
  // the last valid row's K-th element): rows past M / N fall outside it and read as zero, and a k chunk past K
  // gets an offset outside it -- no branches around the loads, so that several k-tiles can stay in flight.
  // (The whole offset is the vector offset: only that one is range-checked.)
  const int a_last = min(BT, M - m0) - 1, w_last = min(BC, N - n0) - 1;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(A + (int64_t)m0 * lda), 0, (int)(((int64_t)a_last * lda + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(Wq + (int64_t)n0 * ldw), 0, (int)((int64_t)w_last * ldw + K), 0x00020000);
  const int idle_off = (int)0x80000000u;
  const int voff_a = (a_row * (int)lda + a_chunk * 8) * 2, step_a = 32 * (int)lda * 2;
  const int voff_w = w_row * (int)ldw + w_chunk * 16, step_w = 64 * (int)ldw;
  auto load_tile = [&](int set, int k0) {  // k chunks past K load zeros
    const int off_a = k0 + a_chunk * 8 < K ? voff_a + k0 * 2 : idle_off;
    const int off_w = k0 + w_chunk * 16 < K ? voff_w + k0 : idle_off;
#pragma unroll
    for (int i = 0; i < NA; ++i)
      ra[set][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, off_a + i * step_a, 0, 0));
#pragma unroll
    for (int i = 0; i < NW; ++i)
      rw[set][i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, off_w + i * step_w, 0, 0));
  };
  float wscale[TC], woff[TC];
#pragma unroll
  for (int i = 0; i < TC; ++i) {
    const int n = n0 + w_row + 64 * i;
    wscale[i] = n < N ? scale[n] : 0.f;
    woff[i] = -128.f * wscale[i];
  }
  auto store_tile = [&](int set, int stage) {
    unsigned char* sa = smem + stage * STAGE_BYTES;
    unsigned char* sw = sa + A_BYTES;
#pragma unroll
    for (int i = 0; i < NA; ++i) *reinterpret_cast<u32x4_t*>(sa + swz(a_row + 32 * i, a_chunk)) = ra[set][i];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const int lrow = wrow_to_lds(w_row + 64 * i);
      u32x4_t q = rw[set][i];
      q.x ^= 0x80808080u;
      q.y ^= 0x80808080u;
      q.z ^= 0x80808080u;
      q.w ^= 0x80808080u;
      u32x4_t lo, hi;
      lo.x = dequant2(q.x, 0, wscale[i], woff[i]);
      lo.y = dequant2(q.x, 1, wscale[i], woff[i]);
      lo.z = dequant2(q.y, 0, wscale[i], woff[i]);
      lo.w = dequant2(q.y, 1, wscale[i], woff[i]);
      hi.x = dequant2(q.z, 0, wscale[i], woff[i]);
      hi.y = dequant2(q.z, 1, wscale[i], woff[i]);
      hi.z = dequant2(q.w, 0, wscale[i], woff[i]);
      hi.w = dequant2(q.w, 1, wscale[i], woff[i]);
      *reinterpret_cast<u32x4_t*>(sw + swz(lrow, 2 * w_chunk)) = lo;
      *reinterpret_cast<u32x4_t*>(sw + swz(lrow, 2 * w_chunk + 1)) = hi;
    }
  };

  // ---- MFMA tiling: wave (wc, wt) owns channels [wc*32*TC, +32*TC) x tokens [wt*32*TT, +32*TT)
  const int wc = wave & 1, wt = wave >> 1;
  const int fr = lane & 31, fg = lane >> 5;
  f32x16_t acc[TC][TT];
#pragma unroll
  for (int i = 0; i < TC; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  const int KT = (K + BK - 1) / BK;
#pragma unroll
  for (int d = 0; d < DEPTH; ++d) load_tile(d, d * BK);
  store_tile(0, 0);
  __syncthreads();
  // k-tile kt is multiplied from LDS stage kt % 2 while register set kt % DEPTH (which held it) is refilled with
  // k-tile kt + DEPTH and set (kt + 1) % DEPTH goes to the other stage; unrolled by DEPTH so the set is static.
  // The loop runs whole rounds of DEPTH: k-tiles past K are all zeros (they add nothing), and a body without
  // exits keeps the compiler's count of outstanding loads exact.
  for (int kt0 = 0; kt0 < KT; kt0 += DEPTH) {
#pragma unroll
   for (int d = 0; d < DEPTH; ++d) {
    const int kt = kt0 + d;
    const int cur = kt & 1;
    load_tile(d, (kt + DEPTH) * BK);
    const unsigned char* sa = smem + cur * STAGE_BYTES;
    const unsigned char* sw = sa + A_BYTES;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      u32x4_t fw[TC], fa[TT];
#pragma unroll
      for (int i = 0; i < TC; ++i)
        fw[i] = *reinterpret_cast<const u32x4_t*>(sw + swz(wc * 32 * TC + 32 * i + fr, 2 * ks + fg));
#pragma unroll
      for (int j = 0; j < TT; ++j)
        fa[j] = *reinterpret_cast<const u32x4_t*>(sa + swz(wt * 32 * TT + 32 * j + fr, 2 * ks + fg));
#pragma unroll
      for (int i = 0; i < TC; ++i)
#pragma unroll
        for (int j = 0; j < TT; ++j)
          acc[i][j] = mfma_32x32x16<T>(fw[i], fa[j], acc[i][j]);
    }
    store_tile((d + 1) % DEPTH, cur ^ 1);
    __syncthreads();
   }
  }

  // ---- epilogue.  acc[i][j][r]: token m0 + wt*32*TT + 32*j + lane%32,
  // channel n0 + wc*32*TC + 32*i + 16*(lane/32) + r
  constexpr bool HAS_BIAS = EPI != SANA_EPI_NONE;
#pragma unroll
  for (int i = 0; i < TC; ++i) {
    const int n = n0 + wc * 32 * TC + 32 * i + 16 * fg;
    float bv[16];
    if (HAS_BIAS) {
#pragma unroll
      for (int r = 0; r < 16; ++r) bv[r] = (ep.bias && n + r < N) ? lo16<T>(ep.bias[n + r]) : 0.f;
    }
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      const int m = m0 + wt * 32 * TT + 32 * j + fr;
      if (m >= M) continue;
      uint16_t* cp = C + (int64_t)m * ldc + n;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        if (n + 8 * half < N) {  // N % 8 == 0: a chunk is either fully inside or outside
          float a8[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) a8[r] = acc[i][j][8 * half + r];
          u32x4_t o = epi_pack8<EPI == SANA_EPI_GATE_RES ? SANA_EPI_BIAS : EPI, T>(a8, bv + 8 * half);
          if (EPI == SANA_EPI_GATE_RES) o = gate_res8<T>(o, ep, m, n + 8 * half);
          *reinterpret_cast<u32x4_t*>(cp + 8 * half) = o;
        }
      }
    }
  }
}


// Epilogue of the pipelined kernels.  acc[i][j][r] (MFMA 16x16 tiles: i = channel tile of the wave, j = token tile):
// token m0 + wt*128 + 16*j + lane%16, channel n0 + wc*32*NI + 8*NI*(lane/16) + 4*i + r.  bpk: the lane's 8*NI bias
// values, packed (the caller requests them ahead of its last k-tile so that their latency hides behind its MFMAs).
template <int EPI, int NI, bool SPLIT, typename T = BF16>
__device__ __forceinline__ void finish_tile16(f32x4_t (&acc)[2 * NI][8], const u32x4_t (&bpk)[NI], unsigned char* smem,
                                              const EpiArgs& ep, uint16_t* __restrict__ C, int M, int N, int64_t ldc,
                                              int m0, int n0) {
  constexpr int NWT = 2 * NI;
  constexpr bool HAS_BIAS = EPI != SANA_EPI_NONE;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int wc = wave & 1, wt = wave >> 1;
  const int fr = lane & 15, fg = lane >> 4;
  const int o_chunk = lane & 15, o_rsub = lane >> 4;
  const int o_n = n0 + wc * 32 * NI + o_chunk * 8;
  const bool o_live = o_chunk < 4 * NI && o_n < N;  // a staged row holds 4*NI chunks (the row pitch stays 256 bytes)
  // ---- epilogue.  acc[i][j][r]: token m0 + wt*128 + 16*j + lane%16,
  // channel n0 + wc*32*NI + 8*NI*(lane/16) + 4*i + r.  The wave's sub-tile goes through its own 32 KB of
  // LDS ([128 tokens][256 bytes], 16-byte chunks XOR-swizzled by token % 16) and comes back
  // row-contiguous, so each store instruction writes four full 256-byte row segments.  It goes in four
  // groups of 32 tokens: the stores of one group drain while the next group's activations are computed.
  if (SPLIT) {
    // raw accumulators -> partial[z][M][N] (fp32, dense).  A lane owns 8*NI consecutive channels of one token per
    // token tile j, but one store instruction of that layout would write 64 separate 16-byte pieces (16 rows x 4
    // lane groups): measured, such an epilogue took as long as the 22 k-tiles in front of it.  So the sub-tile
    // goes through the wave's 32 KB of LDS, 64 tokens at a time ([64 tokens][128 channels] fp32, 16-byte chunks
    // XOR-swizzled by token % 16), and leaves as whole row segments: a store instruction writes two rows of 512
    // contiguous bytes.  Rows past M fall outside the buffer resource and are dropped; chunks past N get the idle
    // offset.
    __syncthreads();  // every wave is done with the operand tiles
    unsigned char* stg = smem + wave * 32768;
    const int prow0 = m0 + __builtin_amdgcn_readfirstlane(wt) * 128;
    const int prows = max(0, min(128, M - prow0));
    float* plane = reinterpret_cast<float*>(C) + ((int64_t)blockIdx.y * M + prow0) * N;
    const __amdgpu_buffer_rsrc_t rsrc_p =
        __builtin_amdgcn_make_buffer_rsrc(plane, 0, (int)((int64_t)prows * N * 4), 0x00020000);
    const int s_chunk = lane & 31, s_rsub = lane >> 5;               // store side: 32 chunks of 4 channels, 2 rows
    const int s_n = n0 + wc * 32 * NI + 4 * s_chunk;
    const bool s_live = s_chunk < 8 * NI && s_n < N;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const int tok = 16 * jj + fr;                                 // token of this half, 0 .. 63
#pragma unroll
        for (int i = 0; i < NWT; ++i) {
          const int chunk = 2 * NI * fg + i;                          // 4 channels each: 8*NI*fg + 4*i
          const u32x4_t o = {__float_as_uint(acc[i][4 * half + jj][0]), __float_as_uint(acc[i][4 * half + jj][1]),
                             __float_as_uint(acc[i][4 * half + jj][2]), __float_as_uint(acc[i][4 * half + jj][3])};
          *reinterpret_cast<u32x4_t*>(stg + tok * 512 + ((chunk ^ (tok & 15)) << 4)) = o;
        }
      }
      // wave-private LDS is in order: the reads below see the writes above
#pragma unroll
      for (int it = 0; it < 32; ++it) {
        const int row = 2 * it + s_rsub;                              // 0 .. 63
        const u32x4_t o = *reinterpret_cast<const u32x4_t*>(stg + row * 512 + ((s_chunk ^ (row & 15)) << 4));
        const int off = s_live ? ((64 * half + row) * N + s_n) * 4 : (int)0x80000000u;
        __builtin_amdgcn_raw_buffer_store_b128(o, rsrc_p, off, 0, 0);
      }
    }
    return;
  }
  __syncthreads();  // every wave is done with the operand tiles
  unsigned char* stg = smem + wave * 32768;
  // Global accesses of the epilogue are buffer loads / stores on the wave's 128 rows of C (and of the
  // residual): a row costs one vector add for its offset, rows past M and channel pieces past N fall
  // outside the resource (loads return zero, stores are dropped) -- no 64-bit address arithmetic, no
  // per-row predication.
  const int wrow0 = m0 + __builtin_amdgcn_readfirstlane(wt) * 128;  // first row of this wave (a scalar: it goes into resources)
  const int wrows = max(0, min(128, M - wrow0));          // its rows that exist
  const int idle_off = (int)0x80000000u;
  const __amdgpu_buffer_rsrc_t rsrc_c = __builtin_amdgcn_make_buffer_rsrc(
      C + (int64_t)wrow0 * ldc, 0, wrows ? (int)((((int64_t)wrows - 1) * ldc + N) * 2) : 0, 0x00020000);
  const int c_off0 = o_live ? (o_rsub * (int)ldc + o_n) * 2 : idle_off, c_step = 4 * (int)ldc * 2;
  // Gated residual: the residual rows this lane will add are requested now, a whole epilogue ahead
  // of their use (128 registers that the main loop no longer needs; asking for them before the last
  // k-tile makes the compiler spill).
  u32x4_t res[4][8];
  const bool gated = EPI == SANA_EPI_GATE_RES;
  const __amdgpu_buffer_rsrc_t rsrc_r = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(gated ? ep.res + (int64_t)wrow0 * ep.ldr : nullptr), 0,
      gated && wrows ? (int)((((int64_t)wrows - 1) * ep.ldr + N) * 2) : 0, 0x00020000);
  const int r_off0 = o_live ? (o_rsub * (int)ep.ldr + o_n) * 2 : idle_off, r_step = 4 * (int)ep.ldr * 2;
  if (EPI == SANA_EPI_GATE_RES) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int it = 0; it < 8; ++it)
        res[j][it] = __builtin_bit_cast(
            u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, r_off0 + (8 * j + it) * r_step, 0, 0));
  }
  float bv[NI][8];
  if (HAS_BIAS) {
#pragma unroll
    for (int c = 0; c < NI; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        bv[c][2 * e] = lo16<T>(bpk[c][e]);
        bv[c][2 * e + 1] = hi16<T>(bpk[c][e]);
      }
  }
  // Software-pipelined over the four groups of 32 tokens: step s of phase j converts piece s of group j
  // (accumulators -> activation -> LDS) and stores row chunk s of group j - 1 (LDS -> gate / residual -> global).
  // Handing a 16-byte-per-lane store to the memory pipeline keeps it busy for ~130 clocks, during which the
  // wave can issue VALU work but not another store: one store between two pieces of arithmetic costs a
  // fraction of what eight stores in a row cost.
  auto convert_piece = [&](int jg, int p) {  // group jg of 32 tokens = token tiles 2*jg, 2*jg + 1; p = NI * (tile & 1) + c
    const int j = 2 * jg + p / NI, c = p % NI;  // c: the lane's c-th chunk of 8 channels = W tiles 2c, 2c + 1
    const int tok = 16 * j + fr;
    float a8[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) a8[r] = acc[2 * c][j][r], a8[4 + r] = acc[2 * c + 1][j][r];
    const u32x4_t o = epi_pack8<EPI == SANA_EPI_GATE_RES ? SANA_EPI_BIAS : EPI, T>(a8, bv[c]);
    const int chunk = NI * fg + c;
    *reinterpret_cast<u32x4_t*>(stg + tok * 256 + ((chunk ^ (tok & 15)) << 4)) = o;
  };
  auto read_row = [&](int j, int it) {
    const int row = 32 * j + it * 4 + o_rsub;
    return *reinterpret_cast<const u32x4_t*>(stg + row * 256 + ((o_chunk ^ (row & 15)) << 4));
  };
#pragma unroll
  for (int j = 0; j <= 4; ++j) {
    const int js = j - 1;  // the group whose rows are stored in this phase
    // The lane's eight gate values, as floats.  One gate row serves the whole group of 32 tokens unless a
    // batch boundary runs through it: then the rows from m_switch on take the next gate row (gates are per
    // batch entry; entries shorter than 32 tokens take the slow way, a division per row).
    const int m_first = wrow0 + 32 * js;
    int m_switch = 0;
    bool two_gates = false;
    float gf[8] = {1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f, 1.f};  // no gate: 1.0, a plain residual add
    u32x4_t o_next = {0u, 0u, 0u, 0u};
    if (js >= 0) {
      if (EPI == SANA_EPI_GATE_RES) {
        const int g_first = m_first / ep.rows_per_gate;
        m_switch = (g_first + 1) * ep.rows_per_gate;
        two_gates = ep.gate && m_switch < min(m_first + 32, M);
        if (ep.gate && o_live && m_first < M) {
          const u32x4_t gate = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)g_first * ep.gate_stride + o_n);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            gf[2 * e] = lo16<T>(gate[e]);
            gf[2 * e + 1] = hi16<T>(gate[e]);
          }
        }
      }
      o_next = read_row(js, 0);  // wave-private LDS is in order: the group's writes are behind it
    }
#pragma unroll
    for (int st = 0; st < 8; ++st) {
      u32x4_t o = o_next;
      if (js >= 0 && st + 1 < 8) o_next = read_row(js, st + 1);
      __builtin_amdgcn_sched_barrier(0);
      if (j < 4 && st < 2 * NI) convert_piece(j, st);
      __builtin_amdgcn_sched_barrier(0);
      if (js >= 0) {
        if (EPI == SANA_EPI_GATE_RES) o = gate_res8f<T>(o, gf, res[js][st]);
        __builtin_amdgcn_raw_buffer_store_b128(o, rsrc_c, c_off0 + (8 * js + st) * c_step, 0, kBufferNt);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (js >= 0 && two_gates) {  // uniform, rare: rows behind the boundary are redone with their own gate row and stored again
#pragma unroll 1
      for (int it = 0; it < 8; ++it) {
        const int row = 32 * js + it * 4 + o_rsub, m = wrow0 + row;
        if (o_live && m >= m_switch && m < M) {
          const u32x4_t y = *reinterpret_cast<const u32x4_t*>(stg + row * 256 + ((o_chunk ^ (row & 15)) << 4));
          const u32x4_t r = __builtin_bit_cast(
              u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rsrc_r, r_off0 + (8 * js + it) * r_step, 0, 0));
          const u32x4_t g2 = *reinterpret_cast<const u32x4_t*>(
              ep.gate + (int64_t)(m / ep.rows_per_gate) * ep.gate_stride + o_n);
          __builtin_amdgcn_raw_buffer_store_b128(gate_res8v<T>(y, g2, r), rsrc_c, c_off0 + (8 * js + it) * c_step, 0, 0);
        }
      }
    }
  }
}

// ============================================================================
// Pipelined kernel (K % 32 == 0, K >= 64; int8 weights): 256 threads, one
// wave per SIMD with the whole register file (256 accumulators + 256 VGPRs), each
// wave a sub-tile of 128 tokens x 32*NI channels = 2*NI x 8 MFMA tiles of 16x16
// (NI = 4: 128x128; NI = 3 narrows the workgroup's channel tile to 192 where that fills
// the last round of workgroups better, NI = 2 to 128 for few tokens and wide N, where the
// shorter k-tile and the larger grid shorten the latency chain).  With a single wave per SIMD nothing
// else hides a stalled memory instruction, so the main loop is one hand-ordered
// stream (pinned with sched_barrier): a k-tile is two k-steps of 32 = 2 * 16*NI MFMA
// slots of 16 cycles, and a lone wave issues about one other instruction per 5 cycles,
// so a slot carries at most a fragment read, a store or a load:
//   * k-step 0: the fragments of k-step 1; A quad q (k-tile kt+1) is stored into the
//     other LDS stage and the same registers are re-loaded with k-tile kt+2 one slot
//     later, so every global load has a whole k-tile (about 1 us) to land;
//   * weights, 16 values per quad, are converted two at a time in the MFMA slots before
//     they are stored, the quad reloaded after its last piece; the only barrier stands
//     at the end of the k-tile.
// The MFMAs are asm statements with the accumulator tied in and out (see mfma_acc).
// Rows past M / N read as zero (buffer range check) and only feed outputs that are
// never stored; the last k-tile runs just the k-steps that exist.
// ============================================================================
// SPLIT (split-k, for shapes with too few tiles to fill the chip): grid row z multiplies its own range of
// k-tiles and stores the raw fp32 accumulators to C taken as float [gridDim.y][M][N]; splitk_epilogue_kernel
// adds the ranges up in order and applies the epilogue.
template <int EPI, int NI, bool SPLIT = false>
__global__ __launch_bounds__(256) void gemm4_kernel(const uint16_t* __restrict__ A_, const int8_t* __restrict__ W_,
                                                    const float* __restrict__ scale, const EpiArgs ep,
                                                    uint16_t* __restrict__ C, int M, int N, int K_, int64_t lda,
                                                    int64_t ldw, int64_t ldc, int tiles_t, int tiles_c,
                                                    const Taps tp) {
  __shared__ __attribute__((aligned(1024))) unsigned char smem[4 * TILE_BYTES];  // [stage][A | W]
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  typedef BF16 T;
  const uint16_t* A = A_;
  const int8_t* W = W_;
  int K = K_;
  if (SPLIT) {  // this grid row's k range becomes "the" K of everything below
    const int z = blockIdx.y;
    const int kb = (z * tp.split_tiles + min(z, tp.split_rem)) * BK;
    const int kn = (tp.split_tiles + (z < tp.split_rem ? 1 : 0)) * BK;
    A += kb;
    W += kb;
    K = min(K_ - kb, kn);
  }
  const int total = tiles_t * tiles_c;
  int pid = blockIdx.x;
  {
    const int xcd = pid & 7, local = pid >> 3;
    const int base = total >> 3, rem = total & 7;
    pid = xcd * base + min(xcd, rem) + local;
  }
  // tile rows per group: an XCD's 32 concurrent tiles are GROUP rows x 32/GROUP columns.  Measured: 4 is 1-2 % better
  // for the short-K wide-N shapes (qkv, inverted conv), 8 is 2-3 % better for the long-K point conv.
  const int GROUP = K >= 4096 ? 8 : 4;
  const int group_sz = GROUP * tiles_c;
  const int gid = pid / group_sz;
  const int first_t = gid * GROUP;
  const int gt = min(tiles_t - first_t, GROUP);
  const int tile_t = first_t + (pid % group_sz) % gt;
  const int tile_c = (pid % group_sz) / gt;
  constexpr int BCN = 64 * NI;  // channels per workgroup: two waves x NI MFMA tiles of 32
  const int m0 = tile_t * BT, n0 = tile_c * BCN;

  // global -> VGPR -> LDS: thread -> k chunk tid%8, rows tid/8 + 32*q, q < 8 for A.
  // W: thread -> 16-value chunk tid%4, rows tid/4 + 64*q (q < NI); dequantised on the way to LDS.
  const int g_chunk = tid & 7, g_row = tid >> 3;
  const int a_last = min(BT, M - m0) - 1, w_last = min(BCN, N - n0) - 1;  // last valid row of each tile
  const uint32_t ulda = (uint32_t)lda;
  const int a_dst0 = swz(g_row, g_chunk);               // rows +32*q keep the key: +4096 bytes each
  // LDS row L of a wave's block of 32*NI weight rows belongs to MFMA tile L / 16 as its row L % 16 = 4*g + r, and
  // holds channel 8*NI*g + 4*(L / 16) + r of the block: a lane's accumulators (tile i, registers r) are then the
  // 8*NI contiguous channels 8*NI*g + 4*i + r.
  constexpr int NQ = 8 + NI;
  u32x4_t rs[NQ];  // the k-tile in flight: A quads 0..7, then the W quads
  const int q_chunk = tid & 3, q_row = tid >> 2;
  const int q_dst_lo = TILE_BYTES + swz(q_row, 2 * q_chunk);  // LDS rows q_row + 64*q: +8192 bytes, same key
  const int q_dst_hi = TILE_BYTES + swz(q_row, 2 * q_chunk + 1);
  float wscale[NI], woff[NI];
  int q_voff[NI];  // int8 quads: byte offset of the channel that LDS row q_row + 64*q holds
#pragma unroll
  for (int q = 0; q < NI; ++q) {
    const int L = q_row + 64 * q, blk = L / (32 * NI), l = L % (32 * NI);
    const int chan = blk * 32 * NI + 8 * NI * ((l >> 2) & 3) + 4 * (l >> 4) + (l & 3);
    q_voff[q] = chan * (int)ldw + 16 * q_chunk;
    wscale[q] = scale[n0 + min(chan, w_last)];
    woff[q] = -128.f * wscale[q];
  }
  u32x4_t dq[2];  // dequantised halves of the int8 quad being converted

  const int wc = wave & 1, wt = wave >> 1;
  const int fr = lane & 15, fg = lane >> 4;
  const int x7 = swz_key(fr);
  const int w_off = TILE_BYTES + (wc * 32 * NI + fr) * ROW_BYTES, a_off = (wt * 128 + fr) * ROW_BYTES;
  constexpr int NWT = 2 * NI;  // MFMA tiles of 16 channels per wave (and 8 tiles of 16 tokens)
  f32x4_t acc[NWT][8];
#pragma unroll
  for (int i = 0; i < NWT; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;
  u32x4_t fw[2][NWT], fa[2][8];

#define SANA_G4_PIN() __builtin_amdgcn_sched_barrier(0)
  // Operand tiles are read with buffer loads: the tile's rows are one resource each for A and W (scalar
  // registers), the lane's (row, k chunk) is a constant vector offset, and the quad / k-tile part of the
  // address is scalar, so a load costs one vector add.  The resource ends with the last valid row's
  // K-th element: rows past M / N and anything past the end of the matrix read as zero instead of
  // faulting (k chunks past K inside the matrix read the next row: they are never multiplied).
  const int64_t a_bytes = ((int64_t)a_last * lda + K) * 2;
  const __amdgpu_buffer_rsrc_t rsrc_a = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint16_t*>(A + (int64_t)m0 * lda), 0, (int)a_bytes, 0x00020000);
  const __amdgpu_buffer_rsrc_t rsrc_w = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<int8_t*>(W + (int64_t)n0 * ldw), 0, (int)((int64_t)w_last * ldw + K), 0x00020000);
  const int voff_a = (g_row * (int)ulda + 8 * g_chunk) * 2;
  const int step_a = 32 * (int)ulda * 2;
  auto gload = [&](int q, int k0) {
    if (q < 8) {
      const int off = voff_a + (q * step_a + k0 * 2);
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_a, off, 0, 0);
      rs[q] = __builtin_bit_cast(u32x4_t, v);
    } else {
      const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc_w, q_voff[q - 8] + k0, 0, 0);
      rs[q] = __builtin_bit_cast(u32x4_t, v);
    }
  };
  auto lstore = [&](int q, int stage) {  // A quads
    *reinterpret_cast<u32x4_t*>(smem + stage * 2 * TILE_BYTES + a_dst0 + 4096 * q) = rs[q];
  };
  // int8 quad wq (16 values), piece 0..7 = two values each: convert, and store a 16-byte half when complete
  auto dequant_piece = [&](int wq, int piece, int stage) {
    uint32_t word = rs[8 + wq][piece >> 1] ^ 0x80808080u;
    dq[piece >> 2][piece & 3] = dequant2(word, piece & 1, wscale[wq], woff[wq]);
    if ((piece & 3) == 3) {
      unsigned char* base = smem + stage * 2 * TILE_BYTES + 8192 * wq;
      *reinterpret_cast<u32x4_t*>(base + (piece < 4 ? q_dst_lo : q_dst_hi)) = dq[piece >> 2];
    }
  };
  constexpr int NFR = NWT + 8;  // fragment reads per k-step (of 32)
  // read r of a k-step, in the order the MFMAs need them: W tile 0, the eight A tiles, then W tiles 1 ..
  auto fread = [&](const unsigned char* st, int buf, int ks, int r) {
    const int col = ((4 * ks + fg) ^ x7) << 4;
    if (r == 0 || r > 8) {
      const int i = r == 0 ? 0 : r - 8;
      fw[buf][i] = *reinterpret_cast<const u32x4_t*>(st + w_off + i * 16 * ROW_BYTES + col);
    } else {
      fa[buf][r - 1] = *reinterpret_cast<const u32x4_t*>(st + a_off + (r - 1) * 16 * ROW_BYTES + col);
    }
  };
  // MFMA t of a k-step: weight tile t / 8, and the token tiles in alternating direction (0..7, 7..0, ..), so that
  // every MFMA differs from its predecessor in ONE operand -- at the end of a row of eight only the weight fragment
  // changes, not both.  Less switching on the operand buses: the power-limited clock settles ~1 % higher.
  auto mfma = [&](int buf, int t) {  // t < 8 * NWT
    const int i = t >> 3, j = (i & 1) ? 7 - (t & 7) : (t & 7);
    mfma_acc<T>(acc[i][j], fw[buf][i], fa[buf][j]);
  };

  const int KT = (K + BK - 1) / BK;
  // prologue: k-tile 0 -> stage 0, k-tile 1 in flight
#pragma unroll
  for (int q = 0; q < NQ; ++q) gload(q, 0);
#pragma unroll
  for (int q = 0; q < 8; ++q) lstore(q, 0);
#pragma unroll
  for (int n = 0; n < 8 * NI; ++n) dequant_piece(n >> 3, n & 7, 0);
#pragma unroll
  for (int q = 0; q < NQ; ++q) gload(q, BK);
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NFR; ++q) fread(smem, 0, 0, q);

  // Slots: a k-tile is two k-steps of 32 = 2 * SL MFMAs of 16 cycles each, and a lone wave issues about one
  // other instruction per 5 cycles, so no slot carries more than a fragment read or a store or a load.
  // The fragments of k-step 1 are read in k-step 0 (read r at slot r*SL/NFR), the weights converted in 8*NI pieces over the whole
  // k-tile; the barrier and the next tile's k-step-0 fragments stand at its end.
  constexpr int SL = 8 * NWT, TS = 2 * SL;
  constexpr int BAR = TS - NFR - 1;
  constexpr int PSTR = (BAR - 4) / (8 * NI);                 // piece n (two values) at slot 2 + n*PSTR
  static_assert(4 * 7 + 1 < BAR && PSTR >= 1, "staging does not fit in front of the barrier");
  // The MFMAs below are asm statements: the compiler neither knows that they read the accumulators through the
  // matrix pipe nor places the wait states such a read needs behind the VALU writes that zeroed them.  Pin the
  // order by hand: every accumulator passes through an empty asm statement (its zeroing is complete, in program
  // order, in front of it), then eight wait states, then the first MFMA -- whatever the compiler puts in between.
#pragma unroll
  for (int i = 0; i < NWT; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_nop 7" ::: "memory");
  for (int kt = 0; kt < KT - 1; ++kt) {
    const int cur = kt & 1;
    const unsigned char* st = smem + cur * 2 * TILE_BYTES;
    const unsigned char* stn = smem + (cur ^ 1) * 2 * TILE_BYTES;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int t = 0; t < SL; ++t) {
        const int slot = ks * SL + t;
        mfma(ks, t);
        SANA_G4_PIN();
        if (ks == 0) {
          // read r of k-step 1 goes to slot (r * SL) / NFR of k-step 0
          if (((t * NFR + SL - 1) / SL) * SL / NFR == t && (t * NFR + SL - 1) / SL < NFR)
            fread(st, 1, 1, (t * NFR + SL - 1) / SL);
        }
        if (slot == BAR) {
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own LDS stores done; no fence: loads stay in flight
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
        } else if (slot > BAR && slot - BAR - 1 < NFR) {
          fread(stn, 0, 0, slot - BAR - 1);
        }
        // A quad q: store at slot 4q, reload at 4q+1.  Piece n at slot 2 + n*PSTR (its half is stored with pieces 3 and 7), the quad
        // is reloaded one slot after its last piece.
        if (slot % 4 == 0 && slot / 4 < 8) lstore(slot / 4, cur ^ 1);
        if (slot % 4 == 1 && slot / 4 < 8) gload(slot / 4, (kt + 2) * BK);
        if (slot >= 2 && (slot - 2) % PSTR == 0 && (slot - 2) / PSTR < 8 * NI)
          dequant_piece(((slot - 2) / PSTR) >> 3, ((slot - 2) / PSTR) & 7, cur ^ 1);
        if (slot >= 3 && (slot - 3) % PSTR == 0 && (slot - 3) / PSTR < 8 * NI && (((slot - 3) / PSTR) & 7) == 7)
          gload(8 + (((slot - 3) / PSTR) >> 3), (kt + 2) * BK);
        SANA_G4_PIN();
      }
    }
  }
#undef SANA_G4_PIN
  // The lane's bias values (16 consecutive channels per MFMA tile, packed) are requested here, ahead of
  // the last k-tile, so that their latency hides behind its MFMAs.
  constexpr bool HAS_BIAS = EPI != SANA_EPI_NONE;
  u32x4_t bpk[NI];  // the lane's 8*NI contiguous channels, in chunks of 8
  if (HAS_BIAS) {
#pragma unroll
    for (int c = 0; c < NI; ++c) {
      const int n = n0 + wc * 32 * NI + 8 * NI * fg + 8 * c;  // N % 8 == 0: a chunk is in or out
      bpk[c] = (ep.bias && n < N) ? *reinterpret_cast<const u32x4_t*>(ep.bias + n) : u32x4_t{0u, 0u, 0u, 0u};
    }
  }
  {  // last k-tile: no successor, and K % 64 may leave one k-step of 32 instead of two
    const unsigned char* st = smem + ((KT - 1) & 1) * 2 * TILE_BYTES;
    const int steps = (K - (KT - 1) * BK) / 32;
    for (int ks = 0; ks < steps; ++ks) {
      const int col = ((4 * ks + fg) ^ x7) << 4;
      u32x4_t w8[NWT], a8[8];
#pragma unroll
      for (int i = 0; i < NWT; ++i) w8[i] = *reinterpret_cast<const u32x4_t*>(st + w_off + i * 16 * ROW_BYTES + col);
#pragma unroll
      for (int j = 0; j < 8; ++j) a8[j] = *reinterpret_cast<const u32x4_t*>(st + a_off + j * 16 * ROW_BYTES + col);
#pragma unroll
      for (int i = 0; i < NWT; ++i)
#pragma unroll
        for (int jj = 0; jj < 8; ++jj) {
          const int j = (i & 1) ? 7 - jj : jj;
          mfma_acc<T>(acc[i][j], w8[i], a8[j]);
        }
    }
    // the MFMAs are asm statements, so the compiler does not know that their results are in flight: wait out the
    // last ones before anything reads an accumulator
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  }

  finish_tile16<EPI, NI, SPLIT, T>(acc, bpk, smem, ep, C, M, N, ldc, m0, n0);
}

// Second half of a split-k GEMM: partial[S][M][N] (fp32) -> C = epilogue(sum over the S <= 8 k-ranges, added in
// order).  One thread per row and 8 channels; the same epilogue functions as the fused path.  All planes, the residual and the gate are
// requested at once (plane by plane 0.3 us more a launch); the rest is the planes, 46 MB written and read at 1024 x 2240 in five ranges.
template <int EPI, typename T = BF16>
__global__ __launch_bounds__(256) void splitk_epilogue_kernel(const float* __restrict__ partial, int S,
                                                               const EpiArgs ep, uint16_t* __restrict__ C, int M, int N,
                                                               int64_t ldc) {
  const uint32_t chunks = N >> 3, id = blockIdx.x * 256u + threadIdx.x;  // (M * N * 4 < 2^31)
  if (id >= M * chunks) return;
  const int m = (int)(id / chunks), n = (int)(id - m * chunks) * 8;
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(partial + (int64_t)m * N + n);
  const int64_t plane = (int64_t)M * N / 4;
  constexpr bool GATED = EPI == SANA_EPI_GATE_RES;
  u32x4_t b = {0u, 0u, 0u, 0u}, g, r;
  if (EPI != SANA_EPI_NONE && ep.bias) b = *reinterpret_cast<const u32x4_t*>(ep.bias + n);
  if constexpr (GATED) {
    g = *reinterpret_cast<const u32x4_t*>(ep.gate + (int64_t)((uint32_t)m / (uint32_t)ep.rows_per_gate) * ep.gate_stride + n);
    r = *reinterpret_cast<const u32x4_t*>(ep.res + (int64_t)m * ep.ldr + n);
  }
  f32x4_t lo, hi;
  auto sum = [&](auto s_c) {
    constexpr int Z = decltype(s_c)::value;
    f32x4_t l[Z], h[Z];
#pragma unroll
    for (int z = 0; z < Z; ++z) l[z] = p[z * plane], h[z] = p[z * plane + 1];
    lo = l[0], hi = h[0];
#pragma unroll
    for (int z = 1; z < Z; ++z) lo += l[z], hi += h[z];
  };
  switch (S) {
    case 2: sum(std::integral_constant<int, 2>{}); break;
    case 3: sum(std::integral_constant<int, 3>{}); break;
    case 4: sum(std::integral_constant<int, 4>{}); break;
    case 5: sum(std::integral_constant<int, 5>{}); break;
    case 6: sum(std::integral_constant<int, 6>{}); break;
    case 7: sum(std::integral_constant<int, 7>{}); break;
    default: sum(std::integral_constant<int, 8>{}); break;  // (plan_gemm: 2 .. 8)
  }
  float a[8], bv[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    a[e] = lo[e], a[4 + e] = hi[e];
    bv[2 * e] = lo16<T>(b[e]), bv[2 * e + 1] = hi16<T>(b[e]);
  }
  u32x4_t o = epi_pack8<GATED ? SANA_EPI_BIAS : EPI, T>(a, bv);
  if constexpr (GATED) o = gate_res8v<T>(o, g, r);
  *reinterpret_cast<u32x4_t*>(C + (int64_t)m * ldc + n) = o;
}

// The library is built for one chip, MI355X: 256 compute units in 8 XCDs.  A constant (not a device query)
// keeps the library free of global state and makes the plans -- and sana_hip_gemm_workspace_bytes -- the same on
// every host, with or without a GPU.
constexpr int compute_units() { return 256; }

// Channel tile of the pipelined kernel (int8 weights, and K split: NI = 4: 256 channels, 3: 192).  One workgroup per compute unit at a
// time, so the grid runs in rounds: the tile whose rounds x tile size is smaller wins; the narrower tile
// re-reads a little more per MFMA, hence its 4 % handicap.
int pick_ni(int M, int N) {
  const int64_t cu = compute_units(), tiles_t = (M + BT - 1) / BT;
  const int64_t t256 = tiles_t * ((N + 255) / 256), t192 = tiles_t * ((N + 191) / 192);
  const double cost256 = (double)((t256 + cu - 1) / cu) * 4.0, cost192 = (double)((t192 + cu - 1) / cu) * 3.0 * 1.04;
  return cost192 < cost256 ? 3 : 4;
}

// The split of K that could pay, and the tile of an unsplit GEMM with int8 weights (16-bit weights unsplit: plan16).  A
// workgroup's K loop is a latency chain whatever the grid: about 1.1 us per k-tile for the 256-wide pipelined kernel, 0.8 us
// for the 128 x 128 one (a quarter of the math, but the same load / LDS / barrier round trip).  A grid that covers the chip
// keeps the 256-wide kernel (throughput is what counts, and that kernel has twice the math per byte).  A grid of fewer tiles
// than half the compute units (M = 1024 tokens x N = 2240: 48 workgroups on 256 CUs) leaves most of the chip idle for the
// whole chain; two remedies, by estimate:
//  * split-k: S ranges of >= 8 k-tiles (S <= 8, S x tiles <= CUs) shorten the chain to ceil(KT / S) k-tiles and
//    cost the fp32 partial planes (S x M x N x 4 bytes written and read once, about 6 bytes/ns at these sizes)
//    plus a second launch (about 5 us); a candidate where that beats the unsplit chain by 15 %.  Whether it is taken
//    is split_pays' to say, against the best unsplit 16-bit tile.
//  * the 128 x 128 kernel, when its grid still fits one workgroup per CU and its chain beats the above.  (It rules the
//    split out for 16-bit weights too, which have better small tiles still: both kinds of weight split alike.)
struct GemmPlan {
  bool small;         // the 128 x 128 kernel
  int S, tiles, rem;  // k ranges; k-tiles per range; ranges that take one more
};
GemmPlan plan_gemm(int M, int N, int K, bool w8) {
  GemmPlan pl = {false, 1, 0, 0};
  const int KT = (K + BK - 1) / BK, cu = compute_units();
  const bool pipelined = K % 32 == 0 && K >= 64;
  const double us_tile = pipelined ? 1.1 : 1.4, us_tile_small = 0.8, us_launch = 5.0, bytes_per_us = 6.0e6;
  double best = KT * us_tile;
  if (pipelined) {
    const int ni = pick_ni(M, N);
    const int64_t tiles = (int64_t)((M + BT - 1) / BT) * ((N + 64 * ni - 1) / (64 * ni));
    if (tiles * 2 <= cu && KT >= 16 && (int64_t)M * N * 4 < ((int64_t)1 << 31)) {
      int smax = (int)(cu / tiles);
      if (smax > KT / 8) smax = KT / 8;
      if (smax > 8) smax = 8;
      double bound = best * 0.85;
      for (int s = 2; s <= smax; ++s) {
        const double t = (KT + s - 1) / s * us_tile + (double)s * M * N * 8.0 / bytes_per_us + us_launch;
        if (t < bound) {
          bound = best = t;
          pl.S = s;
        }
      }
    }
  }
  const int64_t tiles128 = (int64_t)((M + 127) / 128) * ((N + 127) / 128);
  if (tiles128 <= cu && K % (w8 ? 16 : 8) == 0 && KT * us_tile_small + 3.0 < best) {
    pl.small = true;
    pl.S = 1;
  }
  pl.tiles = KT / pl.S;
  pl.rem = KT % pl.S;
  return pl;
}
size_t split_bytes(const GemmPlan& pl, int M, int N) { return pl.S > 1 ? (size_t)pl.S * M * N * sizeof(float) : 0; }

// Time of an unsplit 16-bit GEMM in a given tile, us: ceil(K / 64) k-tiles per round of workgroups, at a rate per k-tile that
// grows from `lone` (lone_to workgroups or fewer in the round) to `full` (full_from or more: the weights come from HBM, the
// matrix pipes share a power budget), plus launch, first loads and epilogue.
constexpr int kHalvedTiles = 128;  // up to so many tiles of 64 x 64 run as two workgroups of 32 channels each
struct Tile16 {
  int bm, bn;    // tokens, channels; 256 x 192 and 256 x 256 (256 x 128 below kShortK): gemm8_kernel, 288 channels: gemm288_kernel; else
                 // gemm_ring_kernel
  int resident;  // workgroups on the chip at a time
  int lone_to, full_from;
  double fixed, lone, full;
  bool one_round = false;  // beyond one round of workgroups, every round is charged in full
  double halved = 0;       // > 0: k-tile where there are at most kHalvedTiles of them, in two workgroups each; a fit of its own:
  double halved_few = 0;   // 4 % off.  One row of tiles or a few: every weight comes from HBM to one workgroup (64 x 2240 x 5600 27 us,
                           // split 24), or to few of them
};
// Fitted to 250 shapes (64 .. 32760 tokens, the eight projections of the two image widths and the text's, one block's and a
// step's, weights cold, launches replayed from a graph: issued one by one, a launch of less than 20 us is timed by its issue):
// 7 - 14 % off each.  Of 304 shapes timed with every tile as it is now (profiles/gemm_tiles_by_shape.txt) the choice is 0.6 % from the
// best on the mean, more than 6 % in seven; of 124 at random token counts 0.6 %, more than 6 % in one.  In a second round
// the small tiles were never more than 2 % ahead, and 300 x 17920 x 2240 is 48.7 us in 128 x 128 and 40.4 in 256 x 192: hence
// one_round.  us, the tiles and kernels before this table / now, both timed so: 256 x 1152 x 2880 15.3 / 10.3 (halved), 1024 x 2240 x
// 2240 23.6 / 18.7, 2048 x 1152 x 2880 28.6 / 21.6, 4096 x 1152 x 1152 20.7 / 17.7, 4096 x 1152 x 2880 35.0 / 31.4.
// The 192-wide tile's fixed part was 7.9 before the waves shared its rows (gemm8.h).  With 4.9, of the shapes that this changes (200 ..
// 20000 tokens, widths as above), kernel as it is, 7.9 / 4.9: 14208 x 3456 x 1152 109 / 98, 16576 x 2240 x 2240 167 / 157, 7246 x 9216 x 1152 140 /
// 133, 6017 x 11200 x 2240 251 / 241, 2079 x 18432 x 1152 88 / 84, 12423 x 2240 x 2240 115 / 111; 18219 x 9216 x 1152 307 / 311, 6400 x 6720 x 2240
// 145 / 151; 0.979 on the mean of 48.  (Against the former kernel at its price those two are ties, 313 / 312 and 151 / 151.  3.9: 993 x 18432 x
// 1152 42.7 / 48.1.)
// 160 x 192 is chosen where one, two, four or five rows of its tiles are one round, and the rows of 256 would be padded by two fifths and
// more, smaller tiles take two rounds: 71 .. 160 tokens from 32800 channels, 257 .. 320 from 16500, 519 .. 640 from 10900 (K > 4096), 771 .. 799 from
// 8300 (K > 2800).  us, the best other tile / so, weights cold: 150 x 46080 x 2240 47.1 / 42.8, 260 x 17920 x 2240 39.2 / 33.7, 300 x 24000 x 1152 26.2 / 22.6,
// 300 x 20480 x 1536 with a gate 34.0 / 31.6, 519 x 10960 x 4608 74.0 / 55.5, 784 x 9216 x 4096 58.5 / 52.4; 0.75 .. 1.00 of it at 247 such shapes; 57 of K =
// 5600, whose rows are 87.5 lines of 128 bytes, 0.88 .. 1.10 (784 x 9216 x 5600 83.6 / 92.4).  A prompt's 300 tokens take it for the keys and values of 8 blocks
// of 1152 channels or 4 of 2240; for those of 28 and 20 256 channels or two widths are faster (55.5 / 57.5, 134.6 / 137.1) and chosen.
constexpr Tile16 kTiles16[] = {
    {64, 64, 512, 256, 257, 3.0, 0.288, 0.503, true, 0.165, 0.26}, {64, 128, 256, 32, 256, 3.9, 0.350, 0.414, true},
    {96, 128, 256, 32, 256, 3.7, 0.439, 0.466, true},  {128, 128, 256, 32, 256, 3.9, 0.454, 0.541, true},
    {128, 160, 256, 32, 256, 4.3, 0.517, 0.643, true}, {192, 128, 256, 32, 256, 4.7, 0.497, 0.687, true},
    {256, 128, 256, 32, 256, 5.1, 0.624, 0.825, true}, {256, 192, 256, 32, 256, 4.9, 0.628, 1.150},
    {256, 256, 256, 32, 256, 5.3, 0.999, 1.404},       {256, 288, 256, 32, 256, 9.5, 0.955, 1.603},
    {160, 192, 256, 32, 256, 7.4, 0.487, 0.975, true},
};
constexpr int kTile192 = 7, kTile256 = 8, kTile288 = 9;
// The same for K % 32, where rows that follow one another straddle the 64-byte sectors, with no residual: the price that the 192-wide tile had
// before (above), which keeps such GEMMs in 256 or 288 channels; two widths read the rows of A twice.  us, 4.9 / 7.9, weights cold: 6893 x 4016 x 2064
// 119 / 107 (but x 2048 99 / 97), 12506 x 5144 x 4584 511 / 476, 17278 x 3928 x 1200 177 / 145, 4502 x 11456 x 1656 165 / 148, 28755 x 1128 x 1264 85 / 75;
// one round of 192 the slower way: 2100 x 5280 x 1072 28 / 31; 0.963 on the mean of the 100 shapes timed.  With a residual 4.9 gains there too (0.98 of 37).
constexpr auto kTilesStraddling = [] {
  struct { Tile16 t[sizeof(kTiles16) / sizeof(Tile16)]; } r = {};
  for (size_t i = 0; i < sizeof(kTiles16) / sizeof(Tile16); ++i) r.t[i] = kTiles16[i];
  r.t[kTile192].fixed = 7.9;
  return r;
}();
// K below 1024.  These are the times that the tiles had in GEMMs of K = 1152 .. 5600 before the loop over whole k-tiles; at such K
// no other loop runs, and 256 x 128 is gemm8_kernel's there.  As times they are up to 30 % off (epilogues and the fill of the rings are most of
// a launch), as a choice they serve: of 560 shapes (64 .. 24576 tokens, 320 .. 6144 channels, K 64 .. 960, the ten tiles forced in turn)
// 2.7 % from the best tile on the mean, more than 6 % in 91 (sizes just past a round of 256 x 192 or 256 x 128, mostly).  Constants fitted to
// those shapes come to 2.0 %.
constexpr Tile16 kTilesShort[] = {
    {256, 128, 256, 32, 256, 3.8, 0.73, 0.85}, {256, 192, 256, 32, 256, 5.7, 0.86, 1.17}, {256, 256, 256, 32, 256, 6.1, 1.12, 1.37},
    {64, 64, 512, 64, 512, 2.1, 0.255, 0.466}, {64, 128, 256, 32, 256, 2.0, 0.42, 0.42},  {128, 128, 256, 32, 256, 2.4, 0.50, 0.59},
    {128, 160, 256, 32, 256, 4.2, 0.58, 0.68},
};
double cost16(const Tile16& t, int64_t M, int64_t N, int K) {
  const int64_t n = (M + t.bm - 1) / t.bm * ((N + t.bn - 1) / t.bn), rounds = n / t.resident, rest = n % t.resident;
  const double kt = (K + BK - 1) / BK;
  if (t.halved > 0 && n <= kHalvedTiles) return t.fixed + kt * (M > t.bm && n > kHalvedTiles / 4 ? t.halved : t.halved_few);
  if (t.one_round && n > t.resident) return (rounds + (rest ? 1 : 0)) * (kt * t.full + t.fixed);
  double us = t.fixed + rounds * (kt * t.full + 0.5 * t.fixed);
  if (rest)
    us += kt * (t.lone + (t.full - t.lone) * std::min(1.0, std::max(0.0, double(rest - t.lone_to) / (t.full_from - t.lone_to))));
  return us;
}
// The 288-wide tile at such K: its k-tile costs 1.18 times the 256-wide one's for 1.125 times the work, so it pays where it saves
// rounds.  Fitted, and the tiles it is compared with too, to 120 shapes of 700 .. 32760 tokens; taken at 0.99 of the others'
// estimate or less.  Of 330 random shapes that took it (K 256 .. 5600, odd sizes) it was at 0.90 of the time on the mean; three
// were 6 - 12 % slower, at K 600 - 830 with several rounds and no epilogue.
constexpr Tile16 kShort288 = {256, 288, 256, 32, 256, 11.3, 1.17, 1.61};
constexpr Tile16 kBesideShort288[] = {
    {256, 128, 256, 32, 256, 4.8, 0.75, 0.89}, {256, 192, 256, 32, 256, 7.4, 0.85, 1.18}, {256, 256, 256, 32, 256, 7.0, 1.20, 1.40},
    {128, 128, 256, 32, 256, 2.3, 0.51, 0.61}, {128, 160, 256, 32, 256, 4.1, 0.62, 0.68},
};
constexpr int64_t kMaxStride288 = 1 << 21;  // rows of W from which the 32-bit offsets inside a tile could overflow
bool short_takes_288(int M, int N, int K, double others_us) {  // others_us: by the constants above, which are lower
  const double us = cost16(kShort288, M, N, K) / 0.99;
  if (us > 1.1 * others_us) return false;
  for (const Tile16& t : kBesideShort288)
    if (us > cost16(t, M, N, K)) return false;
  for (int a = 256; a < N; a += 256)
    if (us > cost16(kBesideShort288[2], M, a, K) + cost16(kBesideShort288[1], M, N - a, K)) return false;
  return true;
}
constexpr int kShortK = 1024;
struct Plan16 {
  const Tile16* tile;
  int bn;      // channels of a workgroup: the tile's, or 32 (halved 64 x 64)
  int n_wide;  // > 0: the first n_wide channels in 256 x 256 tiles, the rest in 256 x 192 ones, two launches
  double us;
};
// the cheapest tile, or two widths where their last rounds fill better (4096 x 6720 tokens x channels, K = 2240: 432 tiles of 256
// are 1.7 rounds, 15 x 16 and 15 x 16 tiles of the mix two that are 94 % full) by more than what the fit tells apart
template <size_t TILES>
Plan16 cheapest16(const Tile16 (&tiles)[TILES], const Tile16& t256, const Tile16& t192, double mix_below, double mix_below_288, int M, int N, int K) {
  Plan16 p = {&tiles[0], 0, 0, 1e30};
  for (const Tile16& t : tiles) {
    const double us = cost16(t, M, N, K);
    if (us < p.us) p.tile = &t, p.us = us;
  }
  const double below = (p.tile->bn == 288 ? mix_below_288 : mix_below) * p.us;
  for (int a = 256; a < N; a += 256) {
    const double us = cost16(t256, M, a, K) + cost16(t192, M, N - a, K);
    if (us < below && us < p.us) p.n_wide = a, p.us = us;
  }
  const bool halved = p.tile->bm == 64 && p.tile->bn == 64 && (int64_t)((M + 63) / 64) * ((N + 63) / 64) <= kHalvedTiles;
  p.bn = p.n_wide ? 256 : halved ? 32 : p.tile->bn;
  return p;
}
// gated: with a residual, two widths take the place of 288 channels by 4 % at least: both launches' epilogues wait for it.  us, two widths / 288
// channels, weights cold, by how far the estimates are apart: 0.8 - 2 % 31676 x 2240 x 2240 286 / 274, 39680 x 2240 x 5600 946 / 830, 24455 x 2224 x 2368 225 /
// 223, 17757 x 4800 x 5248 689 / 702, 1.02 on the mean of 40 shapes; 2 - 4 % 38042 x 2240 x 5600 905 / 801, 17604 x 4968 x 3584 512 / 505, 30494 x 3112 x 5440 872 /
// 841, 1.03 of 22; beyond a tie with cold rows too (1.01 of 38) and 36897 x 2240 x 2240 323 / 335 without.  With no residual they are the faster ones:
// 31250 x 2240 x 2240 238 / 247.
Plan16 plan16(int M, int N, int K, bool gated = false) {
  if (K >= kShortK && K % 32 && !gated)
    return cheapest16(kTilesStraddling.t, kTilesStraddling.t[kTile256], kTilesStraddling.t[kTile192], 0.992, 0.992, M, N, K);
  if (K >= kShortK) return cheapest16(kTiles16, kTiles16[kTile256], kTiles16[kTile192], 0.992, gated ? 0.96 : 0.992, M, N, K);
  const Plan16 p = cheapest16(kTilesShort, kTilesShort[2], kTilesShort[1], 0.98, 0.98, M, N, K);
  return short_takes_288(M, N, K, p.us) ? Plan16{&kShort288, 288, 0, cost16(kShort288, M, N, K)} : p;
}
// Split over k, or not: the split GEMM against the best unsplit one (16-bit and int8 weights decide alike, so that they
// keep giving the same bits).  Time of the split one: fitted to 49 shapes when gemm4_kernel ran the ranges; gemm8_kernel's are 3 - 8 % longer with
// cold weights (42.3 estimated, 46.1 taken at 1024 x 2240 x 5600).  So is the unsplit tiles' fit, by 3 - 13 %, at the K of 5600 where it is taken (their
// weights come from HBM for longer than the prefetch reaches): 1024 x 2240 x 5600 is 46 us either way, 256 x 2240 x 5600 30 split and 34 not, 1560 58 and 53.
// A split GEMM adds up short chains, so that its fp32 sums are closer to the 64-bit ones than those of one chain: 2240 x 5600, rms error
// 1.0e-7 of the result in eight ranges, 2.4e-7 in one.  Precision is not given up for time: where the split was the faster one
// against the tiles as they once were (kTilesShort, their times then), k stays in ranges though some tiles have become faster since.
// 16-bit weights then take the faster tile all the same, which adds the ranges' sums up itself, in their order, with the same bits:
// us, split / so: 72 x 2240 x 5600 24.9 / 17.4, 144 27.6 / 18.4, 400 30.9 / 25.7, 1260 49.9 / 48.1, 2400 74.8 / 68.4.
enum class SplitWay { no, split, ranges };  // ranges: of a ring tile (16-bit weights; int8 ones are split)
SplitWay split_way(const GemmPlan& pl, int M, int N, int K) {
  if (pl.S <= 1) return SplitWay::no;
  const int kt = (K + BK - 1) / BK;
  const double us = 9.4 + 1.12 * ((kt + pl.S - 1) / pl.S) + 0.139e-6 * pl.S * M * N * 8;
  const Plan16 p = plan16(M, N, K);
  if (us < 1.04 * p.us) return SplitWay::split;
  double rival = 1e30;
  for (const Tile16& t : kTilesShort) rival = std::min(rival, cost16(t, M, N, K));
  if (us >= 0.97 * rival) return SplitWay::no;
  const bool ring = !p.n_wide && (p.bn == 32 || (p.tile->bm == 64 && p.bn == 64) || (p.bn == 128 && (p.tile->bm == 96 || p.tile->bm == 192)));
  return ring ? SplitWay::ranges : SplitWay::split;
}
bool split_pays(const GemmPlan& pl, int M, int N, int K) { return split_way(pl, M, N, K) != SplitWay::no; }

// K split into pl.S ranges (ws holds the partial planes): tiles of 256 x 192, which is pick_ni's choice wherever plan_gemm splits (one round).
template <bool W8, typename T>
int launch_split(const uint16_t* a, const void* W, const float* scale, const EpiArgs& ep, uint16_t* c, int M, int N, int K, int64_t lda,
                 int64_t ldw, int64_t ldc, int epilogue, hipStream_t s, const GemmPlan& pl, float* ws) {
  const int tiles_t = (M + BT - 1) / BT, tiles_c = (N + 191) / 192;
  if constexpr (W8) {
    const Taps split = {0, 0, 0, pl.tiles, pl.rem, nullptr};
    hipLaunchKernelGGL((gemm4_kernel<SANA_EPI_NONE, 3, true>), dim3((unsigned)(tiles_t * tiles_c), (unsigned)pl.S), dim3(256), 0, s, a,
                       static_cast<const int8_t*>(W), scale, ep, reinterpret_cast<uint16_t*>(ws), M, N, K, lda, ldw, ldc, tiles_t, tiles_c,
                       split);
    if (hipGetLastError() != hipSuccess) return SANA_ERR_LAUNCH;
  } else {
    const int rc = gemm8_planes_launch(a, static_cast<const uint16_t*>(W), ws, M, N, K, lda, ldw, is_f16<T>, pl.tiles, pl.rem, pl.S, s);
    if (rc != SANA_OK) return rc;
  }
  const dim3 egrid((unsigned)(((int64_t)M * (N / 8) + 255) / 256));
#define SANA_SPLIT_EPI(EPI) hipLaunchKernelGGL((splitk_epilogue_kernel<EPI, T>), egrid, dim3(256), 0, s, ws, pl.S, ep, c, M, N, ldc)
  switch (epilogue) {
    case SANA_EPI_NONE: SANA_SPLIT_EPI(SANA_EPI_NONE); break;
    case SANA_EPI_BIAS: SANA_SPLIT_EPI(SANA_EPI_BIAS); break;
    case SANA_EPI_BIAS_SILU: SANA_SPLIT_EPI(SANA_EPI_BIAS_SILU); break;
    case SANA_EPI_GATE_RES: SANA_SPLIT_EPI(SANA_EPI_GATE_RES); break;
    default: return SANA_ERR_ARG;
  }
#undef SANA_SPLIT_EPI
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

// The pipelined kernel (int8 weights).
template <int NI>
int launch4(const uint16_t* a, const void* W, const float* scale, const EpiArgs& ep, uint16_t* c, int M, int N, int K,
            int64_t lda, int64_t ldw, int64_t ldc, int epilogue, hipStream_t s) {
  const int tiles_t = (M + BT - 1) / BT, tiles_c = (N + 64 * NI - 1) / (64 * NI);
  dim3 grid((unsigned)(tiles_t * tiles_c)), block(256);
  const Taps none = {0, 0, 0, 0, 0, nullptr};
#define SANA_LAUNCH4(EPI)                                                                                                     \
  hipLaunchKernelGGL((gemm4_kernel<EPI, NI>), grid, block, 0, s, a, static_cast<const int8_t*>(W), scale, ep, c, M, N, K, lda, ldw, ldc, \
                     tiles_t, tiles_c, none)
  switch (epilogue) {
    case SANA_EPI_NONE: SANA_LAUNCH4(SANA_EPI_NONE); break;
    case SANA_EPI_BIAS: SANA_LAUNCH4(SANA_EPI_BIAS); break;
    case SANA_EPI_BIAS_SILU: SANA_LAUNCH4(SANA_EPI_BIAS_SILU); break;
    case SANA_EPI_GATE_RES: SANA_LAUNCH4(SANA_EPI_GATE_RES); break;
    default: return SANA_ERR_ARG;
  }
#undef SANA_LAUNCH4
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

// The compiler-scheduled kernel (int8 weights): 64*TT tokens x 64*TC channels.
template <int TT, int TC>
int launch_w8(const uint16_t* a, const void* W, const float* scale, const EpiArgs& ep, uint16_t* c, int M, int N, int K,
              int64_t lda, int64_t ldw, int64_t ldc, int epilogue, hipStream_t s) {
  const int tiles_t = (M + 64 * TT - 1) / (64 * TT), tiles_c = (N + 64 * TC - 1) / (64 * TC);
  dim3 grid((unsigned)(tiles_t * tiles_c)), block(256);
#define SANA_LAUNCH_W8(EPI)                                                                                      \
  hipLaunchKernelGGL((gemm_w8_kernel<EPI, TT, TC>), grid, block, 0, s, a, static_cast<const int8_t*>(W), scale, ep, c, M, N, \
                     K, lda, ldw, ldc, tiles_t, tiles_c)
  switch (epilogue) {
    case SANA_EPI_NONE: SANA_LAUNCH_W8(SANA_EPI_NONE); break;
    case SANA_EPI_BIAS: SANA_LAUNCH_W8(SANA_EPI_BIAS); break;
    case SANA_EPI_BIAS_SILU: SANA_LAUNCH_W8(SANA_EPI_BIAS_SILU); break;
    case SANA_EPI_GATE_RES: SANA_LAUNCH_W8(SANA_EPI_GATE_RES); break;
    default: return SANA_ERR_ARG;
  }
#undef SANA_LAUNCH_W8
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

template <bool W8, typename T = BF16>
int launch(const void* A, const void* W, const float* scale, const EpiArgs& ep, void* C, int M, int N, int K,
           int64_t lda, int64_t ldw, int64_t ldc, int epilogue, hipStream_t s, void* workspace = nullptr,
           size_t workspace_bytes = 0) {
  const int64_t tiles_t = (M + BT - 1) / BT;
  if (tiles_t * ((N + 127) / 128) > (1 << 30)) return SANA_ERR_SHAPE;
  const uint16_t* a = static_cast<const uint16_t*>(A);
  uint16_t* c = static_cast<uint16_t*>(C);
  const GemmPlan pl = plan_gemm(M, N, K, W8);
  float* ws = aligned16(workspace) ? static_cast<float*>(workspace) : nullptr;
  const SplitWay way = ws && workspace_bytes >= split_bytes(pl, M, N) ? split_way(pl, M, N, K) : SplitWay::no;
  if (way == SplitWay::split || (W8 && way == SplitWay::ranges))
    return launch_split<W8, T>(a, W, scale, ep, c, M, N, K, lda, ldw, ldc, epilogue, s, pl, ws);
  if constexpr (!W8) {
    const uint16_t* w = static_cast<const uint16_t*>(W);
    const Plan16 p = plan16(M, N, K, epilogue == SANA_EPI_GATE_RES);
    if (p.n_wide) {
      const int rc = gemm8_launch(a, w, ep, c, M, p.n_wide, K, lda, ldw, ldc, epilogue, is_f16<T>, 4, nullptr, s);
      if (rc != SANA_OK) return rc;
      EpiArgs ep2 = ep;
      if (ep2.bias) ep2.bias += p.n_wide;
      if (ep2.gate) ep2.gate += p.n_wide;
      if (ep2.res) ep2.res += p.n_wide;
      return gemm8_launch(a, w + (int64_t)p.n_wide * ldw, ep2, c + p.n_wide, M, N - p.n_wide, K, lda, ldw, ldc, epilogue,
                          is_f16<T>, 3, nullptr, s);
    }
    if (p.tile->bn == 288 && ldw < kMaxStride288 && aligned16(ep.bias))  // (its bias row is loaded straight to LDS, 16 bytes a lane)
      return gemm288_launch(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, is_f16<T>, nullptr, s);
    if (p.tile->bn == 288) return gemm8_launch(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, is_f16<T>, 4, nullptr, s);
    // 256 x 128 at short k: the persistent kernel, whose next tile loads behind this one's epilogue.  us, ring / here: 16384 x 768 x 64
    // 17.3 / 13.5, 2048 x 3072 x 512 13.2 / 12.5, 16384 x 1536 x 512 36.6 / 33.5, 8192 x 768 x 768 17.4 / 16.4; from K = 1024 on ties or worse
    if (p.tile->bm == 256 && (p.tile->bn >= 192 || K < kShortK))
      return gemm8_launch(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, is_f16<T>, p.tile->bn / 64, nullptr, s);
    return gemm_ring_launch(a, w, ep, c, M, N, K, lda, ldw, ldc, epilogue, is_f16<T>, p.tile->bm, p.bn,
                            way == SplitWay::ranges ? KRanges{pl.tiles, pl.rem, pl.S} : KRanges{0, 0, 1}, s);
  } else {
    const bool pipelined = K % 32 == 0 && K >= 64;
    const int KT = (K + BK - 1) / BK;
    // the 128 x 128 tile where its grid fits one workgroup per compute unit and its chain is the shorter one (plan_gemm)
    if (pl.small || (pl.S > 1 && (int64_t)((M + 127) / 128) * ((N + 127) / 128) <= compute_units() && KT >= 11))
      return launch_w8<2, 2>(a, W, scale, ep, c, M, N, K, lda, ldw, ldc, epilogue, s);
    if (!pipelined) return launch_w8<4, 4>(a, W, scale, ep, c, M, N, K, lda, ldw, ldc, epilogue, s);
    // Few tokens, wide N (qkv of one 1024 px image: 4 x 35 tiles of 192 channels on 256 CUs): 128-wide tiles put
    // half as much math behind every k-tile of the chain and fill more of the chip (4 x 53 workgroups).
    // Taken when the 192-wide grid leaves a fifth of the CUs idle and the 128-wide one still fits.
    const int64_t t128 = tiles_t * ((N + 127) / 128), t192 = tiles_t * ((N + 191) / 192);
    if (t128 <= compute_units() && t192 < compute_units() * 4 / 5)
      return launch4<2>(a, W, scale, ep, c, M, N, K, lda, ldw, ldc, epilogue, s);
    return pick_ni(M, N) == 3 ? launch4<3>(a, W, scale, ep, c, M, N, K, lda, ldw, ldc, epilogue, s)
                              : launch4<4>(a, W, scale, ep, c, M, N, K, lda, ldw, ldc, epilogue, s);
  }
}

// Row strides from which the 32-bit offsets inside a tile's 256 rows could overflow.
constexpr int64_t kMaxTileStride = 1 << 22;

int check_common(const void* A, const void* W, const void* bias, const void* C, int M, int N, int K, int64_t lda,
                 int64_t ldw, int64_t ldc, int epilogue, int kmult, int ldw_mult) {
  if (!A || !W || !C || M <= 0 || N <= 0 || K <= 0) return SANA_ERR_ARG;
  if ((epilogue == SANA_EPI_BIAS || epilogue == SANA_EPI_BIAS_SILU) && !bias) return SANA_ERR_ARG;
  if (epilogue < SANA_EPI_NONE || epilogue > SANA_EPI_GATE_RES) return SANA_ERR_ARG;
  if (K % kmult || N % 8) return SANA_ERR_SHAPE;
  if (lda < K || ldw < K || ldc < N) return SANA_ERR_ARG;
  if (lda >= kMaxTileStride || ldw >= kMaxTileStride || ldc >= kMaxTileStride) return SANA_ERR_SHAPE;
  if (lda % 8 || ldw % ldw_mult || ldc % 8 || !aligned16(A) || !aligned16(W) || !aligned16(C)) return SANA_ERR_ALIGN;
  return SANA_OK;
}

int check_gate_res(const void* gate, const void* residual, int M, int N, int64_t ldr, int rows_per_gate,
                   int64_t gate_stride) {
  if (!gate || !residual || rows_per_gate <= 0) return SANA_ERR_ARG;
  if (ldr < N || gate_stride < 0) return SANA_ERR_ARG;
  if (ldr % 8 || gate_stride % 8 || !aligned16(gate) || !aligned16(residual)) return SANA_ERR_ALIGN;
  return SANA_OK;
}

// C = residual + gate * (A . W^T + bias).  Rows of the residual further apart than a tile's offsets reach (one token of each
// of many long sequences, say) are added by the elementwise kernel, whose addresses have 64 bits, on the linear output in C:
// the same three roundings.
template <bool W8, typename T = BF16>
int launch_gate_res(const void* A, const void* W, const float* scale, EpiArgs e, void* C, int M, int N, int K, int64_t lda,
                    int64_t ldw, int64_t ldc, void* stream, void* workspace, size_t workspace_bytes) {
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (M == 1) e.ldr = N;  // a single row has no stride (and may be C itself)
  if (e.ldr < kMaxTileStride)
    return launch<W8, T>(A, W, scale, e, C, M, N, K, lda, ldw, ldc, SANA_EPI_GATE_RES, s, workspace, workspace_bytes);
  EpiArgs lin = e;
  lin.gate = lin.res = nullptr, lin.ldr = lin.gate_stride = 0;
  const int rc = launch<W8, T>(A, W, scale, lin, C, M, N, K, lda, ldw, ldc, SANA_EPI_BIAS, s, workspace, workspace_bytes);
  return rc != SANA_OK ? rc
                       : sana_hip_gate_residual(C, e.gate, e.res, C, M, N, ldc, e.ldr, ldc, e.rows_per_gate, e.gate_stride,
                                                is_f16<T> ? SANA_DT_F16 : SANA_DT_BF16, stream);
}

// Sum of the per-token-tile partial states of the fused qkv projection: part[bh][nsplit][33 * 32] -> state[bh][33 * 32].
// One thread per element of one (batch, head) adds G-th tiles in tile order (batches of eight independent loads);
// with G = 4 (many tiles per batch entry) four threads share an element and their sums are added in a fixed order.
// Deterministic either way.
template <int G>
__global__ __launch_bounds__(256) void qkv_state_reduce_kernel(const float* __restrict__ part, float* __restrict__ state,
                                                                int nsplit, int total) {
  constexpr int ELEMS = 33 * 32, PER = 256 / G;
  __shared__ float red[G][PER];
  const int local = threadIdx.x % PER, grp = threadIdx.x / PER;
  const int gid = blockIdx.x * PER + local;  // element of the whole state array
  float s = 0.f;
  if (gid < total) {
    const int bh = gid / ELEMS, e = gid - bh * ELEMS;
    const float* p = part + ((int64_t)bh * nsplit) * ELEMS + e;
    for (int sp0 = grp; sp0 < nsplit; sp0 += 8 * G) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = (sp0 + G * u < nsplit) ? p[(int64_t)(sp0 + G * u) * ELEMS] : 0.f;
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
  }
  if (G == 1) {
    if (gid < total) state[gid] = s;
    return;
  }
  red[grp][local] = s;
  __syncthreads();
  if (grp == 0 && gid < total) {
    float t = red[0][local];
#pragma unroll
    for (int g = 1; g < G; ++g) t += red[g][local];
    state[gid] = t;
  }
}

// Rows of the fused qkv projection's weight layout for C = 32 * heads channels: the q rows padded to whole 256-wide
// tiles, then one tile per four heads, [K h | V h | K h+1 | V h+1] for the tile's first and second pair of heads.
int qkv_state_q_pad(int C) { return (C + 255) / 256 * 256; }
int qkv_state_rows_total(int C, int heads) { return qkv_state_q_pad(C) + (heads + 3) / 4 * 256; }

EpiArgs plain_epi(const void* bias) {
  EpiArgs e = {static_cast<const uint16_t*>(bias), nullptr, nullptr, 0, 0, 1, nullptr, 0, 0, 0, 0};
  return e;
}

}  // namespace
}  // namespace sana

using namespace sana;

#define SANA_API extern "C" __attribute__((visibility("default")))

SANA_API size_t sana_hip_gemm_workspace_bytes(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || N % 8) return 0;
  const GemmPlan pl = plan_gemm(M, N, K, false);
  return split_pays(pl, M, N, K) ? split_bytes(pl, M, N) : 0;
}

SANA_API int sana_hip_gemm_plan(int M, int N, int K, int plan[4]) {
  if (!plan || M <= 0 || N <= 0 || K <= 0) return SANA_ERR_ARG;
  if (N % 8 || K % 8) return SANA_ERR_SHAPE;
  const GemmPlan split = plan_gemm(M, N, K, false);
  const Plan16 p = plan16(M, N, K);
  const SplitWay way = split_way(split, M, N, K);
  const bool cut = way == SplitWay::split;
  plan[0] = cut ? BT : p.tile->bm, plan[1] = cut ? 64 * pick_ni(M, N) : p.bn;
  plan[2] = cut ? 0 : p.n_wide, plan[3] = way == SplitWay::no ? 1 : split.S;
  return SANA_OK;
}

// From 4096 rows on always (converting in the main loop costs it 14 % at every M, the expansion a fixed 5 - 16 us); below that, of GEMMs that
// are not split, where
//  * N <= K: there the bf16 GEMM has its small tiles and the int8 one a chain of long k-tiles.  us, converting / expanding (the weights of
//    12 calls in turn): 256 x 1152 x 2880 37 / 20, 2048 x 2240 x 2240 36 / 32, 2048 x 2240 x 5600 91 / 79; split 1024 x 2240 x 5600 45 / 54;
//  * the int8 tiles need a second round: 1536 x 11200 x 2240 98 / 82, 2916 x 5760 x 1152 57 / 49, 3584 x 5760 x 1152 59.1 / 58.4;
//  * long rows of weights meet more than six token tiles: 1600 x 6720 x 2240 55.2 / 54.4, 2048 x 6720 x 2240 64 / 59, 2300 x 4480 x 2240 53 / 49; but
//    1024 x 11200 x 2240 58 / 60, 2048 x 5760 x 1152 33 / 38, 3072 x 3456 x 1152 30 / 33.
SANA_API int sana_hip_gemm_w8_expand(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  if (M >= 4096) return 1;
  const int64_t tiles = (int64_t)((M + BT - 1) / BT) * ((N + 64 * pick_ni(M, N) - 1) / (64 * pick_ni(M, N)));
  return (N <= K || tiles > compute_units() || (K >= 2048 && M > 6 * BT)) && !split_pays(plan_gemm(M, N, K, true), M, N, K);
}

SANA_API int sana_hip_gemm_bf16(const void* A, const void* W, const void* bias, void* C, int M, int N, int K,
                                int64_t lda, int64_t ldw, int64_t ldc, int epilogue, void* workspace,
                                size_t workspace_bytes, void* stream) {
  if (epilogue == SANA_EPI_GATE_RES) return SANA_ERR_ARG;
  const int rc = check_common(A, W, bias, C, M, N, K, lda, ldw, ldc, epilogue, 8, 8);
  if (rc != SANA_OK) return rc;
  return launch<false>(A, W, nullptr, plain_epi(bias), C, M, N, K, lda, ldw, ldc, epilogue,
                       static_cast<hipStream_t>(stream), workspace, workspace_bytes);
}

SANA_API int sana_hip_gemm_f16(const void* A, const void* W, const void* bias, void* C, int M, int N, int K,
                               int64_t lda, int64_t ldw, int64_t ldc, int epilogue, void* workspace,
                               size_t workspace_bytes, void* stream) {
  if (epilogue == SANA_EPI_GATE_RES) return SANA_ERR_ARG;
  const int rc = check_common(A, W, bias, C, M, N, K, lda, ldw, ldc, epilogue, 8, 8);
  if (rc != SANA_OK) return rc;
  return launch<false, F16>(A, W, nullptr, plain_epi(bias), C, M, N, K, lda, ldw, ldc, epilogue,
                            static_cast<hipStream_t>(stream), workspace, workspace_bytes);
}

SANA_API int sana_hip_gemm_w8a16(const void* A, const int8_t* Wq, const float* scale, const void* bias, void* C,
                                 int M, int N, int K, int64_t lda, int64_t ldw, int64_t ldc, int epilogue,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  if (!scale || epilogue == SANA_EPI_GATE_RES) return SANA_ERR_ARG;
  const int rc = check_common(A, Wq, bias, C, M, N, K, lda, ldw, ldc, epilogue, 16, 16);
  if (rc != SANA_OK) return rc;
  return launch<true>(A, Wq, scale, plain_epi(bias), C, M, N, K, lda, ldw, ldc, epilogue,
                      static_cast<hipStream_t>(stream), workspace, workspace_bytes);
}

SANA_API int sana_hip_gemm_gate_residual(const void* A, const void* W, const float* w8_scale, const void* bias,
                                         const void* gate, const void* residual, void* C, int M, int N, int K,
                                         int64_t lda, int64_t ldw, int64_t ldr, int64_t ldc, int rows_per_gate,
                                         int64_t gate_stride, void* workspace, size_t workspace_bytes,
                                         void* stream) {
  const bool w8 = w8_scale != nullptr;
  int rc = check_common(A, W, bias, C, M, N, K, lda, ldw, ldc, SANA_EPI_GATE_RES, w8 ? 16 : 8, w8 ? 16 : 8);
  if (rc != SANA_OK) return rc;
  rc = check_gate_res(gate, residual, M, N, ldr, rows_per_gate, gate_stride);
  if (rc != SANA_OK) return rc;
  const EpiArgs e = {static_cast<const uint16_t*>(bias), static_cast<const uint16_t*>(gate),
                     static_cast<const uint16_t*>(residual), ldr, gate_stride, rows_per_gate, nullptr, 0, 0, 0, 0};
  return w8 ? launch_gate_res<true>(A, W, w8_scale, e, C, M, N, K, lda, ldw, ldc, stream, workspace, workspace_bytes)
            : launch_gate_res<false>(A, W, nullptr, e, C, M, N, K, lda, ldw, ldc, stream, workspace, workspace_bytes);
}

SANA_API int sana_hip_gemm_gate_residual_f16(const void* A, const void* W, const void* bias, const void* gate,
                                             const void* residual, void* C, int M, int N, int K, int64_t lda,
                                             int64_t ldw, int64_t ldr, int64_t ldc, int rows_per_gate,
                                             int64_t gate_stride, void* workspace, size_t workspace_bytes,
                                             void* stream) {
  int rc = check_common(A, W, bias, C, M, N, K, lda, ldw, ldc, SANA_EPI_GATE_RES, 8, 8);
  if (rc != SANA_OK) return rc;
  rc = check_gate_res(gate, residual, M, N, ldr, rows_per_gate, gate_stride);
  if (rc != SANA_OK) return rc;
  const EpiArgs e = {static_cast<const uint16_t*>(bias), static_cast<const uint16_t*>(gate),
                     static_cast<const uint16_t*>(residual), ldr, gate_stride, rows_per_gate, nullptr, 0, 0, 0, 0};
  return launch_gate_res<false, F16>(A, W, nullptr, e, C, M, N, K, lda, ldw, ldc, stream, workspace, workspace_bytes);
}

SANA_API int sana_hip_tconv_residual(const void* X, const void* W, void* out, int M, int C, int taps,
                                     int64_t tap_rows, int64_t x_rows, const unsigned char* zero_last_tap,
                                     int64_t ldx, int64_t ldw, int64_t ldo, void* stream) {
  if (!X || !W || !out || M <= 0 || C <= 0 || taps <= 0 || !(taps & 1) || tap_rows <= 0) return SANA_ERR_ARG;
  if (zero_last_tap && taps < 3) return SANA_ERR_ARG;
  if (C % 64) return SANA_ERR_SHAPE;  // a tap is a whole number of k-tiles
  if (x_rows < (taps / 2) * tap_rows + M) return SANA_ERR_ARG;  // the centre tap (= the residual) must exist for every row
  if (ldx < C || ldw < (int64_t)taps * C || ldo < C) return SANA_ERR_ARG;
  if (ldx % 8 || ldw % 8 || ldo % 8 || !aligned16(X) || !aligned16(W) || !aligned16(out)) return SANA_ERR_ALIGN;
  if (x_rows * ldx * 2 >= ((int64_t)1 << 31)) return SANA_ERR_SHAPE;  // 32-bit byte offsets inside the buffer
  if (M == 1) ldo = C;  // a single row has no stride
  if (ldo >= 2 * kMaxTileStride) return SANA_ERR_SHAPE;  // .. and inside the 128 rows of out that a wave stores
  const uint16_t* x = static_cast<const uint16_t*>(X);
  const EpiArgs e = {nullptr, nullptr, x + (taps / 2) * tap_rows * ldx, ldx, 0, M, nullptr, 0, 0, 0, 0};
  const Taps tp = {C, tap_rows, x_rows, 0, 0, zero_last_tap};
  const uint16_t* w = static_cast<const uint16_t*>(W);
  uint16_t* o = static_cast<uint16_t*>(out);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // one of the three widest tiles: the others have no taps
  const int k = taps * C;
  const bool brief = k < kShortK, may288 = ldw < kMaxStride288;
  // (192 channels at the price that they have in every GEMM; with 7.9, what its fixed part was, / so: 39680 x 1152 taken from 288 channels 265 / 252,
  // 50160 x 1152 320 / 316, 55760 x 1536 from 256 channels 606 / 596; 27 shapes 0.96 .. 1.00; at 2240 channels the choice is the same)
  const double us192 = cost16(brief ? kTilesShort[1] : kTiles16[kTile192], M, C, k);
  const double us256 = cost16(brief ? kTilesShort[2] : kTiles16[kTile256], M, C, k), us = std::min(us192, us256);
  if (may288 && (brief ? short_takes_288(M, C, k, us) : cost16(kTiles16[kTile288], M, C, k) < us))
    return gemm288_launch(x, w, e, o, M, C, k, ldx, ldw, ldo, SANA_EPI_GATE_RES, false, &tp, s);
  return gemm8_launch(x, w, e, o, M, C, k, ldx, ldw, ldo, SANA_EPI_GATE_RES, false, us192 < us256 ? 3 : 4, &tp, s);
}

SANA_API int sana_hip_dequant_w8(const int8_t* Wq, const float* scale, void* W, int N, int K, int64_t ldw,
                                 int64_t ldo, void* stream) {
  if (!Wq || !scale || !W || N <= 0 || K <= 0) return SANA_ERR_ARG;
  if (K % 16) return SANA_ERR_SHAPE;
  if (ldw < K || ldo < K) return SANA_ERR_ARG;
  if (ldw % 16 || ldo % 8 || !aligned16(Wq) || !aligned16(W)) return SANA_ERR_ALIGN;
  if ((int64_t)N * (K / 16) > (int64_t)0x7fffffff * 256) return SANA_ERR_SHAPE;
  const unsigned rows = ((unsigned)N + 3) / 4, y = std::min(rows, 1u << 15);
  hipLaunchKernelGGL(dequant_w8_kernel, dim3(((unsigned)K + 511) / 512, y, (rows + y - 1) / y), dim3(256), 0,
                     static_cast<hipStream_t>(stream), Wq, scale, static_cast<uint16_t*>(W), N, K, ldw, ldo);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}

SANA_API int sana_hip_qkv_state_rows(int C, int heads, int32_t* rows, int capacity) {
  if (C <= 0 || heads <= 0 || C != 32 * heads) return SANA_ERR_SHAPE;
  const int q_pad = qkv_state_q_pad(C), total = qkv_state_rows_total(C, heads);
  if (!rows) return total;
  if (capacity < total) return SANA_ERR_ARG;
  for (int i = 0; i < q_pad; ++i) rows[i] = i < C ? i : -1;
  for (int i = q_pad; i < total; ++i) {
    const int l = (i - q_pad) & 255, tile = (i - q_pad) >> 8;
    const int head = 4 * tile + 2 * (l >> 7) + ((l >> 6) & 1), is_v = (l >> 5) & 1, e = l & 31;
    rows[i] = head < heads ? (1 + is_v) * C + 32 * head + e : -1;
  }
  return total;
}

SANA_API size_t sana_hip_gemm_qkv_state_workspace_bytes(int B, int N, int heads) {
  if (B <= 0 || N <= 0 || heads <= 0 || (N % 256 && B != 1)) return 0;
  return (size_t)B * heads * ((N + 255) / 256) * 33 * 32 * sizeof(float);
}

SANA_API int sana_hip_gemm_qkv_state(const void* A, const void* W_tiled, const void* bias_tiled, void* Q, float* state,
                                     void* workspace, size_t workspace_bytes, int B, int N, int C, int heads,
                                     int64_t lda, int64_t ldw, int64_t ldq, void* stream) {
  if (!A || !W_tiled || !Q || !state || B <= 0 || N <= 0 || C <= 0 || heads <= 0) return SANA_ERR_ARG;
  if (C != 32 * heads || C < 64) return SANA_ERR_SHAPE;
  // a token tile must not straddle two batch entries, and the rows of a ragged last tile must contribute nothing to
  // the state: they read as zero activations, which stay zero only without a bias
  if (N % 256 && (B != 1 || bias_tiled)) return SANA_ERR_SHAPE;
  if ((int64_t)B * N >= ((int64_t)1 << 30) || (int64_t)B * heads * 33 * 32 >= ((int64_t)1 << 31)) return SANA_ERR_SHAPE;
  const int M = B * N, rows_t = qkv_state_rows_total(C, heads);
  if (lda < C || ldw < C || ldq < C) return SANA_ERR_ARG;
  if (lda >= (1 << 22) || ldw >= (1 << 22) || ldq >= (1 << 22)) return SANA_ERR_SHAPE;
  if (lda % 8 || ldw % 8 || ldq % 8 || !aligned16(A) || !aligned16(W_tiled) || !aligned16(Q) ||
      (bias_tiled && !aligned16(bias_tiled)) || !aligned16(state))
    return SANA_ERR_ALIGN;
  const size_t need = sana_hip_gemm_qkv_state_workspace_bytes(B, N, heads);
  if (!workspace || workspace_bytes < need) return SANA_ERR_WORKSPACE;
  if (!aligned16(workspace)) return SANA_ERR_ALIGN;
  const int64_t tiles_t = (M + BT - 1) / BT, tiles_c = rows_t / 256;
  if (tiles_t * tiles_c > (1 << 30)) return SANA_ERR_SHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const EpiArgs e = {static_cast<const uint16_t*>(bias_tiled), nullptr, nullptr, 0, 0, 1, static_cast<float*>(workspace),
                     C, qkv_state_q_pad(C), heads, (N + 255) / 256};
  const int rc = gemm8_launch(static_cast<const uint16_t*>(A), static_cast<const uint16_t*>(W_tiled), e, static_cast<uint16_t*>(Q),
                              M, rows_t, C, lda, ldw, ldq, SANA_EPI_QKV_STATE, false, 4, nullptr, s);
  if (rc != SANA_OK) return rc;
  const int total = B * heads * 33 * 32, nsplit = (N + 255) / 256;
  if (nsplit > 16)
    hipLaunchKernelGGL(qkv_state_reduce_kernel<4>, dim3((unsigned)((total + 63) / 64)), dim3(256), 0, s,
                       static_cast<const float*>(workspace), state, nsplit, total);
  else
    hipLaunchKernelGGL(qkv_state_reduce_kernel<1>, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       static_cast<const float*>(workspace), state, nsplit, total);
  return hipGetLastError() == hipSuccess ? SANA_OK : SANA_ERR_LAUNCH;
}
