// One image block (SanaMSBlock, 16-bit weights) as one call: the launches of the entry points below, in order, on one
// scratch buffer.  No kernels of its own.  A block is eleven launches (4 - 14 us each at a few hundred tokens), plus up to two where
// the attention is not one launch and one for each GEMM in two widths or split over k, and issuing them one by one from Python
// took 220 us per block where the device needs about 100.
#include <algorithm>

#include "common.h"

namespace {

struct Layout {  // byte offsets into the scratch buffer
  size_t h, wide, o, x1, x2, y, ws, total, ws_bytes;  // o and x1: inside wide
};

bool plan(const sana_block_args& a, Layout& l) {
  if (a.B <= 0 || a.N <= 0 || a.C <= 0 || a.hidden <= 0 || a.C % 32) return false;
  const size_t M = (size_t)a.B * a.N;
  if (M > 0x7fffffff) return false;
  const int heads = a.C / 32, rows = (int)M;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t p = at;
    at += (bytes + 255) & ~(size_t)255;
    return p;
  };
  // The attention's output and the sum behind it lie behind q, k and v and are dead when the hidden pairs are written: 9.5 C
  // values per token at 2.5 C hidden channels, what the calls one by one hold (h, x2, the pairs, the gated values).  A step of
  // 8 blocks at 256 x 1152 bf16 / 2048 x 1152 f16, us: this 835 / 1462, all buffers side by side (11.5 C) 833 / 1462, the gated
  // values on h, o and x1 (9 C) 845 / 1498.
  const size_t row = (M * a.C * 2 + 255) & ~(size_t)255;
  l.h = take(row);                                                     // normalised input; cross-attention's queries
  l.wide = take(std::max(5 * row, M * 4 * (size_t)a.hidden));          // q, k, v; the Mix-FFN's hidden pairs
  l.o = l.wide + 3 * row;                                              // attention outputs
  l.x1 = l.o + row;                                                    // behind the attention
  l.x2 = take(row);                                                    // behind the cross-attention
  l.y = take(M * a.hidden * 2);                                        // gated hidden values
  l.ws_bytes = sana_hip_linattn_scratch_bytes(a.B, a.N, heads, 32, a.io_dtype);
  if (a.split_k)
    for (size_t b : {sana_hip_gemm_workspace_bytes(rows, 3 * a.C, a.C), sana_hip_gemm_workspace_bytes(rows, a.C, a.C),
                     sana_hip_gemm_workspace_bytes(rows, 2 * a.hidden, a.C), sana_hip_gemm_workspace_bytes(rows, a.C, a.hidden)})
      l.ws_bytes = std::max(l.ws_bytes, b);
  l.ws = take(l.ws_bytes);
  l.total = at;
  return true;
}

}  // namespace

#define SANA_API extern "C" __attribute__((visibility("default")))

SANA_API size_t sana_hip_block_scratch_bytes(const sana_block_args* args) {
  Layout l;
  return args && plan(*args, l) ? l.total : 0;
}

SANA_API int sana_hip_block(const sana_block_args* args, void* stream) {
  if (!args) return SANA_ERR_ARG;
  const sana_block_args& a = *args;
  Layout l;
  if (!plan(a, l) || a.H <= 0 || a.W <= 0 || (int64_t)a.H * a.W != a.N || a.cross_heads <= 0) return SANA_ERR_ARG;
  if (a.io_dtype != SANA_DT_BF16 && a.io_dtype != SANA_DT_F16) return SANA_ERR_DTYPE;
  if (a.C % a.cross_heads) return SANA_ERR_SHAPE;
  if (!a.scratch || a.scratch_bytes < l.total) return SANA_ERR_WORKSPACE;
  // everything is checked before the first launch: what the entry points below would refuse in the middle
  for (const void* p : {a.x, a.text_kv, a.shift_msa, a.scale_msa, a.gate_msa, a.shift_mlp, a.scale_mlp, a.gate_mlp, a.qkv_w,
                        a.proj_w, a.proj_b, a.q_w, a.q_b, a.o_w, a.o_b, a.ones, a.inv_w, a.inv_b, a.dw_w, a.point_w,
                        (const void*)a.out})
    if (!p) return SANA_ERR_ARG;
  for (const void* p : {a.x, a.text_kv, a.shift_msa, a.scale_msa, a.gate_msa, a.shift_mlp, a.scale_mlp, a.gate_mlp, a.qkv_w,
                        a.qkv_b, a.proj_w, a.proj_b, a.q_w, a.q_b, a.o_w, a.o_b, a.ones, a.inv_w, a.inv_b, a.dw_w, a.dw_b,
                        a.point_w, a.point_b, (const void*)a.out, (const void*)a.scratch})
    if (!sana::aligned16(p)) return SANA_ERR_ALIGN;
  const int d = a.C / a.cross_heads;
  if (d <= 64 || d > 112 || d % 8 || a.text_len <= 0 || a.text_len > 320 || a.C % 8 || a.C > 8192 || a.hidden % 8)
    return SANA_ERR_SHAPE;
  if (a.text_ld < 2 * (int64_t)a.C || (a.key_bias && a.key_bias_ld < a.text_len) || a.mod_stride < 0) return SANA_ERR_ARG;
  if (a.text_ld % 8 || a.mod_stride % 8) return SANA_ERR_ALIGN;

  const int M = a.B * a.N, C = a.C, heads = C / 32, hid = a.hidden, dt = a.io_dtype;
  const bool f16 = dt == SANA_DT_F16;
  char* s = static_cast<char*>(a.scratch);
  void *h = s + l.h, *wide = s + l.wide, *o = s + l.o, *x1 = s + l.x1, *x2 = s + l.x2, *y = s + l.y;
  void* ws = l.ws_bytes ? s + l.ws : nullptr;
  void* gws = a.split_k ? ws : nullptr;
  auto gemm = [&](const void* A, const void* W, const void* bias, void* out, int N, int K, int epi) {
    return (f16 ? sana_hip_gemm_f16 : sana_hip_gemm_bf16)(A, W, bias, out, M, N, K, K, K, N, epi, gws, gws ? l.ws_bytes : 0, stream);
  };
  auto gated = [&](const void* A, const void* W, const void* bias, const void* gate, int64_t stride, const void* res, void* out, int K) {
    return f16 ? sana_hip_gemm_gate_residual_f16(A, W, bias, gate, res, out, M, C, K, K, K, C, C, a.N, stride, gws,
                                                 gws ? l.ws_bytes : 0, stream)
               : sana_hip_gemm_gate_residual(A, W, nullptr, bias, gate, res, out, M, C, K, K, K, C, C, a.N, stride, gws,
                                             gws ? l.ws_bytes : 0, stream);
  };
#define SANA_DO(call)              \
  do {                             \
    const int rc = (call);         \
    if (rc != SANA_OK) return rc;  \
  } while (0)
  // x1 = x + gate * proj(attention(modulate(norm1(x))))
  SANA_DO(sana_hip_layernorm_modulate(a.x, a.scale_msa, a.shift_msa, h, M, C, C, C, a.N, a.mod_stride, a.eps_norm1, dt, stream));
  SANA_DO(gemm(h, a.qkv_w, a.qkv_b, wide, 3 * C, C, a.qkv_b ? SANA_EPI_BIAS : SANA_EPI_NONE));
  const char* qkv = static_cast<const char*>(wide);
  const int64_t sb = a.B > 1 ? (int64_t)a.N * 3 * C : 0, ob = a.B > 1 ? (int64_t)a.N * C : 0;
  SANA_DO(sana_hip_linattn(qkv, qkv + 2 * (size_t)C, qkv + 4 * (size_t)C, o, ws, l.ws_bytes, a.B, a.N, heads, 32, sb, 3 * C, sb,
                           3 * C, ob, C, a.eps_attn, dt, stream));
  SANA_DO(gated(o, a.proj_w, a.proj_b, a.gate_msa, a.mod_stride, a.x, x1, C));
  // x2 = x1 + cross_attention(x1)
  SANA_DO(gemm(x1, a.q_w, a.q_b, h, C, C, SANA_EPI_BIAS));
  SANA_DO((f16 ? sana_hip_cross_attention_f16 : sana_hip_cross_attention)(
      h, a.text_kv, a.key_bias, o, a.B, a.N, a.text_len, a.cross_heads, d, C, a.text_ld, C, a.key_bias ? a.key_bias_ld : 0,
      a.cross_scale, stream));
  SANA_DO(gated(o, a.o_w, a.o_b, a.ones, 0, x1, x2, C));
  // out = x2 + gate * mix_ffn(modulate(norm2(x2)))
  SANA_DO(sana_hip_layernorm_modulate(x2, a.scale_mlp, a.shift_mlp, h, M, C, C, C, a.N, a.mod_stride, a.eps_norm2, dt, stream));
  SANA_DO(gemm(h, a.inv_w, a.inv_b, wide, 2 * hid, C, SANA_EPI_BIAS_SILU));
  SANA_DO(sana_hip_dwconv3x3_silu_gate(wide, a.dw_w, a.dw_b, y, a.B, a.H, a.W, hid, a.round_like_reference, dt, stream));
  SANA_DO(gated(y, a.point_w, a.point_b, a.gate_mlp, a.mod_stride, x2, a.out, hid));
#undef SANA_DO
  return SANA_OK;
}
