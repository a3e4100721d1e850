// One encoder layer as one host call: the launches of the projections, the
// attention and the output blocks, in order, on the caller's stream.
//
// No kernel of its own.  A forward of few tokens is bound by the host: from Python
// every launch costs 8-13 us (argument checks, allocations, ctypes), about 80 us a
// layer for 45 us of kernels.  Here a launch costs the runtime's own 2 us.

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dflash.h"

namespace {

constexpr size_t kAlign = 256;

size_t padded(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

// Intermediates of a layer in the workspace.  `scratch` serves the attention's partial
// rows and both output blocks, one after the other.
struct Layout {
  size_t qkv, context, attended, inner, scratch, scratch_bytes, total;
  int splits;
  size_t attention_bytes;
};

int plan(const dflash_encoder_layer& p, int B, int L, Layout* out) {
  const int64_t rows = static_cast<int64_t>(B) * L;
  const size_t row = static_cast<size_t>(rows) * 2;  // 16-bit elements
  const int width = p.heads * p.head_dim;
  Layout l{};
  l.splits = 0;
  const int rc = dflash_attention_rel_split_plan(B, p.heads, L, p.head_dim, &l.splits,
                                                 &l.attention_bytes);
  if (rc != DFLASH_OK) return rc;
  const size_t first = dflash_output_block_workspace_bytes(static_cast<int>(rows), p.hidden, width);
  const size_t second =
      dflash_output_block_workspace_bytes(static_cast<int>(rows), p.hidden, p.inner);
  l.scratch_bytes = l.attention_bytes > first ? l.attention_bytes : first;
  if (second > l.scratch_bytes) l.scratch_bytes = second;
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t here = at;
    at += padded(bytes);
    return here;
  };
  l.qkv = take(row * 3 * width);
  l.context = take(row * width);
  l.attended = take(row * p.hidden);
  l.inner = take(row * p.inner);
  l.scratch = take(l.scratch_bytes);
  l.total = at;
  *out = l;
  return DFLASH_OK;
}

int check(const dflash_encoder_layer* p, int B, int L) {
  if (!p) return DFLASH_ERR_NULL;
  if (B < 0 || L < 1 || p->heads < 1 || p->head_dim < 1 || p->hidden < 1 || p->inner < 1)
    return DFLASH_ERR_SHAPE;
  if (p->head_dim != 32 && p->head_dim != 64 && p->head_dim != 128) return DFLASH_ERR_HEAD_DIM;
  if (p->dtype != DFLASH_DTYPE_FP16 && p->dtype != DFLASH_DTYPE_BF16) return DFLASH_ERR_DTYPE;
  if (static_cast<int64_t>(B) * L >= (int64_t{1} << 24)) return DFLASH_ERR_TOO_LARGE;
  return DFLASH_OK;
}

}  // namespace

extern "C" size_t dflash_encoder_layer_workspace_bytes(const dflash_encoder_layer* layer, int B,
                                                       int L) {
  if (check(layer, B, L) != DFLASH_OK || B == 0) return 0;
  Layout l;
  return plan(*layer, B, L, &l) == DFLASH_OK ? l.total : 0;
}

extern "C" int dflash_encoder_layer_fwd(const dflash_encoder_layer* layer, const void* x,
                                        const uint8_t* mask, void* out, int B, int L,
                                        void* workspace, size_t workspace_bytes, void* stream) {
  int rc = check(layer, B, L);
  if (rc != DFLASH_OK) return rc;
  if (B == 0) return DFLASH_OK;
  if (!x || !mask || !out || !workspace) return DFLASH_ERR_NULL;
  const dflash_encoder_layer& p = *layer;
  Layout l;
  rc = plan(p, B, L, &l);
  if (rc != DFLASH_OK) return rc;
  if (workspace_bytes < l.total) return DFLASH_ERR_WORKSPACE;
  if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0) return DFLASH_ERR_ALIGN;
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  const int rows = B * L;
  const int width = p.heads * p.head_dim;
  unsigned char* qkv = ws + l.qkv;
  unsigned char* scratch = ws + l.scratch;
  rc = dflash_linear_fwd(x, p.qkv_weight, p.qkv_bias, nullptr, qkv, rows, 3 * width, p.hidden,
                         DFLASH_GEMM_BIAS, p.dtype, stream);
  if (rc != DFLASH_OK) return rc;
  const size_t part = static_cast<size_t>(width) * 2;
  rc = dflash_attention_rel_fwd_split(
      qkv, qkv + part, qkv + 2 * part, static_cast<int64_t>(L) * 3 * width, p.head_dim, 3 * width,
      p.pos_key, p.pos_query, p.delta_to_local, mask, ws + l.context, B, p.heads, L, p.head_dim,
      p.slots, p.score_scale_log2, p.pos_key != nullptr, p.pos_query != nullptr, p.dtype, 1,
      l.splits, scratch, l.attention_bytes, stream);
  if (rc != DFLASH_OK) return rc;
  rc = dflash_output_block_fwd(ws + l.context, p.attention_weight, p.attention_bias, x,
                               p.attention_gamma, p.attention_beta, ws + l.attended, rows, p.hidden,
                               width, p.attention_eps, p.dtype, scratch, l.scratch_bytes, stream);
  if (rc != DFLASH_OK) return rc;
  rc = dflash_linear_fwd(ws + l.attended, p.inner_weight, p.inner_bias, nullptr, ws + l.inner, rows,
                         p.inner, p.hidden, DFLASH_GEMM_BIAS_GELU, p.dtype, stream);
  if (rc != DFLASH_OK) return rc;
  return dflash_output_block_fwd(ws + l.inner, p.output_weight, p.output_bias, ws + l.attended,
                                 p.output_gamma, p.output_beta, out, rows, p.hidden, p.inner,
                                 p.output_eps, p.dtype, scratch, l.scratch_bytes, stream);
}
