// One layer of the paged hot path in one host call: KV append (RoPE optionally fused), decode + merge,
// prefill, in that order on one stream (reference TorchRefBackend.forward = write_kv + paged_attention,
// src/minillm/attention/torch_ref.py:46-48).  The launches and their results are those of the separate
// entry points; what changes is the host's cost per layer, one foreign call instead of three or four.
#include "common.h"

extern "C" int mllm_attention_forward(const mllm_layer_step* s, const void* q, int64_t q_stride_tok,
                                      int64_t q_stride_head, const void* k, int64_t k_stride_tok,
                                      int64_t k_stride_head, const void* v, int64_t v_stride_tok,
                                      int64_t v_stride_head, const void* cos, const void* sin, int64_t cs_stride_tok,
                                      void* q_rot, void* k_cache, void* v_cache, float k_scale, float v_scale,
                                      void* out, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(s, MLLM_ERR_INVALID, "mllm_attention_forward: null step");
  MLLM_REQUIRE(s->kv_fp8 || (k_scale == 1.f && v_scale == 1.f), MLLM_ERR_INVALID,
               "mllm_attention_forward: k_scale / v_scale apply to fp8 pools only");
  MLLM_REQUIRE(!cos == !sin && (!cos || q_rot), MLLM_ERR_INVALID,
               "mllm_attention_forward: cos, sin and q_rot go together");
  const bool fp8 = s->kv_fp8 != 0;
  const int64_t slots = s->num_blocks * s->block_size;
  const int64_t row = (int64_t)s->num_heads * s->head_dim;  // q_rot and out: contiguous [N, H, Dh]
  int rc;
  const void* qa = q;
  int64_t qa_st = q_stride_tok, qa_sh = q_stride_head;
  if (cos) {
    rc = fp8 ? mllm_rope_kv_append_fp8(q, q_stride_tok, q_stride_head, k, k_stride_tok, k_stride_head, v, v_stride_tok,
                                       v_stride_head, cos, sin, cs_stride_tok, s->num_heads, s->num_kv_heads,
                                       s->head_dim, s->dtype, q_rot, row, s->head_dim, k_cache, v_cache, slots,
                                       s->slot_mapping, s->num_tokens, k_scale, v_scale, stream)
             : mllm_rope_kv_append(q, q_stride_tok, q_stride_head, k, k_stride_tok, k_stride_head, v, v_stride_tok,
                                   v_stride_head, cos, sin, cs_stride_tok, s->num_heads, s->num_kv_heads, s->head_dim,
                                   s->dtype, q_rot, row, s->head_dim, k_cache, v_cache, slots, s->slot_mapping,
                                   s->num_tokens, stream);
    qa = q_rot;
    qa_st = row;
    qa_sh = s->head_dim;
  } else {
    rc = fp8 ? mllm_kv_append_fp8(k, k_stride_tok, k_stride_head, v, v_stride_tok, v_stride_head, s->dtype, k_cache,
                                  v_cache, slots, s->num_kv_heads, s->head_dim, s->slot_mapping, s->num_tokens,
                                  k_scale, v_scale, stream)
             : mllm_kv_append(k, k_stride_tok, k_stride_head, v, v_stride_tok, v_stride_head, s->dtype, k_cache,
                              v_cache, s->dtype, slots, s->num_kv_heads, s->head_dim, s->slot_mapping, s->num_tokens,
                              stream);
  }
  if (rc != MLLM_OK) return rc;
  if (s->num_decode_work > 0) {
    rc = fp8 ? mllm_paged_decode_fp8(qa, qa_st, qa_sh, k_cache, v_cache, s->num_blocks, s->block_size, s->num_heads,
                                     s->num_kv_heads, s->head_dim, s->qo_indptr, s->kv_indptr, s->kv_indices,
                                     s->seq_lens, s->decode_work, s->num_decode_work, s->merge_work,
                                     s->num_merge_work, s->pages_per_split, s->softmax_scale, s->dtype, k_scale,
                                     v_scale, out, row, s->head_dim, s->workspace, s->workspace_bytes, stream)
             : mllm_paged_decode(qa, qa_st, qa_sh, k_cache, v_cache, s->num_blocks, s->block_size, s->num_heads,
                                 s->num_kv_heads, s->head_dim, s->qo_indptr, s->kv_indptr, s->kv_indices, s->seq_lens,
                                 s->decode_work, s->num_decode_work, s->merge_work, s->num_merge_work,
                                 s->pages_per_split, s->softmax_scale, s->dtype, out, row, s->head_dim, s->workspace,
                                 s->workspace_bytes, stream);
    if (rc != MLLM_OK) return rc;
    rc = mllm_merge_splits(s->merge_work, s->num_merge_work, s->num_decode_work, s->num_heads, s->head_dim,
                           s->qo_indptr, s->dtype, out, row, s->head_dim, s->workspace, s->workspace_bytes, stream);
    if (rc != MLLM_OK) return rc;
  }
  if (s->num_prefill_work > 0) {
    rc = fp8 ? mllm_paged_prefill_fp8(qa, qa_st, qa_sh, k_cache, v_cache, s->num_blocks, s->block_size,
                                      s->num_heads, s->num_kv_heads, s->head_dim, s->qo_indptr, s->kv_indptr,
                                      s->kv_indices, s->seq_lens, s->prefill_work, s->num_prefill_work,
                                      s->q_tile_tokens, s->softmax_scale, s->dtype, k_scale, v_scale, out, row,
                                      s->head_dim, stream)
             : mllm_paged_prefill(qa, qa_st, qa_sh, k_cache, v_cache, s->num_blocks, s->block_size, s->num_heads,
                                  s->num_kv_heads, s->head_dim, s->qo_indptr, s->kv_indptr, s->kv_indices,
                                  s->seq_lens, s->prefill_work, s->num_prefill_work, s->q_tile_tokens,
                                  s->softmax_scale, s->dtype, out, row, s->head_dim, stream);
  }
  return rc;
}

// ---------------------------------------------------------------- a whole decoder layer of few rows
//
// Eleven launches on the stream: norm, the q k v products and their sum, RoPE + append, decode + merge (prefill), the o
// product, its sum with the residual and the second norm, gate and up with SwiGLU, the down product and its sum.
// Bound by the host when each launch is a foreign call of its own: 8 rows of a Llama-3.1-8B layer took the host 174 us
// and the GPU 119 us; in one call the host takes 99 us and the layer 118.6 us instead of 142.8.

namespace {

constexpr int64_t align256(int64_t n) { return (n + 255) / 256 * 256; }

// The call's scratch, laid out once; `part` is shared by the three products (each is summed before the next).
struct LayerScratch {
  int64_t h, qkv, q_rot, attn, x2, act, part, total;
  int ks_qkv, ks_o, ks_down;
};

LayerScratch layer_scratch(int64_t m, int64_t hidden, int64_t ffn, int64_t q, int64_t kv) {
  LayerScratch s;
  s.ks_qkv = mllm_linear_ksplit(hidden, q, kv, kv, 0);
  s.ks_o = mllm_linear_ksplit(q, hidden, 0, 0, 0);
  s.ks_down = mllm_linear_ksplit(ffn, hidden, 0, 0, 0);
  int64_t at = 0;
  auto take = [&](int64_t bytes) {
    const int64_t here = at;
    at += align256(bytes);
    return here;
  };
  s.h = take(2 * m * hidden);
  s.qkv = take(2 * m * (q + 2 * kv));
  s.q_rot = take(2 * m * q);
  s.attn = take(2 * m * q);
  s.x2 = take(2 * m * hidden);
  s.act = take(2 * m * ffn);
  const int64_t parts[3] = {s.ks_qkv * (q + 2 * kv), s.ks_o * hidden, s.ks_down * hidden};
  int64_t most = parts[0] > parts[1] ? parts[0] : parts[1];
  most = most > parts[2] ? most : parts[2];
  s.part = take(4 * m * most);
  s.total = at;
  return s;
}

}  // namespace

extern "C" int64_t mllm_decoder_layer_scratch_bytes(int64_t rows, int64_t hidden, int64_t ffn, int32_t num_heads,
                                                    int32_t num_kv_heads, int32_t head_dim) {
  if (rows <= 0 || hidden <= 0 || ffn <= 0 || num_heads <= 0 || num_kv_heads <= 0 || head_dim <= 0) return 0;
  return layer_scratch(rows, hidden, ffn, (int64_t)num_heads * head_dim, (int64_t)num_kv_heads * head_dim).total;
}

extern "C" int mllm_decoder_layer(const mllm_layer_step* s, const void* x, int64_t hidden, const void* norm1,
                                  float eps1, const void* wq, const void* wk, const void* wv, const void* wo,
                                  const void* norm2, float eps2, const void* gate, const void* up, const void* down,
                                  int64_t ffn, const void* cos, const void* sin, int64_t cs_stride_tok, void* k_cache,
                                  void* v_cache, float k_scale, float v_scale, void* scratch, int64_t scratch_bytes,
                                  void* out, void* stream) {
  using namespace mllm;
  MLLM_REQUIRE(s, MLLM_ERR_INVALID, "mllm_decoder_layer: null step");
  MLLM_REQUIRE(s->num_heads > 0 && s->num_kv_heads > 0 && s->head_dim > 0 && s->num_tokens >= 0 && hidden > 0 && ffn > 0,
               MLLM_ERR_INVALID, "mllm_decoder_layer: bad sizes");
  if (s->num_tokens == 0) return MLLM_OK;
  MLLM_REQUIRE(cos && sin && scratch && out, MLLM_ERR_INVALID, "mllm_decoder_layer: null pointer");
  const int64_t m = s->num_tokens, dh = s->head_dim, nq = s->num_heads * dh, nkv = s->num_kv_heads * dh;
  const int64_t cols = nq + 2 * nkv;
  const LayerScratch at = layer_scratch(m, hidden, ffn, nq, nkv);
  MLLM_REQUIRE(scratch_bytes >= at.total && (uintptr_t)scratch % 256 == 0, MLLM_ERR_INVALID,
               "mllm_decoder_layer: scratch too small or not 256-byte aligned");
  char* base = static_cast<char*>(scratch);
  char *h = base + at.h, *qkv = base + at.qkv, *attn = base + at.attn, *x2 = base + at.x2, *act = base + at.act;
  float* part = reinterpret_cast<float*>(base + at.part);
  const int dt = s->dtype;
  int rc = mllm_rms_norm(x, nullptr, norm1, m, hidden, eps1, dt, nullptr, h, stream);
  if (rc == MLLM_OK) rc = mllm_linear_partial(h, m, hidden, wq, nq, wk, nkv, wv, nkv, at.ks_qkv, part, dt, stream);
  if (rc == MLLM_OK) rc = mllm_sum_partials(part, at.ks_qkv, m, cols, nullptr, dt, qkv, stream);
  if (rc == MLLM_OK)
    rc = mllm_attention_forward(s, qkv, cols, dh, qkv + 2 * nq, cols, dh, qkv + 2 * (nq + nkv), cols, dh, cos, sin,
                                cs_stride_tok, base + at.q_rot, k_cache, v_cache, k_scale, v_scale, attn, stream);
  if (rc == MLLM_OK) rc = mllm_linear_partial(attn, m, nq, wo, hidden, nullptr, 0, nullptr, 0, at.ks_o, part, dt, stream);
  if (rc == MLLM_OK) rc = mllm_sum_partials_norm(part, at.ks_o, x, norm2, m, hidden, eps2, dt, x2, h, stream);
  if (rc == MLLM_OK) rc = mllm_linear_swiglu(h, m, hidden, gate, up, ffn, dt, act, stream);
  if (rc == MLLM_OK)
    rc = mllm_linear_partial(act, m, ffn, down, hidden, nullptr, 0, nullptr, 0, at.ks_down, part, dt, stream);
  if (rc == MLLM_OK) rc = mllm_sum_partials(part, at.ks_down, m, hidden, x2, dt, out, stream);
  return rc;
}
