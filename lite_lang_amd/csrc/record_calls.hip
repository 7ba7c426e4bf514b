// Record forms of the entry points an eager program calls most
// (include/litelang_amd.h, "record calls"): host code only.
#include "ll_common.h"

namespace {
template <typename T> T* ptr(int64_t v) { return (T*)(uintptr_t)v; }
}  // namespace

extern "C" int64_t ll_call_rmsnorm(const LLRmsnormCall* c) {
  LL_CHECK_ARG(c, "ll_call_rmsnorm: null record");
  return ll_rmsnorm(ptr<void>(c->x), c->x_row_stride, ptr<const void>(c->residual),
                    c->residual_row_stride, ptr<const void>(c->gamma), ptr<void>(c->out),
                    c->out_row_stride, c->M, c->N, (float)c->eps, (int)c->dtype,
                    ptr<ihipStream_t>(c->stream));
}

extern "C" int64_t ll_call_decode_attention(const LLDecodeAttentionCall* c) {
  LL_CHECK_ARG(c, "ll_call_decode_attention: null record");
  // (shapes the entry point refuses go to it for its error)
  if (c->batch > 0 && c->kv_heads > 0 && c->head_dim > 0 && c->max_len_in_batch >= 0) {
    const int64_t need = ll_decode_attention_workspace_size(c->batch, c->q_heads, c->kv_heads,
                                                            c->head_dim, c->max_len_in_batch);
    if (need > c->workspace_bytes) return need;
  }
  return ll_decode_attention(
      ptr<const void>(c->q), c->q_stride_b, c->q_stride_h, ptr<const void>(c->k_cache),
      c->k_stride_tok, c->k_stride_head, ptr<const void>(c->v_cache), c->v_stride_tok,
      c->v_stride_head, ptr<const int32_t>(c->req_to_tokens), c->req_to_tokens_stride,
      ptr<const void>(c->b_req_idx), (int)c->req_idx_i64, ptr<const void>(c->b_seq_len),
      (int)c->seq_len_i64, ptr<void>(c->out), c->out_stride_b, c->out_stride_h, c->batch,
      c->q_heads, c->kv_heads, c->head_dim, c->max_len_in_batch, (float)c->sm_scale, (int)c->dtype,
      ptr<void>(c->workspace), c->workspace_bytes, ptr<ihipStream_t>(c->stream));
}

extern "C" int64_t ll_call_prefill_attention(const LLPrefillAttentionCall* c) {
  LL_CHECK_ARG(c, "ll_call_prefill_attention: null record");
  return ll_prefill_attention(
      ptr<const void>(c->q), c->q_stride_tok, c->q_stride_h, ptr<const void>(c->k_cache),
      c->k_stride_tok, c->k_stride_head, ptr<const void>(c->v_cache), c->v_stride_tok,
      c->v_stride_head, ptr<void>(c->out), c->out_stride_tok, c->out_stride_h,
      ptr<const int32_t>(c->req_to_tokens), c->req_to_tokens_stride, ptr<const void>(c->b_req_idx),
      (int)c->req_idx_i64, ptr<const void>(c->b_start_loc), (int)c->start_loc_i64,
      ptr<const void>(c->b_seq_len), (int)c->seq_len_i64, ptr<const void>(c->b_shared_seq_len),
      (int)c->shared_i64, c->batch, c->q_heads, c->kv_heads, c->head_dim, c->max_input_len,
      (float)c->sm_scale, (int)c->dtype, ptr<ihipStream_t>(c->stream));
}

extern "C" int64_t ll_call_gemm(const LLGemmCall* c) {
  LL_CHECK_ARG(c, "ll_call_gemm: null record");
  int64_t need = 0;
  if (c->M > 64) {
    if (!c->any_workspace && c->dtype != LL_F32)
      need = ll_gemm_tiles_workspace_size(c->M, c->N, c->K, 2);
  } else if (c->M > 0 && c->N > 0 && c->K > 0) {
    need = ll_gemm_workspace_size(c->M, c->N, c->K);
  }
  if (need > c->workspace_bytes) return need;
  return ll_gemm(ptr<const void>(c->X), c->ldx, ptr<const void>(c->W), c->ldw,
                 ptr<const void>(c->bias), ptr<void>(c->Y), c->ldy, c->M, c->N, c->K,
                 (int)c->dtype, ptr<void>(c->workspace), c->workspace_bytes,
                 ptr<ihipStream_t>(c->stream));
}
