// Launchers of the decode-step glue kernels (decoder_kernels.hip), used by decoder.hip.
#pragma once

#include "common.hpp"

namespace yscv {

// With a RopeTable they also leave the cosines and sines of the position for the attention launches of the step.
struct RopeTable {
  const int32_t *pos = nullptr;
  float *angles = nullptr;  // [2][hd / 2]; null: none wanted
  int hd = 0;
  float theta = 0.0f;
};
int32_t launch_embed(const int32_t *tokens, const _Float16 *table, int batch, int d, int vocab, float *h, hipStream_t s,
                     const RopeTable &rope = RopeTable());
// embedding lookup + the first norm in its folded form (NormFold in kernels.hpp): one partial sum of squares and the
// power-of-two scale of xg per row
int32_t launch_embed_norm(const int32_t *tokens, const _Float16 *table, int batch, int d, int vocab, float eps, float *h,
                          const float *gamma, _Float16 *xg, float *ss_out, int ss_stride, float *pre, hipStream_t s,
                          const RopeTable &rope = RopeTable());
int32_t launch_rmsnorm(const float *h, const float *gamma, int batch, int d, float eps, _Float16 *out,
                       hipStream_t s);
int32_t launch_rope_append(_Float16 *qkv, const int32_t *pos_ptr, int batch, int hq, int hkv, int hd, float theta,
                           int max_ctx, _Float16 *kc, _Float16 *vc, hipStream_t s);
int32_t launch_kv_relayout(const _Float16 *k_nat, const _Float16 *v_nat, int batch, int npos, int hkv, int hd,
                           int max_ctx, _Float16 *kc, _Float16 *vc, hipStream_t s);
// rope + append fused into the attention partials of 128 positions each, then the merge (fp16 cache, head width 128, up to four
// query heads per kv head): `qrot` receives the rotated query heads [batch][hq * 128] (diagnostics; qkv itself keeps the unrotated q),
// `angles` are a RopeTable's, `part` holds batch * hq * (max_ctx / 128) * 130 floats
int32_t launch_attention_chunks(const _Float16 *qkv, _Float16 *kc, _Float16 *vc, const int32_t *pos_ptr, int batch, int hq, int hkv,
                                int hd, const float *angles, int max_ctx, float *part, _Float16 *qrot, _Float16 *out, hipStream_t s);
// decode_attention.hip: one query position per sequence over the fp16 cache (head widths 32, 64, 96, 128, any number of query
// heads per kv head).  With `qrot` the rotary embedding and the cache append happen inside: qkv holds q, k, v unrotated, kc / vc
// receive the new row, qrot [batch][hq * hd] the rotated query heads (diagnostics), by the angles of a RopeTable; without it qkv holds the rotated q and the
// cache already has the row.  `meet`: attention_decode_meet_bytes of memory, every byte 0xff before the first launch; launches that
// share it follow each other.
size_t attention_decode_meet_bytes(int max_batch, int hq, int hkv, int hd, int max_ctx, int num_cus);
int32_t launch_attention_decode(const _Float16 *qkv, _Float16 *kc, _Float16 *vc, const int32_t *pos, int batch, int hq, int hkv, int hd,
                                const float *angles, int max_ctx, int num_cus, uint64_t *meet, _Float16 *qrot, _Float16 *out, hipStream_t s);
// int8 cache (KvCache with KvDtype::I8): K int8 [batch][kv_head][max_ctx][128], V int8 [batch][kv_head][max_ctx/8][128][8],
// one f32 scale per (batch row, position) for each of them
int32_t launch_rope_append_i8(_Float16 *qkv, const int32_t *pos_ptr, int batch, int hq, int hkv, int hd, float theta,
                              int max_ctx, int8_t *kc, float *ks, int8_t *vc, float *vs, hipStream_t s);
// prompt pass: positions start_pos .. start_pos + rows - 1 of batch row 0 rotated, quantised and appended; tk / tv
// (fp16, laid out like the fp16 cache with t_ctx positions) receive what the int8 cache returns for positions
// 0 .. start_pos + rows - 1
int32_t launch_prefill_rope_append_i8(_Float16 *qkv, int rows, int start_pos, int hq, int hkv, int hd, float theta, int max_ctx,
                                      int8_t *kc, float *ks, int8_t *vc, float *vs, int t_ctx, _Float16 *tk, _Float16 *tv,
                                      hipStream_t s);
int32_t launch_kv_relayout_i8(const _Float16 *k_nat, const _Float16 *v_nat, int batch, int npos, int hkv, int hd, int max_ctx,
                              int8_t *kc, float *ks, int8_t *vc, float *vs, hipStream_t s);
int32_t launch_attention_i8(const _Float16 *qkv, const int8_t *kc, const float *ks, const int8_t *vc, const float *vs,
                            const int32_t *pos_ptr, int batch, int hq, int hkv, int hd, int max_ctx, float *part,
                            _Float16 *out, hipStream_t s);
// rope_append_i8 fused into the attention partials, then the merge (int8 cache); `qrot` as in launch_attention_decode
int32_t launch_attention_fused_i8(const _Float16 *qkv, int8_t *kc, float *ks, int8_t *vc, float *vs, const int32_t *pos_ptr,
                                  int batch, int hq, int hkv, int hd, float theta, int max_ctx, float *part, _Float16 *qrot,
                                  _Float16 *out, hipStream_t s);
int32_t launch_kv_random_fill_i8(int8_t *buf, size_t n, float *scales, size_t n_scales, float scale, uint64_t seed, hipStream_t s);
// greedy pick per row of logits, tokens and history recorded, *pos and *step advanced; `parts` keeps what the chunks of 1024
// logits gave: pick_chunks(vocab) per row
constexpr int kPickChunk = 1024;
inline int pick_chunks(int vocab) { return (vocab + kPickChunk - 1) / kPickChunk; }
struct PickPart {
  float best;
  int idx;
  float top;  // largest value that is no NaN
  int flags;  // 1: a NaN, 2: a NaN or +inf
};
int32_t launch_pick_chunks(const float *logits, int batch, int vocab, PickPart *parts, hipStream_t s);
int32_t launch_pick(const float *logits, int batch, int vocab, PickPart *parts, int32_t *tokens, int32_t *history, int32_t *pos_ptr,
                    int32_t *step_ptr, int max_steps, hipStream_t s);
struct TopCandidate {
  float value;
  uint32_t index;
};
// row 0's logits that can be among the k largest (decoder_kernels.hip); counts, out and odd are pinned host memory
int32_t launch_top_candidates(const float *logits, int vocab, const PickPart *parts, int k, float scale, uint32_t *counts, TopCandidate *out,
                              uint32_t *odd, hipStream_t s);
int32_t launch_kv_random_fill(_Float16 *buf, size_t n, uint64_t seed, hipStream_t s);

// glue_ops.hip: attention of the prompt pass over the fp16 cache (any head width that is a multiple of 32 up to 128, any number
// of query heads per kv head): `rows` consecutive positions start_pos .. of batch row 0, causal, q rotated, the rows in the cache.
int32_t launch_gqa_cache(const _Float16 *qkv, const _Float16 *kc, const _Float16 *vc, int rows, int start_pos, int hq, int hkv, int hd,
                         int max_ctx, _Float16 *out, hipStream_t s);
// {cos, sin} of every pair at positions start_pos .. start_pos + rows - 1, for the launches of all layers of a pass
size_t prefill_angles_bytes(size_t rows, int hd);
int32_t launch_prefill_angles(int rows, int start_pos, int hd, float theta, void *angles, hipStream_t s);
int32_t launch_prefill_rope_append(_Float16 *qkv, int rows, int start_pos, int hq, int hkv, int hd, const void *angles, int max_ctx,
                                   _Float16 *kc, _Float16 *vc, hipStream_t s);
int32_t launch_bias_add_f16(_Float16 *x, const _Float16 *bias, size_t rows, size_t n, hipStream_t s);

}  // namespace yscv
