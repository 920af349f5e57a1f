// Interface of the kernels that take one token through all layers of a decoder in one launch (decode_layers.hip: head width 64,
// decode_wide.hip: head width 128).
#pragma once

#include "common.hpp"

namespace yscv {

// One layer as the kernel reads it: projections 0 q/k/v, 1 o, 2 gate/up (rows interleaved), 3 down in the tiled layout of
// int4_common.hpp (groups of 32, fp16 scales), norms 0 attention, 1 FFN.
struct LayersLayer {
  const uint8_t *tiles[4];
  const _Float16 *scales[4];
  const float *gamma[2];
  _Float16 *kc, *vc;
  const _Float16 *qkv_bias;  // null or [(heads + 2 kv_heads) * head width]
};

struct LayersModel {
  const __attribute__((address_space(4))) LayersLayer *layers;  // device, constant while a step runs
  int n_layers, d, heads, kv_heads, ff, vocab, max_ctx;
  int G;       // workgroups = 16-row blocks of the residual stream
  int ktp[4];  // stored 128-k tiles per 16-row block of each projection
  float theta, eps;
  const _Float16 *emb;
  const int32_t *tokens, *pos;
  float *h;  // residual stream behind the last layer
  // exchange buffer of 8-byte {payload, tag} entries: residual before each norm (f32), q/k/v and SwiGLU output (two fp16
  // each), attention partials.  No 128-byte line is written by two workgroups.
  unsigned long long *x;
  int at_attn, at_ffn, at_qkv, at_act, at_part, at_ao;  // (at_ao: decode_wide.hip only)
  uint32_t *steps;    // steps since the entries were cleared
  uint32_t *give_up;  // pinned host memory: a wait gave up
};

constexpr int kLayersChunk = 256;     // cached positions of one attention work item
constexpr int kLayersActSlots = 32;   // entries a workgroup has for its SwiGLU output (at most 28 used)
inline __host__ __device__ int layers_chunks(int max_ctx) { return (max_ctx + kLayersChunk - 1) / kLayersChunk; }
constexpr int kLayersHeadRec = 80;    // entries of one head's partials of a chunk: o[64], max, sum; whole lines

bool layers_supported(const yscv_hip_decoder_config &c, int num_cus);
// entries each part of the exchange buffer needs, in the order of LayersModel
void layers_exchange_entries(const yscv_hip_decoder_config &c, size_t out[5]);
int32_t launch_decode_layers(const LayersModel &m, hipStream_t s);
int32_t launch_layers_report(const LayersModel &m, int pos, _Float16 *qkv, _Float16 *qrot, _Float16 *ao, _Float16 *act, hipStream_t s);

// the same for head width 128
bool wide_supported(const yscv_hip_decoder_config &c, int num_cus);
void wide_exchange_entries(const yscv_hip_decoder_config &c, size_t out[6]);
int32_t launch_decode_wide(const LayersModel &m, hipStream_t s);
int32_t launch_wide_report(const LayersModel &m, int pos, _Float16 *qkv, _Float16 *qrot, _Float16 *ao, _Float16 *act, hipStream_t s);

}  // namespace yscv
