// Which form the decoder's attention takes (decode_attention.hip, decoder_kernels.hip, glue_ops.hip) on a card of num_cus CUs.  Host code
// only, without the HIP headers.
#pragma once

namespace yscv {

// Decode step over the fp16 cache: chunks of 128 positions and a merge launch, or the kernel of decode_attention.hip (times of both in its
// header): the line is a quarter of the CUs, from where on a pair of sequence and kv head needs no more than four workgroups.
inline bool attention_in_chunks(int batch, int hq, int hkv, int hd, int num_cus) {
  return hd == 128 && hq / hkv <= 4 && 4LL * batch * hkv < (num_cus > 0 ? num_cus : 256);
}

// Prompt pass, rows of 16 queries that a wave takes: two where that fills the CUs, else one: twice the workgroups, shorter steps (700
// queries, 16 heads over 2 of 64: 88 workgroups of two).  heads: workgroups side by side, waves_q: query ranges of a workgroup.
inline int prompt_row_tiles(unsigned heads, unsigned queries, unsigned waves_q, int num_cus) {
  const unsigned long long wgs = (unsigned long long)heads * ((queries + 32 * waves_q - 1) / (32 * waves_q));
  return wgs >= (unsigned)(num_cus > 0 ? num_cus : 256) ? 2 : 1;
}

}  // namespace yscv
