// The operators between the MatMuls of an exported LLM graph, as stand-alone entry points on device tensors, so
// that a graph executor stays on the GPU from one projection to the next:
//   rms_norm   crates/yscv-kernels/src/ops/norm.rs:1431-1518   y = x * (1 / sqrt(mean(x^2) + eps)) * gamma, last axis
//   rope       crates/yscv-kernels/src/ops/rope.rs:24-117      rotate-half pairs (i, i + d/2), in place on q and k
//   GroupQueryAttention  crates/yscv-onnx/src/runner/linear.rs:552-646   q [B][Sq][Hq d], k / v [B][Sk][Hkv d],
//              kv_h = q_h / groups, scores * 1/sqrt(d), max-subtracted softmax, no mask
// and the general attention kernel behind the last one, which the decoder also uses where its specialised kernels
// do not apply: any head width that is a multiple of 32 up to 128, any number of query heads per kv head, several
// query positions per call with a causal limit (prompt ingestion), K / V either as the operator's tensors or as the
// decoder's fp16 cache.
//
// Three forms of the attention kernel share the arithmetic below: gqa_generic_kernel (the prompt pass over the decoder's cache with
// short query counts: a workgroup owns 16 queries of one head, the key blocks are split over its waves),
// gqa_shared_kv_kernel (the prompt pass over the cache: the waves of a workgroup share each stage of K / V through LDS)
// and gqa_flat_kernel (the operator on f32 tensors).
// gqa_generic_kernel: a workgroup of four waves owns 16 query positions of one head.  Wave w walks the key blocks
// w, w + 4, ... of 16 positions each:
//   S^T = K Q^T   rows = positions, columns = queries: hd / 32 x v_mfma_f32_16x16x32_f16, A = 16 cache rows as they lie
//                 in memory, B = the 16 query rows as they lie in memory; lane (r, c) then holds positions 4c .. 4c+3
//                 of query r, which is exactly the B operand of the second product
//   online softmax per query (= per lane column r; the four lane groups c are reduced with two permlane swaps)
//   O^T += V^T P^T  hd / 16 x v_mfma_f32_16x16x16_f16, A = V^T (the cache keeps eight consecutive positions of one
//                 channel together, so a lane's four positions are one 8-byte load)
// and the four waves merge their (max, sum, O) through LDS.  Scores and sums are f32; q, k, v and the softmax weights
// enter the MFMAs as fp16, like the decoder's own kernels (tolerance-checked against the f32 restatement).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <mutex>

#include "attention_plan.hpp"
#include "int4_common.hpp"
#include "decoder.hpp"
#include "kernels.hpp"
#include "rope.hpp"

namespace yscv {

namespace {

struct GqaArgs {
  const void *q, *k, *v;
  void *out;
  // element strides: q[b * q_b + s * q_s + h * hd + d], same for k (h = kv head) and out; v natural like k, or
  // v slab: v[b * v_b + kvh * v_h + ((pos / 8) * hd + d) * 8 + pos % 8]
  long long q_b, q_s, k_b, k_s, k_h, v_b, v_s, v_h, o_b, o_s;
  int B, Sq, Sk, Hq, Hkv;
  int causal_base;            // < 0: every query sees all Sk positions; else query s sees positions <= causal_base + s
  float scale;
};

template <typename T>
__device__ __forceinline__ half8_t load8(const T *p);
template <>
__device__ __forceinline__ half8_t load8<_Float16>(const _Float16 *p) {
  return *reinterpret_cast<const half8_t *>(p);
}
template <>
__device__ __forceinline__ half8_t load8<float>(const float *p) {
  const float4_t a = *reinterpret_cast<const float4_t *>(p), b = *reinterpret_cast<const float4_t *>(p + 4);
  return half8_t{(_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3],
                 (_Float16)b[0], (_Float16)b[1], (_Float16)b[2], (_Float16)b[3]};
}
template <typename T>
__device__ __forceinline__ void store4(T *p, float a, float b, float c, float d);
template <>
__device__ __forceinline__ void store4<_Float16>(_Float16 *p, float a, float b, float c, float d) {
  *reinterpret_cast<half4_t *>(p) = half4_t{(_Float16)a, (_Float16)b, (_Float16)c, (_Float16)d};
}
template <>
__device__ __forceinline__ void store4<float>(float *p, float a, float b, float c, float d) {
  *reinterpret_cast<float4_t *>(p) = float4_t{a, b, c, d};
}

constexpr int GQA_WAVES = 4;

template <int HD>
__global__ void __launch_bounds__(64 * GQA_WAVES) gqa_generic_kernel(GqaArgs p) {
  static_assert(HD % 32 == 0 && HD >= 32 && HD <= 128, "head width (the merge buffer must fit the static LDS limit)");
  using TQ = _Float16;
  using TKV = _Float16;
  using TO = _Float16;
  constexpr int KK = HD / 32, DT = HD / 16;
  __shared__ float m_s[GQA_WAVES][16], l_s[GQA_WAVES][16];
  __shared__ float o_s[GQA_WAVES][16][HD + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, c = lane >> 4;
  const int q0 = blockIdx.x * 16, h = blockIdx.y, b = blockIdx.z;
  const int kvh = h / (p.Hq / p.Hkv);
  const int Sk = p.Sk;
  // query r of this tile (rows past the end repeat the last one and are not stored)
  const int qi = min(q0 + r, p.Sq - 1);
  const int lim_q = p.causal_base < 0 ? Sk - 1 : min(Sk - 1, p.causal_base + qi);           // last position query r sees
  const int lim_tile = p.causal_base < 0 ? Sk - 1 : min(Sk - 1, p.causal_base + min(q0 + 15, p.Sq - 1));
  const int nblocks = lim_tile / 16 + 1;

  const TQ *qrow = static_cast<const TQ *>(p.q) + (size_t)b * p.q_b + (size_t)qi * p.q_s + (size_t)h * HD;
  const TKV *kbase = static_cast<const TKV *>(p.k) + (size_t)b * p.k_b + (size_t)kvh * p.k_h;
  const TKV *vbase = static_cast<const TKV *>(p.v) + (size_t)b * p.v_b + (size_t)kvh * p.v_h;
  half8_t qf[KK];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) qf[kk] = load8<TQ>(qrow + 32 * kk + 8 * c);

  float m_run = -INFINITY, l_run = 0.0f;
  float4_t o_acc[DT];
#pragma unroll
  for (int t = 0; t < DT; t++) o_acc[t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // operands of one key block: 16 cache rows as the A operand of S^T (lane (r, c): row p0 + r, channels 32 kk + 8c .. + 7;
  // rows past the end repeat the last one) and V^T as the A operand of the second product (lane (r, c): channel
  // 16 t + r at positions p0 + 4c .. + 3).  The next block's are requested before this block's arithmetic.
  auto load_block = [&](int blk, half8_t (&kf)[KK], half4_t (&vf)[DT]) {
    const int p0 = blk * 16;
    const TKV *krow = kbase + (size_t)min(p0 + r, Sk - 1) * p.k_s;
#pragma unroll
    for (int kk = 0; kk < KK; kk++) kf[kk] = load8<TKV>(krow + 32 * kk + 8 * c);
#pragma unroll
    for (int t = 0; t < DT; t++) {
      const _Float16 *vp = vbase + ((size_t)((p0 + 4 * c) >> 3) * HD + 16 * t + r) * 8 + ((4 * c) & 7);
      vf[t] = *reinterpret_cast<const half4_t *>(vp);
    }
  };
  half8_t kf[KK], kn[KK];
  half4_t vf[DT], vn[DT];
  if (wave < nblocks) load_block(wave, kf, vf);
  for (int blk = wave; blk < nblocks; blk += GQA_WAVES) {
    const int p0 = blk * 16;
    const bool more = blk + GQA_WAVES < nblocks;  // uniform in the wave
    if (more) load_block(blk + GQA_WAVES, kn, vn);
    float4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < KK; kk++) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[kk], qf[kk], s, 0, 0, 0);
    // lane (r, c): query r, positions p0 + 4c + e
    float sv[4], mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      sv[e] = (p0 + 4 * c + e <= lim_q) ? s[e] * p.scale : -INFINITY;
      mx = fmaxf(mx, sv[e]);
    }
    mx = max_xor16_xor32(mx);
    const float m_new = fmaxf(m_run, mx);
    float pe[4], sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      pe[e] = (sv[e] == -INFINITY) ? 0.0f : __expf(sv[e] - m_new);
      sum += pe[e];
    }
    sum = sum_xor16_xor32(sum);
    const float alpha = (m_run == -INFINITY) ? 0.0f : __expf(m_run - m_new);
    l_run = l_run * alpha + sum;
    m_run = m_new;
    const half4_t pf = {(_Float16)pe[0], (_Float16)pe[1], (_Float16)pe[2], (_Float16)pe[3]};
#pragma unroll
    for (int t = 0; t < DT; t++) {
      // positions past the end of the context meet weight 0 -- but 0 * NaN would poison the sum (the slab may hold
      // anything there), so they are blanked
      half4_t vv = vf[t];
#pragma unroll
      for (int e = 0; e < 4; e++)
        if (p0 + 4 * c + e >= Sk) vv[e] = (_Float16)0.0f;
      o_acc[t] = o_acc[t] * alpha;
      o_acc[t] = __builtin_amdgcn_mfma_f32_16x16x16f16(vv, pf, o_acc[t], 0, 0, 0);
    }
    if (more) {
#pragma unroll
      for (int kk = 0; kk < KK; kk++) kf[kk] = kn[kk];
#pragma unroll
      for (int t = 0; t < DT; t++) vf[t] = vn[t];
    }
  }
  // ---- merge the four waves: lane (r, c) holds O^T[16 t + 4c + e][query r]
  if (c == 0) {
    m_s[wave][r] = m_run;
    l_s[wave][r] = l_run;
  }
#pragma unroll
  for (int t = 0; t < DT; t++)
#pragma unroll
    for (int e = 0; e < 4; e++) o_s[wave][r][16 * t + 4 * c + e] = o_acc[t][e];
  __syncthreads();
  TO *obase = static_cast<TO *>(p.out) + (size_t)b * p.o_b + (size_t)h * HD;
  for (int idx = tid; idx < 16 * (HD / 4); idx += 64 * GQA_WAVES) {
    const int qq = idx / (HD / 4), d4 = (idx % (HD / 4)) * 4;
    if (q0 + qq >= p.Sq) continue;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < GQA_WAVES; w++) M = fmaxf(M, m_s[w][qq]);
    float L = 0.0f, o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < GQA_WAVES; w++) {
      const float f = (m_s[w][qq] == -INFINITY) ? 0.0f : __expf(m_s[w][qq] - M);
      L += l_s[w][qq] * f;
#pragma unroll
      for (int e = 0; e < 4; e++) o[e] += o_s[w][qq][d4 + e] * f;
    }
    const float inv = L > 0.0f ? 1.0f / L : 0.0f;
    store4<TO>(obase + (size_t)(q0 + qq) * p.o_s + d4, o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
  }
}

// One step of a running softmax in powers of two over 32 positions for QT row tiles: lane (r, c) has the scores of positions 8 c .. 8 c + 7
// against row r of tile u, scale2 is the scale with log2(e) in it.  Leaves the weights as fp16 (the B operand of the product with V).  The row
// tiles' chains are independent and run side by side.  The lanes of a row agree on a new maximum, and the output is rescaled, only in
// steps where some score passes the running one (weights that stay within 1 .. 2^8 of an older maximum would need that less often, but
// the largest weight is then no longer exact in fp16: 4 % more error at 512 keys).  l_run is the lane's own part of the sum; the lanes of
// a row meet behind the last step.
template <int QT, int DT>
__device__ __forceinline__ void softmax_step(const float4_t (&sc)[QT][2], float scale2, float (&m_run)[QT], float (&l_run)[QT], float4_t (&o_acc)[QT][DT],
                                             half8_t (&pf)[QT]) {
  float mx[QT];
  bool grows = false;
#pragma unroll
  for (int u = 0; u < QT; u++) {
    mx[u] = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; e++) mx[u] = fmaxf(mx[u], sc[u][e >> 2][e & 3]);
    mx[u] *= scale2;
    grows = grows || mx[u] > m_run[u];
  }
  if (__builtin_amdgcn_ballot_w64(grows) != 0) {
#pragma unroll
    for (int u = 0; u < QT; u++) {
      const float m_new = fmaxf(m_run[u], max_xor16_xor32(mx[u]));
      const float alpha = m_run[u] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run[u] - m_new);
      l_run[u] *= alpha;
      m_run[u] = m_new;
#pragma unroll
      for (int t = 0; t < DT; t++) o_acc[u][t] = o_acc[u][t] * alpha;
    }
  }
#pragma unroll
  for (int u = 0; u < QT; u++) {
    const float m_sub = m_run[u] == -INFINITY ? 0.0f : m_run[u];
    float pe[8];
#pragma unroll
    for (int e = 0; e < 8; e++) pe[e] = __builtin_amdgcn_exp2f(fmaf(sc[u][e >> 2][e & 3], scale2, -m_sub));
    l_run[u] += ((pe[0] + pe[1]) + (pe[2] + pe[3])) + ((pe[4] + pe[5]) + (pe[6] + pe[7]));
    pf[u] = half8_t{(_Float16)pe[0], (_Float16)pe[1], (_Float16)pe[2], (_Float16)pe[3], (_Float16)pe[4], (_Float16)pe[5], (_Float16)pe[6], (_Float16)pe[7]};
  }
}

// Prompt pass over the decoder's fp16 cache: four waves of a workgroup take the same key range -- query heads
// that share a kv head (as many of them as divide four), else neighbouring query ranges of one head -- so a
// stage of cache positions is fetched once per workgroup into LDS (K rows with their 16-byte pieces XOR-swizzled
// so that the 16 rows a fragment read touches fall into 16 different bank groups; V as its slabs lie in memory) and
// read from there by all four: a quarter of the L2 traffic of waves that fetch for themselves, which bounds such a
// kernel at prompt lengths in the thousands.  Two such groups of waves take the halves of a 64-position stage and meet through LDS
// at the end: with one group the time was that of the last query range's chain of stages, one wave per SIMD, on CUs whose other
// workgroup was long done.  Two stage buffers: the next stage's pieces are requested into registers before
// this stage's arithmetic and written to the other buffer behind it, one barrier per stage.  Bound by the chain scores ->
// softmax -> product of a step, two waves per SIMD.
// us a launch, one group and a chain per row tile -> this: 2048 queries, 32 heads over 8 of 128 84 -> 59, 700 queries, 16 heads over 2 of
// 64 21.0 -> 10.6, 150 queries, 32 heads over 8 of 128 11.1 -> 7.8.
constexpr int SHARED_KG = 2;  // key groups of a workgroup
template <int HD, int QT>
__global__ void __launch_bounds__(64 * GQA_WAVES * SHARED_KG, QT == 1 && HD <= 64 ? 4 : 2) gqa_shared_kv_kernel(GqaArgs p, int hw_log2) {
  static_assert(HD % 32 == 0 && HD >= 32 && HD <= 128, "head width");
  constexpr int KK = HD / 32, DT = HD / 16, KB = 32 * SHARED_KG;  // KB: cache positions per stage
  constexpr int CPR = HD / 8;                                  // 16-byte pieces of a K row
  constexpr int PITCH = HD > 64 ? 16 : (HD > 32 ? 8 : 4);      // row pitch in pieces (a power of two)
  constexpr int RPW = 16 / PITCH;                              // rows per 256 bytes
  constexpr int K_BYTES = KB * PITCH * 16, V_BYTES = (KB / 8) * HD * 16, ST_BYTES = K_BYTES + V_BYTES;
  constexpr int K_PIECES = KB * CPR, V_PIECES = (KB / 8) * HD;
  constexpr int THREADS = 64 * GQA_WAVES * SHARED_KG;
  constexpr int K_LD = (K_PIECES + THREADS - 1) / THREADS, V_LD = (V_PIECES + THREADS - 1) / THREADS;
  constexpr int MERGE = GQA_WAVES * DT * 1024;  // one row tile of every wave of a key group
  __shared__ __attribute__((aligned(16))) uint8_t stage[2 * ST_BYTES > MERGE ? 2 * ST_BYTES : MERGE];
  __shared__ float ml_s[GQA_WAVES][QT][16][2];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6 & (GQA_WAVES - 1), kg = tid >> 8;
  const int r = lane & 15, c = lane >> 4;
  const int hw = 1 << hw_log2, qw = GQA_WAVES >> hw_log2;  // heads x query ranges of a workgroup
  const int group = p.Hq / p.Hkv, chunks = group >> hw_log2;
  const int kvh = (int)blockIdx.x / chunks, b = blockIdx.z;
  const int h = kvh * group + ((int)blockIdx.x % chunks) * hw + (wave & (hw - 1));
  // Workgroups start in the order of blockIdx.y: the late query ranges (most positions) first, what is left fills the gaps
  const int tile = (int)(gridDim.y - 1 - blockIdx.y);
  const int q0 = (tile * qw + (wave >> hw_log2)) * 16 * QT;
  const bool active = q0 < p.Sq;
  const int Sk = p.Sk;
  const float scale2 = p.scale * 1.44269504088896341f;
  int qi[QT], lim_q[QT];
  half8_t qf[QT][KK];
#pragma unroll
  for (int u = 0; u < QT; u++) {
    qi[u] = min(q0 + 16 * u + r, p.Sq - 1);
    lim_q[u] = p.causal_base < 0 ? Sk - 1 : min(Sk - 1, p.causal_base + qi[u]);
    const _Float16 *qrow = static_cast<const _Float16 *>(p.q) + (size_t)b * p.q_b + (size_t)qi[u] * p.q_s + (size_t)h * HD;
#pragma unroll
    for (int kk = 0; kk < KK; kk++) qf[u][kk] = load8<_Float16>(qrow + 32 * kk + 8 * c);
  }
  const int lim_wave = p.causal_base < 0 ? Sk - 1 : min(Sk - 1, p.causal_base + min(q0 + 16 * QT - 1, p.Sq - 1));
  const int lim_first = p.causal_base < 0 ? Sk - 1 : min(Sk - 1, p.causal_base + min(q0, p.Sq - 1));  // what the wave's first query sees
  const int q_last = min((tile + 1) * qw * 16 * QT, p.Sq) - 1;  // last query of the workgroup
  const int lim_wg = p.causal_base < 0 ? Sk - 1 : min(Sk - 1, p.causal_base + q_last);
  const int nstages = lim_wg / KB + 1;
  const _Float16 *kbase = static_cast<const _Float16 *>(p.k) + (size_t)b * p.k_b + (size_t)kvh * p.k_h;
  const _Float16 *vbase = static_cast<const _Float16 *>(p.v) + (size_t)b * p.v_b + (size_t)kvh * p.v_h;
  float m_run[QT], l_run[QT];
  float4_t o_acc[QT][DT];
#pragma unroll
  for (int u = 0; u < QT; u++) {
    m_run[u] = -INFINITY;
    l_run[u] = 0.0f;
#pragma unroll
    for (int t = 0; t < DT; t++) o_acc[u][t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  // piece idx of a stage's K: row idx / CPR, piece idx % CPR; of its V: slab idx / HD, channel idx % HD.  Rows and
  // slabs past the end of the context repeat the last one (never used: their positions are masked)
  auto fetch = [&](int st, uint4_t (&kr)[K_LD], uint4_t (&vr)[V_LD]) {
#pragma unroll
    for (int j = 0; j < K_LD; j++) {
      const int idx = tid + THREADS * j;
      if (K_PIECES % THREADS == 0 || idx < K_PIECES) {
        const int pos = min(st * KB + idx / CPR, Sk - 1);
        kr[j] = *reinterpret_cast<const uint4_t *>(kbase + (size_t)pos * p.k_s + (idx % CPR) * 8);
      }
    }
#pragma unroll
    for (int j = 0; j < V_LD; j++) {
      const int idx = tid + THREADS * j;
      if (V_PIECES % THREADS == 0 || idx < V_PIECES) {
        const int slab = min(st * (KB / 8) + idx / HD, (Sk - 1) >> 3);
        vr[j] = *reinterpret_cast<const uint4_t *>(vbase + ((size_t)slab * HD + idx % HD) * 8);
      }
    }
  };
  auto stash = [&](int buf, const uint4_t (&kr)[K_LD], const uint4_t (&vr)[V_LD]) {
    uint8_t *base = stage + buf * ST_BYTES;
#pragma unroll
    for (int j = 0; j < K_LD; j++) {
      const int idx = tid + THREADS * j;
      if (K_PIECES % THREADS == 0 || idx < K_PIECES) {
        const int row = idx / CPR, piece = idx % CPR;
        *reinterpret_cast<uint4_t *>(base + (row * PITCH + (piece ^ ((((row >> 3) & 3) * 4 + (row & 3)) / RPW))) * 16) = kr[j];
      }
    }
#pragma unroll
    for (int j = 0; j < V_LD; j++) {
      const int idx = tid + THREADS * j;
      if (V_PIECES % THREADS == 0 || idx < V_PIECES) *reinterpret_cast<uint4_t *>(base + K_BYTES + idx * 16) = vr[j];
    }
  };
  auto compute = [&](int st) {
    const uint8_t *base = stage + (st & 1) * ST_BYTES;
    const int p0 = st * KB + 32 * kg;
    if (active && p0 <= lim_wave) {  // uniform in the wave
      // Two S^T tiles per stage.  Row rho of tile j is stage position 8 (rho / 4) + 4 j + rho % 4, so lane (r, c)
      // ends up with the weights of positions 8c .. 8c+7 (tile 0: the first four, tile 1: the last four): one 16-byte
      // slab piece of V^T per channel, and the B operand of one 32-deep MFMA.
      half8_t vv[DT], pf[QT];
      float4_t sc[QT][2];
      {
        half8_t kf[2][KK];
#pragma unroll
        for (int j = 0; j < 2; j++) {
          const int row = 8 * (r >> 2) + 4 * j + (r & 3);
#pragma unroll
          for (int kk = 0; kk < KK; kk++)
            kf[j][kk] = *reinterpret_cast<const half8_t *>(base + ((32 * kg + row) * PITCH + ((4 * kk + c) ^ (r / RPW))) * 16);
        }
#pragma unroll
        for (int u = 0; u < QT; u++) sc[u][0] = sc[u][1] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kk = 0; kk < KK; kk++)
#pragma unroll
          for (int u = 0; u < QT; u++)
#pragma unroll
            for (int j = 0; j < 2; j++) sc[u][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j][kk], qf[u][kk], sc[u][j], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < DT; t++) vv[t] = *reinterpret_cast<const half8_t *>(base + K_BYTES + ((4 * kg + c) * HD + 16 * t + r) * 16);
      if (p0 + 32 > Sk) {  // 0 * NaN would poison the sum: positions past the context are blanked
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
          for (int e = 0; e < 8; e++)
            if (p0 + 8 * c + e >= Sk) vv[t][e] = (_Float16)0.0f;
      }
      if (p0 + 31 > lim_first) {  // uniform in the wave: some query does not see the whole stage
#pragma unroll
        for (int u = 0; u < QT; u++)
#pragma unroll
          for (int e = 0; e < 8; e++)
            if (p0 + 8 * c + e > lim_q[u]) sc[u][e >> 2][e & 3] = -INFINITY;
      }
      softmax_step<QT, DT>(sc, scale2, m_run, l_run, o_acc, pf);
#pragma unroll
      for (int t = 0; t < DT; t++)
#pragma unroll
        for (int u = 0; u < QT; u++) o_acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv[t], pf[u], o_acc[u][t], 0, 0, 0);
    }
  };
  uint4_t kr[K_LD], vr[V_LD];
  fetch(0, kr, vr);
  stash(0, kr, vr);
  __syncthreads();
  for (int st = 0; st < nstages; st++) {
    const bool more = st + 1 < nstages;  // uniform in the workgroup
    if (more) fetch(st + 1, kr, vr);
    compute(st);
    if (more) stash((st + 1) & 1, kr, vr);
    __syncthreads();
  }
#pragma unroll
  for (int u = 0; u < QT; u++) l_run[u] = sum_xor16_xor32(l_run[u]);
  // the second key group's part meets the first one's, a row tile at a time, lane by lane
  const float4_t *o_other = reinterpret_cast<const float4_t *>(stage) + wave * DT * 64 + lane;
  _Float16 *obase = static_cast<_Float16 *>(p.out) + (size_t)b * p.o_b + (size_t)h * HD;
  if (kg == 1 && c == 0) {
#pragma unroll
    for (int u = 0; u < QT; u++) {
      ml_s[wave][u][r][0] = m_run[u];
      ml_s[wave][u][r][1] = l_run[u];
    }
  }
#pragma unroll
  for (int u = 0; u < QT; u++) {
    if (u > 0) __syncthreads();
    if (kg == 1) {
#pragma unroll
      for (int t = 0; t < DT; t++) const_cast<float4_t *>(o_other)[t * 64] = o_acc[u][t];
    }
    __syncthreads();
    if (kg == 1 || !active || q0 + 16 * u + r >= p.Sq) continue;
    const float m1 = ml_s[wave][u][r][0], l1 = ml_s[wave][u][r][1], m = fmaxf(m_run[u], m1), m_sub = m == -INFINITY ? 0.0f : m;
    const float f0 = __builtin_amdgcn_exp2f(m_run[u] - m_sub), f1 = __builtin_amdgcn_exp2f(m1 - m_sub), l = l_run[u] * f0 + l1 * f1;
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    _Float16 *orow = obase + (size_t)(q0 + 16 * u + r) * p.o_s;
#pragma unroll
    for (int t = 0; t < DT; t++) {
      const float4_t o = (o_acc[u][t] * f0 + o_other[t * 64] * f1) * inv;
      store4<_Float16>(orow + 16 * t + 4 * c, o[0], o[1], o[2], o[3]);
    }
  }
}

// heads of one kv group that share a workgroup of gqa_shared_kv_kernel: the largest of 4, 2, 1 that divides the group
inline int shared_kv_hw_log2(int group) { return group % 4 == 0 ? 2 : (group % 2 == 0 ? 1 : 0); }

int32_t gqa_launch_shared_kv(const GqaArgs &a, int hd, hipStream_t s) {
  const int hw_log2 = shared_kv_hw_log2(a.Hq / a.Hkv);
  const Context *ctx = nullptr;
  YSCV_TRY(ensure_context(&ctx));
  const unsigned heads = (unsigned)(a.Hq >> hw_log2) * (unsigned)a.B, waves_q = (unsigned)(GQA_WAVES >> hw_log2);
  const bool two = prompt_row_tiles(heads, (unsigned)a.Sq, waves_q, ctx->num_cus) == 2;
  const unsigned q_per_wg = (two ? 32 : 16) * waves_q;
  const dim3 grid((unsigned)(a.Hq >> hw_log2), (a.Sq + q_per_wg - 1) / q_per_wg, (unsigned)a.B), block(64 * GQA_WAVES * SHARED_KG);
#define YSCV_SHARED_KV(HD)                                                                      \
  if (two) hipLaunchKernelGGL((gqa_shared_kv_kernel<HD, 2>), grid, block, 0, s, a, hw_log2);    \
  else hipLaunchKernelGGL((gqa_shared_kv_kernel<HD, 1>), grid, block, 0, s, a, hw_log2);        \
  break
  switch (hd) {
    case 32: YSCV_SHARED_KV(32);
    case 64: YSCV_SHARED_KV(64);
    case 96: YSCV_SHARED_KV(96);
    case 128: YSCV_SHARED_KV(128);
    default: return set_error(YSCV_HIP_ERR_UNSUPPORTED, "attention: head width %d (supported: 32, 64, 96, 128)", hd);
  }
#undef YSCV_SHARED_KV
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// few query rows against the decoder's cache
int32_t gqa_launch_cache(const GqaArgs &a, int hd, hipStream_t s) {
  const dim3 grid((unsigned)((a.Sq + 15) / 16), (unsigned)a.Hq, (unsigned)a.B), block(64 * GQA_WAVES);
  switch (hd) {
    case 32: hipLaunchKernelGGL((gqa_generic_kernel<32>), grid, block, 0, s, a); break;
    case 64: hipLaunchKernelGGL((gqa_generic_kernel<64>), grid, block, 0, s, a); break;
    case 96: hipLaunchKernelGGL((gqa_generic_kernel<96>), grid, block, 0, s, a); break;
    case 128: hipLaunchKernelGGL((gqa_generic_kernel<128>), grid, block, 0, s, a); break;
    default: return set_error(YSCV_HIP_ERR_UNSUPPORTED, "attention: head width %d (supported: 32, 64, 96, 128)", hd);
  }
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// ---- the GroupQueryAttention operator --------------------------------------------------------------------------------
// The GroupQueryAttention operator on f32 tensors (no mask).  The `group` query heads of a kv head and the query
// positions together are the rows of one problem per (sequence, kv head): R = group * Sq rows against Sk keys, so a
// single decode position of four heads fills one row tile instead of four.  A workgroup of eight waves is RW row waves
// (16 QT rows each) times KS = 8 / RW key groups; a key group streams its stages of KB keys through LDS, converted to
// fp16 on the way in and V transposed into slabs of eight positions per channel, where all its row waves read them.
// What bounds that is the f32 K / V every workgroup has to take in (512 KB for 512 keys of 128 channels, 115 GB/s per CU
// from L2), so a workgroup gets as many rows as still leave one workgroup per CU, the waves left over split the keys
// and are merged through LDS, and where even that leaves CUs idle (decode: 8 workgroups) the keys are split over the
// grid too, with the partial results merged by a second kernel: one query x 2048 keys 9.5 + 5.7 us.
// PRE: where several workgroups share a kv head, its stages are converted once by a kernel in front (3.2 us for 512 keys of 8
// heads), travel to LDS by LDS-direct loads ahead of their use, and sixteen waves of one row tile each work on them: 512 queries
// x 512 keys, 32 heads over 8 of 128: 18.3 -> 14.0 us in all, 13.0 with the row tiles' softmax side by side and no rescaling in steps
// that need none.  Its 10 us: 1.9 until the first stage and q are there, 6 of stages, 1.7 the merge and the stores.
// QT: row tiles per wave; RW 1 is the form for few rows (wave-private stages: no barrier in the loop).
template <int HD, int RW, int QT, bool PRE = false>
struct FlatCfg {
  static constexpr int WAVES = PRE && QT == 1 ? 16 : 8, THREADS = 64 * WAVES;
  static constexpr int KS = WAVES / RW, T = 64 * RW;             // key groups, threads of one
  static constexpr int KB = PRE || RW <= 2 ? 32 : 16 * RW;       // keys per stage: the same registers per thread whatever RW
  static constexpr int NBUF = PRE ? (KS > 2 ? 2 : 4) : (RW == 1 ? 1 : 2);
  static constexpr int PITCH = HD > 64 ? 16 : (HD > 32 ? 8 : 4);  // K row pitch in 16-byte pieces
  static constexpr int K_BYTES = KB * PITCH * 16, V_BYTES = (KB / 8) * HD * 16, ST_BYTES = K_BYTES + V_BYTES;
  static constexpr int ROWS = RW * 16 * QT;
  static constexpr int OP = HD + 4;                      // floats per row of the merge buffer
  static constexpr int MERGE_BYTES = KS > 1 ? KS * ROWS * (OP + 2) * 4 : 0;
  static constexpr int Q_AT = KS * NBUF * ST_BYTES;      // PRE: where q changes to operand order
  static constexpr int LOOP_BYTES = Q_AT + (PRE ? ROWS * HD * 2 : 0);
  static constexpr int LDS = LOOP_BYTES > MERGE_BYTES ? LOOP_BYTES : MERGE_BYTES;
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

struct FlatArgs {
  const float *q, *k, *v;
  float *out, *part;       // part: [b * Hkv][gs][R][HD + 2] when gs > 1 (un-normalised output, maximum, sum)
  int Sq, Sk, Hq, Hkv, group, R, gs;  // Sq: query positions from one sequence to the next; R: rows of this launch
  int v16;                 // v is 16-byte aligned
  const uint8_t *pre;      // PRE: the stages of every (sequence, kv head) as they lie in LDS
  uint32_t magic;          // ceil(2^32 / group): row / group = the high half of row * magic (0: divide)
  float scale;             // log2(e) / sqrt(head width)
};

// Where the 16-byte piece (row, piece) of a stage's K lies in LDS
template <typename C>
__device__ __forceinline__ int flat_k_at(int row, int piece) {
  return (row * C::PITCH + (piece ^ ((((row >> 3) & 3) * 4 + (row & 3)) / (16 / C::PITCH)))) * 16;
}

// The stages of every (sequence, kv head) once, as gqa_flat_kernel has them in LDS: fp16, K swizzled, V in slabs of eight
// positions per channel (positions past the end 0).  What that kernel would do once per workgroup: with 32 workgroups to a
// kv head (512 queries of four heads, 64 rows each) 32 times.
template <int HD>
__global__ void __launch_bounds__(256) gqa_flat_prepare_kernel(FlatArgs p, uint8_t *__restrict__ pre, int stages) {
  using C = FlatCfg<HD, 4, 1, true>;  // (a stage is the same in all forms)
  constexpr int KB = C::KB, CPR = HD / 8, K_PIECES = KB * CPR, V_UNITS = (KB / 8) * (HD / 4), BLOCKS = (K_PIECES + V_UNITS + 255) / 256;
  const int nb = blockIdx.x, b = nb / p.Hkv, kvh = nb % p.Hkv, st = blockIdx.y / BLOCKS, idx = (int)(blockIdx.y % BLOCKS) * 256 + (int)threadIdx.x;
  const size_t kv_s = (size_t)p.Hkv * HD, base = (size_t)b * p.Sk * kv_s + (size_t)kvh * HD;
  const int left = min(KB, p.Sk - st * KB);
  uint8_t *dst = pre + ((size_t)nb * stages + st) * C::ST_BYTES;
  if (idx < K_PIECES) {
    const int row = idx / CPR, piece = idx % CPR;
    const float *src = p.k + base + (size_t)(st * KB + min(row, left - 1)) * kv_s + piece * 8;
    *reinterpret_cast<half8_t *>(dst + flat_k_at<C>(row, piece)) = load8<float>(src);
  } else if (idx < K_PIECES + V_UNITS) {
    const int u = idx - K_PIECES, pos = u / (HD / 4) * 8, ch = u % (HD / 4) * 4;
    float v[8][4];
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float *src = p.v + base + (size_t)(st * KB + min(pos + e, left - 1)) * kv_s + ch;
      if (p.v16) {
        const float4_t q = *reinterpret_cast<const float4_t *>(src);
#pragma unroll
        for (int i = 0; i < 4; i++) v[e][i] = q[i];
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) v[e][i] = src[i];
      }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
      half8_t h;
#pragma unroll
      for (int e = 0; e < 8; e++) h[e] = pos + e < left ? (_Float16)v[e][i] : (_Float16)0.0f;
      *reinterpret_cast<half8_t *>(dst + C::K_BYTES + (u * 4 + i) * 16) = h;
    }
  }
}

template <int HD, int RW, int QT, bool PRE>
__global__ void __launch_bounds__((FlatCfg<HD, RW, QT, PRE>::THREADS)) gqa_flat_kernel(FlatArgs p) {
  using C = FlatCfg<HD, RW, QT, PRE>;
  static_assert(!PRE || C::ST_BYTES % 1024 == 0, "a stage travels in KiB");
  constexpr int KK = HD / 32, DT = HD / 16, KB = C::KB, PITCH = C::PITCH, RPW = 16 / PITCH, CPR = HD / 8, T = C::T, KS = C::KS;
  constexpr int K_PIECES = KB * CPR, V_UNITS = (KB / 8) * (HD / 4);  // V unit: eight positions x four channels
  constexpr int K_LD = (K_PIECES + T - 1) / T, V_LD = (V_UNITS + T - 1) / T;
  // the values are read behind the scores' MFMAs and arrive during the softmax, where registers allow it
  constexpr bool V_EARLY = PRE && QT == 1;
  extern __shared__ __attribute__((aligned(16))) uint8_t flat_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const int kg = wave / RW, rw = wave % RW, gt = tid - kg * T;  // key group, row wave, thread of the group
  // kv heads are the fast grid dimension: with eight of them the workgroups of one share an XCD, and its L2 holds one head
  const int nb = blockIdx.x, b = nb / p.Hkv, kvh = nb % p.Hkv, gs = blockIdx.z;
  const int row0 = (int)blockIdx.y * C::ROWS + rw * 16 * QT;
  uint8_t *lds = flat_lds + kg * C::NBUF * C::ST_BYTES;
  const size_t q_s = (size_t)p.Hq * HD, kv_s = (size_t)p.Hkv * HD;
  const float *kbase = p.k + (size_t)b * p.Sk * kv_s + (size_t)kvh * HD;
  const float *vbase = p.v + (size_t)b * p.Sk * kv_s + (size_t)kvh * HD;
  const int stages = (p.Sk + KB - 1) / KB, st_lo = (int)((long long)stages * gs / p.gs), st_hi = (int)((long long)stages * (gs + 1) / p.gs);
  const int iters = (st_hi - st_lo + KS - 1) / KS;

  // where row `row` of this problem starts in q and out
  auto row_offset = [&](int row) {
    const int qpos = p.magic ? (int)__umulhi((uint32_t)row, p.magic) : row / p.group;
    return ((size_t)b * p.Sq + qpos) * q_s + (size_t)(kvh * p.group + row - qpos * p.group) * HD;
  };
  float4_t kr[K_LD][2], vr[V_LD][8];
  // A stage's base is wave-uniform and a lane's byte offsets inside a whole stage are the same for every stage: 32 bits
  // each, worked out once.  In the last stage rows past the end repeat the last key (their positions are masked).
  const uint32_t ks = (uint32_t)kv_s * 4u;  // bytes from one key to the next
  uint32_t koff[K_LD], voff[V_LD];
  // The loads of a round end with a wave's last piece, not inside a wave: lanes past the end repeat the last piece (and drop
  // it in stash).  A guard per lane there made the registers of a load live across both sides of it: 59 of them spilled at
  // head width 96 with few rows (one query x 2048 keys 15.7 us, 12.6 without; 512 x 512 16.2 -> 15.1).
  auto wave_has = [&](int j, int count) { return count % T == 0 || rw * 64 + T * j < count; };  // uniform
  auto unit = [&](int j, int count) { return (uint32_t)(count % T == 0 ? gt + T * j : min(gt + T * j, count - 1)); };
#pragma unroll
  for (int j = 0; j < K_LD; j++) koff[j] = unit(j, K_PIECES) / CPR * ks + unit(j, K_PIECES) % CPR * 32u;
#pragma unroll
  for (int j = 0; j < V_LD; j++) voff[j] = unit(j, V_UNITS) / (HD / 4) * 8u * ks + unit(j, V_UNITS) % (HD / 4) * 16u;
  auto fetch = [&](int st) {
    const char *kst = reinterpret_cast<const char *>(kbase) + (size_t)st * KB * ks, *vst = reinterpret_cast<const char *>(vbase) + (size_t)st * KB * ks;
    if (p.v16 && (st + 1) * KB <= p.Sk) {  // uniform
      // (opaque to the optimiser, or it hoists base + offset out of the loop as 64-bit addresses per lane and load)
#pragma unroll
      for (int j = 0; j < K_LD; j++) asm volatile("" : "+v"(koff[j]));
#pragma unroll
      for (int j = 0; j < V_LD; j++) asm volatile("" : "+v"(voff[j]));
#pragma unroll
      for (int j = 0; j < K_LD; j++) {
        if (wave_has(j, K_PIECES)) {
          kr[j][0] = *reinterpret_cast<const float4_t *>(kst + koff[j]);
          kr[j][1] = *reinterpret_cast<const float4_t *>(kst + 16 + koff[j]);
        }
      }
#pragma unroll
      for (int j = 0; j < V_LD; j++) {
        if (wave_has(j, V_UNITS)) {
#pragma unroll
          for (int e = 0; e < 8; e++) vr[j][e] = *reinterpret_cast<const float4_t *>(vst + e * ks + voff[j]);
        }
      }
      return;
    }
    const uint32_t last = (uint32_t)min(KB, p.Sk - st * KB) - 1u;
#pragma unroll
    for (int j = 0; j < K_LD; j++) {
      const uint32_t idx = unit(j, K_PIECES);
      if (wave_has(j, K_PIECES)) {
        const char *src = kst + (min(idx / CPR, last) * ks + idx % CPR * 32u);
        kr[j][0] = *reinterpret_cast<const float4_t *>(src);
        kr[j][1] = *reinterpret_cast<const float4_t *>(src + 16);
      }
    }
#pragma unroll
    for (int j = 0; j < V_LD; j++) {
      const uint32_t idx = unit(j, V_UNITS);
      if (wave_has(j, V_UNITS)) {
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float *src = reinterpret_cast<const float *>(vst + (min(idx / (HD / 4) * 8 + e, last) * ks + idx % (HD / 4) * 16u));
#pragma unroll
          for (int u = 0; u < 4; u++) vr[j][e][u] = src[u];
        }
      }
    }
  };
  auto stash = [&](int buf, int st) {
    uint8_t *base = lds + buf * C::ST_BYTES;
    const int left = p.Sk - st * KB;  // keys of the stage that exist; the V of the others is 0 (0 * inf would not be)
#pragma unroll
    for (int j = 0; j < K_LD; j++) {
      const int idx = gt + T * j;
      if (K_PIECES % T == 0 || idx < K_PIECES) {
        const int row = idx / CPR, piece = idx % CPR;
        half8_t h;
#pragma unroll
        for (int e = 0; e < 8; e++) h[e] = (_Float16)kr[j][e >> 2][e & 3];
        *reinterpret_cast<half8_t *>(base + flat_k_at<C>(row, piece)) = h;
      }
    }
#pragma unroll
    for (int j = 0; j < V_LD; j++) {
      const int idx = gt + T * j;
      if (V_UNITS % T == 0 || idx < V_UNITS) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          half8_t h;
#pragma unroll
          for (int e = 0; e < 8; e++) h[e] = (_Float16)vr[j][e][u];
          if (left < KB) {  // uniform
#pragma unroll
            for (int e = 0; e < 8; e++)
              if (idx / (HD / 4) * 8 + e >= left) h[e] = (_Float16)0.0f;
          }
          *reinterpret_cast<half8_t *>(base + C::K_BYTES + (idx * 4 + u) * 16) = h;
        }
      }
    }
  };

  // PRE: a stage is one run of bytes and goes to LDS as it is; a wave moves every RW-th KiB of its group's, the last one again
  // where they do not come out even, and stages past the end repeat the last one: every wave has COPIES loads per stage
  constexpr int KIB = C::ST_BYTES / 1024, COPIES = (KIB + RW - 1) / RW;
  const uint32_t lds_at = (uint32_t)(size_t)lds, lane16 = lane * 16;
  auto copy = [&](int buf, int stage) {
    const uint8_t *src = p.pre + (size_t)__builtin_amdgcn_readfirstlane(nb * stages + min(stage, st_hi - 1)) * C::ST_BYTES;
#pragma unroll
    for (int j = 0; j < COPIES; j++) {
      const int kib = min(rw + RW * j, KIB - 1);
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane(lds_at + (uint32_t)(buf * C::ST_BYTES + kib * 1024))),
                   "v"(lane16), "s"(src + kib * 1024)
                   : "memory");
    }
  };

  int st = st_lo + kg;
  const bool any = st < st_hi;
  if constexpr (PRE) copy(0, st);
  else if (any) fetch(st);

  half8_t qf[QT][KK];
  if constexpr (PRE) {
    // The workgroup's rows come once, whole lines, and change to operand order through LDS.  (Every wave for itself, in pieces
    // of 32 bytes, the key groups all the same rows: 256 load instructions of 16 lines each, 3.2 us until the first stage
    // could start.)
    constexpr int Q_ALL = C::ROWS * (HD / 4), Q_LD = (Q_ALL + C::THREADS - 1) / C::THREADS;  // threads past the end repeat the last piece
    uint8_t *qs = flat_lds + C::Q_AT;
    float4_t qr[Q_LD];
#pragma unroll
    for (int j = 0; j < Q_LD; j++) {
      const int idx = min(tid + C::THREADS * j, Q_ALL - 1), row = min((int)blockIdx.y * C::ROWS + idx / (HD / 4), p.R - 1);  // rows past the end repeat the last one
      qr[j] = *reinterpret_cast<const float4_t *>(p.q + row_offset(row) + idx % (HD / 4) * 4);
    }
#pragma unroll
    for (int i = 1; i < C::NBUF - 1; i++) copy(i, st + i * KS);
    constexpr int QX = HD == 128 ? 15 : (HD == 64 ? 7 : 3);  // the 16-byte pieces of a row change places so that 16 rows meet different banks
#pragma unroll
    for (int j = 0; j < Q_LD; j++) {
      const int idx = min(tid + C::THREADS * j, Q_ALL - 1), row = idx / (HD / 4), ch = idx % (HD / 4);
      *reinterpret_cast<half4_t *>(qs + row * HD * 2 + (((ch >> 1) ^ (row & QX)) * 16) + (ch & 1) * 8) =
          half4_t{(_Float16)qr[j][0], (_Float16)qr[j][1], (_Float16)qr[j][2], (_Float16)qr[j][3]};
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < QT; u++) {
      const int row = rw * 16 * QT + 16 * u + r;
#pragma unroll
      for (int kk = 0; kk < KK; kk++) qf[u][kk] = *reinterpret_cast<const half8_t *>(qs + row * HD * 2 + ((4 * kk + c) ^ (row & QX)) * 16);
    }
  } else {
#pragma unroll
    for (int u = 0; u < QT; u++) {
      const int row = min(row0 + 16 * u + r, p.R - 1);  // rows past the end repeat the last one and are not stored
      const float *qrow = p.q + row_offset(row);
#pragma unroll
      for (int kk = 0; kk < KK; kk++) qf[u][kk] = load8<float>(qrow + 32 * kk + 8 * c);
    }
  }
  float m_run[QT], l_run[QT];
  float4_t o_acc[QT][DT];
#pragma unroll
  for (int u = 0; u < QT; u++) {
    m_run[u] = -INFINITY;
    l_run[u] = 0.0f;
#pragma unroll
    for (int t = 0; t < DT; t++) o_acc[u][t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  const bool active = row0 < p.R;  // uniform in the wave

  // 32 keys of a stage; layout and arithmetic as in gqa_shared_kv_kernel.  The scores of all row tiles come first and V
  // is read behind them: K and V fragments together would not fit beside the next stage's loads in flight.
  auto compute32 = [&](const uint8_t *base, int sub, int p0) {
    half8_t pf[QT], vv[DT];
    auto read_v = [&]() {
#pragma unroll
      for (int t = 0; t < DT; t++) vv[t] = *reinterpret_cast<const half8_t *>(base + C::K_BYTES + ((sub * 4 + c) * HD + 16 * t + r) * 16);
    };
    float4_t sc[QT][2];
    {
      half8_t kf[2][KK];
#pragma unroll
      for (int j = 0; j < 2; j++) {
        const int row = 8 * (r >> 2) + 4 * j + (r & 3);
#pragma unroll
        for (int kk = 0; kk < KK; kk++)
          kf[j][kk] = *reinterpret_cast<const half8_t *>(base + ((sub * 32 + row) * PITCH + ((4 * kk + c) ^ (r / RPW))) * 16);
      }
#pragma unroll
      for (int u = 0; u < QT; u++) sc[u][0] = sc[u][1] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kk = 0; kk < KK; kk++)
#pragma unroll
        for (int u = 0; u < QT; u++)
#pragma unroll
          for (int j = 0; j < 2; j++) sc[u][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[j][kk], qf[u][kk], sc[u][j], 0, 0, 0);
    }
    if constexpr (V_EARLY) {
      __builtin_amdgcn_sched_barrier(0);
      read_v();
      __builtin_amdgcn_sched_barrier(0);
    }
    if (p0 + 32 > p.Sk) {  // uniform
#pragma unroll
      for (int u = 0; u < QT; u++)
#pragma unroll
        for (int e = 0; e < 8; e++)
          if (p0 + 8 * c + e >= p.Sk) sc[u][e >> 2][e & 3] = -INFINITY;  // (an existing key's scores repeated)
    }
    softmax_step<QT, DT>(sc, p.scale, m_run, l_run, o_acc, pf);
    if constexpr (!V_EARLY) {
      __builtin_amdgcn_sched_barrier(0);
      read_v();
    }
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
      for (int u = 0; u < QT; u++) o_acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vv[t], pf[u], o_acc[u][t], 0, 0, 0);
  };
  auto compute = [&](int stage_index, int buf) {
    if (!active) return;
#pragma unroll 1
    for (int sub = 0; sub < KB / 32; sub++) {
      const int p0 = stage_index * KB + sub * 32;
      if (p0 < p.Sk) compute32(lds + buf * C::ST_BYTES, sub, p0);
    }
  };

  if constexpr (RW == 1) {
    // the wave's own stages: LDS serves a wave's accesses in order, only the compiler must keep that order
    for (; st < st_hi; st += KS) {
      stash(0, st);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (st + KS < st_hi) fetch(st + KS);
      compute(st, 0);
      asm volatile("" ::: "memory");
    }
  } else if constexpr (PRE) {
    int buf = 0;
    for (int it = 0; it < iters; it++, st += KS) {  // uniform in the workgroup
      // this wave's part of the stage has landed and its reads of the last one have returned; then everyone's
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((C::NBUF - 2) * COPIES) : "memory");
      copy(buf == 0 ? C::NBUF - 1 : buf - 1, st + (C::NBUF - 1) * KS);
      if (st < st_hi) compute(st, buf);
      buf = buf + 1 == C::NBUF ? 0 : buf + 1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // nothing is in flight to LDS any more
  } else {
    if (any) stash(0, st);
    __syncthreads();
    for (int it = 0; it < iters; it++, st += KS) {  // uniform in the workgroup
      const bool more = st + KS < st_hi;
      if (more) fetch(st + KS);
      if (st < st_hi) compute(st, it & 1);
      if (more) stash((it + 1) & 1, st + KS);
      __syncthreads();
    }
  }

#pragma unroll
  for (int u = 0; u < QT; u++) l_run[u] = sum_xor16_xor32(l_run[u]);
  // lane (r, c) holds O^T[16 t + 4c + e][row r]
  const size_t part_row0 = ((size_t)nb * p.gs + gs) * p.R;
  if constexpr (KS == 1) {
#pragma unroll
    for (int u = 0; u < QT; u++) {
      const int row = row0 + 16 * u + r;
      if (row >= p.R) continue;
      float *dst;
      float f = 1.0f;
      if (p.gs > 1) {
        dst = p.part + (part_row0 + row) * (HD + 2);
        if (c == 0) {
          dst[HD] = m_run[u];
          dst[HD + 1] = l_run[u];
        }
#pragma unroll
        for (int t = 0; t < DT; t++)
#pragma unroll
          for (int e = 0; e < 4; e++) dst[16 * t + 4 * c + e] = o_acc[u][t][e];
        continue;
      }
      dst = p.out + row_offset(row);
      f = l_run[u] > 0.0f ? 1.0f / l_run[u] : 0.0f;
#pragma unroll
      for (int t = 0; t < DT; t++) store4<float>(dst + 16 * t + 4 * c, o_acc[u][t][0] * f, o_acc[u][t][1] * f, o_acc[u][t][2] * f, o_acc[u][t][3] * f);
    }
  } else {
    // merge the key groups through LDS (the stages are done with it)
    __syncthreads();
    float *o_s = reinterpret_cast<float *>(flat_lds);                       // [KS][ROWS][OP]
    float *ml = o_s + KS * C::ROWS * C::OP;                                 // [KS][ROWS][2]
#pragma unroll
    for (int u = 0; u < QT; u++) {
      const int lr = rw * 16 * QT + 16 * u + r;
      float *dst = o_s + (kg * C::ROWS + lr) * C::OP;
#pragma unroll
      for (int t = 0; t < DT; t++) *reinterpret_cast<float4_t *>(dst + 16 * t + 4 * c) = o_acc[u][t];
      if (c == 0) {
        ml[(kg * C::ROWS + lr) * 2] = m_run[u];
        ml[(kg * C::ROWS + lr) * 2 + 1] = l_run[u];
      }
    }
    __syncthreads();
    for (int idx = tid; idx < C::ROWS * (HD / 4); idx += C::THREADS) {
      const int lr = idx / (HD / 4), d4 = idx % (HD / 4) * 4, row = (int)blockIdx.y * C::ROWS + lr;
      if (row >= p.R) continue;
      float M = -INFINITY, L = 0.0f;
#pragma unroll
      for (int g = 0; g < KS; g++) M = fmaxf(M, ml[(g * C::ROWS + lr) * 2]);
      float4_t o = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int g = 0; g < KS; g++) {
        const float mg = ml[(g * C::ROWS + lr) * 2];
        const float f = mg == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mg - M);
        L += ml[(g * C::ROWS + lr) * 2 + 1] * f;
        o += *reinterpret_cast<const float4_t *>(o_s + (g * C::ROWS + lr) * C::OP + d4) * f;
      }
      if (p.gs > 1) {
        float *dst = p.part + (part_row0 + row) * (HD + 2);
        if (d4 == 0) {
          dst[HD] = M;
          dst[HD + 1] = L;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) dst[d4 + e] = o[e];
        continue;
      }
      const float inv = L > 0.0f ? 1.0f / L : 0.0f;
      store4<float>(p.out + row_offset(row) + d4, o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
    }
  }
}

// merges the grid's key splits: one thread per (row, channel)
__global__ void __launch_bounds__(256) gqa_flat_merge_kernel(FlatArgs p, int hd, int total_rows) {
  const int idx = (int)(blockIdx.x * 256 + threadIdx.x), grow = idx / hd, ch = idx % hd;
  if (grow >= total_rows) return;
  const int nb = grow / p.R, row = grow % p.R;
  const size_t step = (size_t)p.R * (hd + 2);
  const float *src = p.part + ((size_t)nb * p.gs * p.R + row) * (hd + 2);
  float M = -INFINITY, L = 0.0f, o = 0.0f;
  for (int g = 0; g < p.gs; g++) M = fmaxf(M, src[g * step + hd]);
  for (int g = 0; g < p.gs; g++) {
    const float mg = src[g * step + hd];
    const float f = mg == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(mg - M);
    L += src[g * step + hd + 1] * f;
    o += src[g * step + ch] * f;
  }
  p.out[((size_t)(nb / p.Hkv) * p.Sq + row / p.group) * p.Hq * hd + (size_t)(nb % p.Hkv * p.group + row % p.group) * hd + ch] =
      L > 0.0f ? o / L : 0.0f;
}

template <int HD, int RW, int QT, bool PRE>
int32_t gqa_flat_go(const FlatArgs &p, int nbs, hipStream_t s) {
  using C = FlatCfg<HD, RW, QT, PRE>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kern = gqa_flat_kernel<HD, RW, QT, PRE>;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS); });
  YSCV_HIP_TRY(attr_err);
  hipLaunchKernelGGL(kern, dim3((unsigned)nbs, (unsigned)((p.R + C::ROWS - 1) / C::ROWS), (unsigned)p.gs), dim3(C::THREADS), C::LDS, s, p);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// Which form takes a problem of R rows x Sk keys per (sequence, kv head), by estimated time in units of 0.1 us: rounds of
// workgroups over the CUs x (start and merge + steps of keys), and what runs in front or behind.  The prepared forms take
// 32 keys of each of their 16-wave key groups in 1.6 us at 128 channels whatever their rows; the form for few rows takes 256
// keys in 2.9, bound by the f32 K / V that every 16 rows take in again.  Measured (us): 512 x 512, 32 heads over 8 of 128: 18.3 in
// 64 rows converting for themselves, 14.0 prepared; 1000 x 1111 42 -> 34.5 in 128 rows; 4 x 300 x 2000, 8 over 8: 79 in 16
// rows, 43 in 64; 200 x 2000, 32 over 8: 47 -> 28.6, keys in two parts; 4 x 1024 x 2048, 32 over 8 of 64: 151 -> 133 in 256 rows.
// In 256 rows the preparation is paid back late: 4 x 512 x 512 at 128 channels 35 as it was, 38 prepared, 2 x 1024 x 1024 57 and 58.
struct FlatPlan {
  int rows;  // 16, 64, 128 or 256
  bool pre;
  int gs;    // parts the keys are split into over the grid
};
FlatPlan flat_plan(int nbs, int R, int Sk, int hd, int num_cus, bool may_prepare) {
  auto wgs = [&](int rows) { return (long long)nbs * ((R + rows - 1) / rows); };
  auto rounds = [&](long long n) { return (n + num_cus - 1) / num_cus; };
  auto ceil_of = [](long long n, long long d) { return (n + d - 1) / d; };
  // without a prepared copy: the most rows that still give every CU a workgroup; 16 rows and a split of the keys over the grid
  // where no choice does.  A split pays where it takes whole rounds of stages off the longest workgroup.
  FlatPlan best{wgs(256) >= num_cus ? 256 : (wgs(128) >= num_cus ? 128 : (wgs(64) >= num_cus ? 64 : 16)), false, 1};
  if (best.rows == 16) {
    const long long steps = ceil_of(Sk, 32 * 8), room = num_cus / wgs(16);
    const long long gs = steps < room ? steps : room;
    if (gs >= 2) best.gs = (int)(gs > 64 ? 64 : gs);
  }
  if (!may_prepare || (best.rows == 256 && Sk <= 8 * hd)) return best;
  const long long step = 8 + 8 * hd / 128, prep = 30 + (long long)nbs * Sk * hd * 8 / 330000;
  long long cost;
  if (best.rows == 16) cost = rounds(wgs(16) * best.gs) * (30 + 29 * hd / 128 * ceil_of(ceil_of(Sk, 256), best.gs)) + (best.gs > 1 ? 50 : 0);
  else cost = rounds(wgs(best.rows)) * (80 + (step + 4) * ceil_of(Sk, 8192 / best.rows));
  for (int rows : {64, 128, 256})
    for (int gs : {1, 2, 4}) {
      const long long steps = ceil_of(Sk, 8192 / rows);  // 4, 2, 1 key groups
      if ((R + rows - 1) / rows > 65535) continue;  // a grid's y
      if (gs > 1 && (rows > 64 || wgs(rows) * gs > num_cus || steps < 4 * gs)) continue;
      const long long c = prep + rounds(wgs(rows) * gs) * (50 + step * ceil_of(steps, gs)) + (gs > 1 ? 50 : 0);
      if (c < cost) {
        cost = c;
        best = FlatPlan{rows, true, gs};
      }
    }
  return best;
}

template <int HD>
int32_t gqa_flat_launch(FlatArgs p, int B, int num_cus, hipStream_t s) {
  const int nbs = B * p.Hkv;
  using C = FlatCfg<HD, 4, 1, true>;
  constexpr unsigned BLOCKS = (C::KB * (HD / 8) + C::KB / 8 * (HD / 4) + 255) / 256;  // of the preparation, per stage
  const size_t stages = ceil_div((size_t)p.Sk, (size_t)C::KB), pre_bytes = (size_t)nbs * stages * C::ST_BYTES;
  auto part_bytes = [&](const FlatPlan &f) { return f.gs > 1 ? (size_t)nbs * f.gs * p.R * (HD + 2) * sizeof(float) : 0; };
  FlatPlan f = flat_plan(nbs, p.R, p.Sk, HD, num_cus, pre_bytes <= ((size_t)64 << 20) && stages * BLOCKS <= 65535);
  Scratch scratch;
  if (f.pre && scratch.take(pre_bytes + part_bytes(f), s) != YSCV_HIP_OK) {
    (void)hipGetLastError();  // no memory for the copy: the forms that need none
    f = flat_plan(nbs, p.R, p.Sk, HD, num_cus, false);
  }
  p.gs = f.gs;
  if (f.pre) {
    hipLaunchKernelGGL((gqa_flat_prepare_kernel<HD>), dim3((unsigned)nbs, (unsigned)stages * BLOCKS), dim3(256), 0, s, p, scratch.as<uint8_t>(), (int)stages);
    YSCV_HIP_TRY(hipGetLastError());
    p.pre = scratch.as<uint8_t>();
    p.part = scratch.as<float>(pre_bytes);
    if (f.rows == 64) YSCV_TRY((gqa_flat_go<HD, 4, 1, true>(p, nbs, s)));
    else if (f.rows == 128) YSCV_TRY((gqa_flat_go<HD, 8, 1, true>(p, nbs, s)));
    else YSCV_TRY((gqa_flat_go<HD, 16, 1, true>(p, nbs, s)));
  } else {
    if (f.gs > 1) {
      YSCV_TRY(scratch.take(part_bytes(f), s));
      p.part = scratch.as<float>();
    }
    if (f.rows == 256) YSCV_TRY((gqa_flat_go<HD, 8, 2, false>(p, nbs, s)));
    else if (f.rows == 128) YSCV_TRY((gqa_flat_go<HD, 4, 2, false>(p, nbs, s)));
    else if (f.rows == 64) YSCV_TRY((gqa_flat_go<HD, 2, 2, false>(p, nbs, s)));
    else YSCV_TRY((gqa_flat_go<HD, 1, 1, false>(p, nbs, s)));
  }
  if (p.gs > 1) {
    const size_t total = (size_t)nbs * p.R * HD;
    hipLaunchKernelGGL(gqa_flat_merge_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, p, HD, nbs * p.R);
    YSCV_HIP_TRY(hipGetLastError());
  }
  return YSCV_HIP_OK;
}

// ---- RMSNorm over the last axis, f32 in and out ---------------------------------------------------------------
// Latency- and HBM-bound: the row (KEEP x 1024 values, sixteen bytes per lane and load) and, with GAIN, gamma behind it are asked for at once
// and wait in registers, so that one memory round trip is all there is between launch and stores (each load of the row was waited for inside its
// test, and gamma behind the sum).  us: 512 x 8192 6.3 -> 5.7, 4096 x 1024 6.3 -> 5.1, 2048 x 4096 10.7 -> 10.3, 512 x 4096 with the
// attention behind it 19.5 -> 19.1.  KEEP 0: longer, odd or unaligned rows, read twice.
template <int KEEP, bool GAIN>
__global__ void __launch_bounds__(256) rms_norm_f32_kernel(const float *__restrict__ x, const float *__restrict__ gamma, int d,
                                                           float eps, float *__restrict__ y) {
  __shared__ float red[4];
  const float *row = x + (size_t)blockIdx.x * d;
  float *out = y + (size_t)blockIdx.x * d;
  constexpr int REGS = KEEP > 0 ? KEEP : 1;
  float4_t v[REGS], g[REGS];
  float ss = 0.0f;
  if constexpr (KEEP > 0) {
    norm_load<KEEP, GAIN>(row, gamma, d, v, g);
#pragma unroll
    for (int j = 0; j < KEEP; j++) ss += (v[j][0] * v[j][0] + v[j][1] * v[j][1]) + (v[j][2] * v[j][2] + v[j][3] * v[j][3]);
  } else {
    for (int i = threadIdx.x; i < d; i += 256) ss += row[i] * row[i];
  }
  ss = wave_sum(ss);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
  __syncthreads();
  ss = red[0] + red[1] + red[2] + red[3];
  // rms = sqrt(sum / n + eps); inv_rms = 1 / rms; y = x * inv_rms * gamma (ops/norm.rs:1507-1516, in that order)
  const float inv_rms = 1.0f / sqrtf(ss / (float)d + eps);
  if constexpr (KEEP > 0) {
#pragma unroll
    for (int j = 0; j < KEEP; j++) {
      const int i = (j * 256 + (int)threadIdx.x) * 4;
      if (i < d) *reinterpret_cast<float4_t *>(out + i) = v[j] * inv_rms * (GAIN ? g[j] : *reinterpret_cast<const float4_t *>(gamma + i));
    }
  } else {
    for (int i = threadIdx.x; i < d; i += 256) out[i] = row[i] * inv_rms * gamma[i];
  }
}

// ---- rotate-half RoPE in place on [seq][heads][d] f32 ------------------------------------------------------------
__global__ void __launch_bounds__(64) rope_f32_kernel(float *__restrict__ x, int heads, int d, int seq_offset, float theta) {
  const int pos = blockIdx.y, head = blockIdx.x;
  float *row = x + ((size_t)pos * heads + head) * d;
  const int half_d = d / 2;
  const float abs_pos = (float)(pos + seq_offset);
  for (int i = threadIdx.x; i < half_d; i += 64) {
    const float inv_freq = 1.0f / powf(theta, 2.0f * (float)i / (float)d);
    float sn, cs;
    sincosf(inv_freq * abs_pos, &sn, &cs);
    const float x0 = row[i], x1 = row[i + half_d];
    row[i] = x0 * cs - x1 * sn;
    row[i + half_d] = x0 * sn + x1 * cs;
  }
}


// ---- small kernels of the prompt pass (rows = consecutive positions of one sequence) ------------------------------
// {cos, sin} of every pair at the positions of a prompt pass, row p of the table for position p0 + p: once for all layers and heads
__global__ void __launch_bounds__(256) prefill_angles_kernel(int p0, int positions, int hd, float theta, float2 *__restrict__ angles) {
  const int idx = (int)(blockIdx.x * 256 + threadIdx.x), half_d = hd / 2;
  if (idx >= positions * half_d) return;
  const SinCos a = rope_sincos(theta, idx % half_d, hd, p0 + idx / half_d);
  angles[idx] = float2{a.cs, a.sn};
}

// RoPE on the q and k heads of every row (row i sits at position start_pos + i), k and v appended to batch row 0 of
// the cache: the arithmetic of the decode step's rope + append, one launch for all rows.  Workgroups take the (up
// to eight) rows whose positions share one 8-position slab of the V layout; the values of a channel at the slab's positions leave as one
// 16-byte store where the whole slab is new.  Memory-bound: a thread has eight pairs of one position, whose angles it keeps, in up to
// ROPE_HEADS heads, and asks for all of that and its first channel of v at once: one memory round trip.  With the angles worked out here,
// once per layer and workgroup, and an item at a time behind them it was 6 .. 8 in turn.  us a launch, 40 heads of 128: 2048 rows
// 12.2 -> 9.8 (5.1 TB/s), 1500 10.6 -> 7.8, 700 7.0 -> 5.9; 18 heads of 64: 43 rows 4.3 -> 3.1, from 500 rows on no change; the angles
// take 3.3 a pass.
constexpr int ROPE_HEADS = 3;
__global__ void __launch_bounds__(256) prefill_rope_append_kernel(_Float16 *__restrict__ qkv, int rows, int start_pos, int hq, int hkv,
                                                                  int hd, const float2 *__restrict__ angles, int max_ctx, _Float16 *__restrict__ kc,
                                                                  _Float16 *__restrict__ vc, int parts) {
  const int slab = start_pos / 8 + (int)blockIdx.x;
  const int p_lo = max(start_pos, slab * 8), p_hi = min(start_pos + rows, slab * 8 + 8);  // positions [p_lo, p_hi)
  const size_t row_elems = (size_t)(hq + 2 * hkv) * hd;
  const int half_d = hd / 2, slots = hq + hkv, vecs = half_d / 8, channels = hkv * hd;
  const int first = (int)threadIdx.x + 256 * (int)blockIdx.y, step = 256 * parts;
  // Thread `first` of the slab's step: the (first % width)-th eight pairs of a head, positions last, in heads head0, head0 + stride, ..
  // Requests past the ends repeat a neighbour's and are not stored.
  const int width = 8 * vecs, stride = step / width, head0 = first / width, pair8 = first % width;
  const int pos = slab * 8 + pair8 / vecs, i0 = pair8 % vecs * 8, row = min(max(pos, p_lo), p_hi - 1) - start_pos;
  _Float16 *at = qkv + (size_t)row * row_elems + i0;
  half8_t x0[ROPE_HEADS], x1[ROPE_HEADS];
  float4_t ang[4];
#pragma unroll
  for (int u = 0; u < ROPE_HEADS; u++) {
    const _Float16 *src = at + min(head0 + u * stride, slots - 1) * hd;
    x0[u] = *reinterpret_cast<const half8_t *>(src);
    x1[u] = *reinterpret_cast<const half8_t *>(src + half_d);
  }
  const float4_t *arow = reinterpret_cast<const float4_t *>(angles + (size_t)row * half_d + i0);
#pragma unroll
  for (int j = 0; j < 4; j++) ang[j] = arow[j];
  // v: channel ch of kv head kvh at the slab's positions; those that are not of this call repeat a neighbour and are not stored
  half8_t v;
  auto load_v = [&](int idx) {
    const _Float16 *src = qkv + (size_t)slots * hd + min(idx, channels - 1);
#pragma unroll
    for (int e = 0; e < 8; e++) v[e] = src[(size_t)(min(max(slab * 8 + e, p_lo), p_hi - 1) - start_pos) * row_elems];
  };
  auto put_v = [&](int idx) {
    if (idx >= channels) return;
    const int kvh = idx / hd, ch = idx % hd;
    _Float16 *dst = vc + (((size_t)kvh * (max_ctx / 8) + slab) * hd + ch) * 8;
    if (p_hi - p_lo == 8) {
      *reinterpret_cast<half8_t *>(dst) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 8; e++)
        if (slab * 8 + e >= p_lo && slab * 8 + e < p_hi) dst[e] = v[e];
    }
  };
  load_v(first);
  if (head0 < stride && pos >= p_lo && pos < p_hi) {  // (threads behind the last whole width have no head)
#pragma unroll
    for (int u = 0; u < ROPE_HEADS; u++) {
      const int slot = head0 + u * stride;
      if (slot >= slots) break;
      half8_t y0, y1;
#pragma unroll
      for (int j = 0; j < 8; j++) {
        const float cs = ang[j / 2][j % 2 * 2], sn = ang[j / 2][j % 2 * 2 + 1];
        const float a = (float)x0[u][j], b = (float)x1[u][j];
        float f0 = fmaf(a, cs, -(b * sn)), f1 = fmaf(a, sn, b * cs);
        asm volatile("" : "+v"(f0), "+v"(f1));  // the f32 value exists before it is narrowed (no mixed-precision fma)
        y0[j] = (_Float16)f0;
        y1[j] = (_Float16)f1;
      }
      _Float16 *dst = slot < hq ? at + slot * hd : kc + ((size_t)(slot - hq) * max_ctx + pos) * hd + i0;
      *reinterpret_cast<half8_t *>(dst) = y0;
      *reinterpret_cast<half8_t *>(dst + half_d) = y1;
    }
  }
  put_v(first);
  for (int idx = first + step; idx < channels; idx += step) {
    load_v(idx);
    put_v(idx);
  }
}

__global__ void bias_add_f16_kernel(_Float16 *__restrict__ x, const _Float16 *__restrict__ bias, size_t rows, size_t n) {
  for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < rows * n; idx += (size_t)gridDim.x * blockDim.x)
    x[idx] = (_Float16)((float)x[idx] + (float)bias[idx % n]);
}

unsigned flat_grid(size_t n) {
  const size_t b = (n + 255) / 256;
  return (unsigned)(b > 65535 ? 65535 : (b < 1 ? 1 : b));
}

}  // namespace

size_t prefill_angles_bytes(size_t rows, int hd) { return rows * (hd / 2) * sizeof(float2); }
int32_t launch_prefill_angles(int rows, int start_pos, int hd, float theta, void *angles, hipStream_t s) {
  const size_t total = (size_t)rows * (hd / 2);
  if (total > 0x7fffffff) return set_error(YSCV_HIP_ERR_UNSUPPORTED, "rope: %d rows of head width %d", rows, hd);
  hipLaunchKernelGGL(prefill_angles_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, start_pos, rows, hd, theta, static_cast<float2 *>(angles));
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}
int32_t launch_prefill_rope_append(_Float16 *qkv, int rows, int start_pos, int hq, int hkv, int hd, const void *angles, int max_ctx,
                                   _Float16 *kc, _Float16 *vc, hipStream_t s) {
  if (hd > 128 || hd % 16 != 0) return set_error(YSCV_HIP_ERR_UNSUPPORTED, "rope + append: head width %d", hd);
  const int slabs = (start_pos + rows - 1) / 8 - start_pos / 8 + 1, width = hd / 2;  // width: threads of a head
  // Workgroups of a slab: as many as cover its heads with ROPE_HEADS each; few slabs leave CUs idle and are spread further, down to a head each
  const int heads = hq + hkv, least = ((heads + ROPE_HEADS - 1) / ROPE_HEADS * width + 255) / 256, most = (heads * width + 255) / 256;
  const int parts = std::max(least, std::min(most, 512 / slabs));
  hipLaunchKernelGGL(prefill_rope_append_kernel, dim3(slabs, parts), dim3(256), 0, s, qkv, rows, start_pos, hq, hkv, hd,
                     static_cast<const float2 *>(angles), max_ctx, kc, vc, parts);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}
int32_t launch_bias_add_f16(_Float16 *x, const _Float16 *bias, size_t rows, size_t n, hipStream_t s) {
  hipLaunchKernelGGL(bias_add_f16_kernel, dim3(flat_grid(rows * n)), dim3(256), 0, s, x, bias, rows, n);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// Attention of the prompt pass against the decoder's fp16 cache of one layer.  qkv: [rows][(hq + 2 hkv) hd] with the query heads
// already rotated; out: [rows][hq hd].  The rows are consecutive positions start_pos .. of batch row 0, row i sees cache rows
// [0, start_pos + i].
int32_t launch_gqa_cache(const _Float16 *qkv, const _Float16 *kc, const _Float16 *vc, int rows, int start_pos, int hq, int hkv, int hd,
                         int max_ctx, _Float16 *out, hipStream_t s) {
  GqaArgs a{};
  a.q = qkv;
  a.k = kc;
  a.v = vc;
  a.out = out;
  a.k_s = hd;
  a.k_h = a.v_h = (long long)max_ctx * hd;
  a.Hq = hq;
  a.Hkv = hkv;
  a.scale = 1.0f / sqrtf((float)hd);
  a.B = 1;
  a.Sq = rows;
  a.Sk = start_pos + rows;
  a.causal_base = start_pos;
  a.q_s = (long long)(hq + 2 * hkv) * hd;
  a.o_s = (long long)hq * hd;
  // enough rows: the kernel that stages K / V in LDS for four waves (its K rows must be contiguous 16-byte pieces, which the
  // cache's are)
  if (rows >= 64 && (max_ctx & 7) == 0) return gqa_launch_shared_kv(a, hd, s);
  return gqa_launch_cache(a, hd, s);
}

extern "C" {

int32_t yscv_hip_rms_norm_dev(const float *x, const float *gamma, size_t rows, size_t d, float eps, float *y, void *stream) {
  const Context *ctx = nullptr;
  YSCV_TRY(ensure_context(&ctx));
  YSCV_REQUIRE(x && gamma && y, "null argument");
  YSCV_REQUIRE(std::isfinite(eps) && eps > 0.0f, "rms_norm: epsilon must be finite and > 0");
  YSCV_REQUIRE(d > 0 && d < ((size_t)1 << 31) && rows < ((size_t)1 << 31), "rms_norm: bad shape %zu x %zu", rows, d);
  const size_t step = (size_t)1 << 23;  // a grid holds less than 2^32 threads
  const bool vec = d % 4 == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(gamma)) & 15) == 0;
  for (size_t r0 = 0; r0 < rows; r0 += step) {
    auto go = [&](auto keep, auto gain) {
      hipLaunchKernelGGL((rms_norm_f32_kernel<decltype(keep)::value, decltype(gain)::value>), dim3((unsigned)std::min(step, rows - r0)), dim3(256), 0,
                         as_stream(stream), x + r0 * d, gamma, (int)d, eps, y + r0 * d);
    };
    if (vec) norm_keep(d, rows, (size_t)ctx->num_cus, go);
    else go(std::integral_constant<int, 0>{}, std::false_type{});
    YSCV_HIP_TRY(hipGetLastError());
  }
  return YSCV_HIP_OK;
}

int32_t yscv_hip_rope_dev(float *q, float *k, size_t num_q_heads, size_t num_kv_heads, size_t d_head, size_t seq_len,
                          size_t seq_offset, float theta, void *stream) {
  YSCV_TRY(ensure_context(nullptr));
  YSCV_REQUIRE(q && k, "null argument");
  YSCV_REQUIRE(d_head % 2 == 0 && d_head > 0, "rope: d_head must be even (got %zu)", d_head);
  YSCV_REQUIRE(seq_len + seq_offset < ((size_t)1 << 24), "rope: position beyond 2^24");
  YSCV_REQUIRE(seq_len < 65536 && num_q_heads < ((size_t)1 << 31) && num_kv_heads < ((size_t)1 << 31), "rope: shape too large");
  if (seq_len == 0) return YSCV_HIP_OK;
  hipStream_t s = as_stream(stream);
  if (num_q_heads > 0) {
    hipLaunchKernelGGL(rope_f32_kernel, dim3((unsigned)num_q_heads, (unsigned)seq_len), dim3(64), 0, s, q, (int)num_q_heads, (int)d_head,
                       (int)seq_offset, theta);
    YSCV_HIP_TRY(hipGetLastError());
  }
  if (num_kv_heads > 0) {
    hipLaunchKernelGGL(rope_f32_kernel, dim3((unsigned)num_kv_heads, (unsigned)seq_len), dim3(64), 0, s, k, (int)num_kv_heads, (int)d_head,
                       (int)seq_offset, theta);
    YSCV_HIP_TRY(hipGetLastError());
  }
  return YSCV_HIP_OK;
}

int32_t yscv_hip_gqa_attention_dev(const float *q, const float *k, const float *v, size_t batch, size_t seq_q, size_t seq_k,
                                   size_t num_q_heads, size_t num_kv_heads, size_t d_head, float *out, void *stream) {
  YSCV_TRY(ensure_context(nullptr));
  YSCV_REQUIRE(q && k && v && out, "null argument");
  YSCV_REQUIRE(num_q_heads > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0,
               "GroupQueryAttention: %zu query heads over %zu kv heads", num_q_heads, num_kv_heads);
  YSCV_REQUIRE(batch < 65536 && num_q_heads < 65536 && seq_q < ((size_t)1 << 24) && seq_k < ((size_t)1 << 24),
               "GroupQueryAttention: shape too large");
  YSCV_REQUIRE(((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) | reinterpret_cast<uintptr_t>(out)) & 15) == 0,
               "GroupQueryAttention: tensors must be 16-byte aligned");
  if (batch == 0 || seq_q == 0) return YSCV_HIP_OK;
  YSCV_REQUIRE(seq_k > 0, "GroupQueryAttention: no key positions");
  const Context *ctx = nullptr;
  YSCV_TRY(ensure_context(&ctx));
  FlatArgs p{};
  p.Sq = (int)seq_q;
  p.Sk = (int)seq_k;
  p.Hq = (int)num_q_heads;
  p.Hkv = (int)num_kv_heads;
  p.group = (int)(num_q_heads / num_kv_heads);
  p.v16 = (reinterpret_cast<uintptr_t>(v) & 15) == 0;
  p.scale = 1.44269504f / sqrtf((float)d_head);
  // exact while row * group < 2^32
  p.magic = p.group > 1 && p.group <= 256 ? (uint32_t)((((uint64_t)1 << 32) + p.group - 1) / p.group) : 0;
  // What one launch takes: 2^22 problems (2^32 threads along x) and 65535 workgroups of 256 rows along y.  Sequences and
  // query positions beyond that go in further launches.
  const size_t b_step = std::max<size_t>(1, ((size_t)1 << 22) / num_kv_heads), q_step = (size_t)65535 * 256 / p.group;
  for (size_t b0 = 0; b0 < batch; b0 += b_step) {
    for (size_t q0 = 0; q0 < seq_q; q0 += q_step) {
      const int bs = (int)std::min(b_step, batch - b0);
      p.R = p.group * (int)std::min(q_step, seq_q - q0);
      const size_t q_at = (b0 * seq_q + q0) * num_q_heads * d_head, kv_at = b0 * seq_k * num_kv_heads * d_head;
      p.q = q + q_at;
      p.out = out + q_at;
      p.k = k + kv_at;
      p.v = v + kv_at;
      switch (d_head) {
        case 32: YSCV_TRY(gqa_flat_launch<32>(p, bs, ctx->num_cus, as_stream(stream))); break;
        case 64: YSCV_TRY(gqa_flat_launch<64>(p, bs, ctx->num_cus, as_stream(stream))); break;
        case 96: YSCV_TRY(gqa_flat_launch<96>(p, bs, ctx->num_cus, as_stream(stream))); break;
        case 128: YSCV_TRY(gqa_flat_launch<128>(p, bs, ctx->num_cus, as_stream(stream))); break;
        default: return set_error(YSCV_HIP_ERR_UNSUPPORTED, "attention: head width %zu (supported: 32, 64, 96, 128)", d_head);
      }
    }
  }
  return YSCV_HIP_OK;
}

}  // extern "C"

}  // namespace yscv
