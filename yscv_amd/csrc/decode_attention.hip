// Attention of one decode step over the fp16 cache, with the rotary embedding, the cache append and the merge of the key ranges in
// the same launch.  Restates exec_grouped_query_attention over KvCache (crates/yscv-onnx/src/runner/linear.rs:552-646,
// kv_cache.rs:36-79) for one query position per sequence.
//
// A workgroup of eight waves takes up to sixteen query heads of one kv head of one sequence, and a share of its positions.  Bound
// by the read of K and V, so: few long workgroups (the shares are cut so that all of them are on the chip at once, and only
// above kAttMin positions), whole blocks of 32 positions per wave straight into registers, two in flight per wave (256 KB per CU).
//   S^T = K Q^T   a block's K rows are the A operand; row i of tile u is position 8 (i / 4) + 4 u + i % 4, so that a lane ends
//                 up with the weights of eight consecutive positions of one query head, which is
//   O^T += V^T P^T  the B operand here; A is a slab piece of the cache as it lies (eight positions of a channel).
// Shares of one kv head meet pairwise, two channels of a head at a time: a thread exchanges {maximum, sum of weights} with the first word of
// a slot and its two sums of weighted values with the second, both on their way at once.  Who finds the second word empty leaves; who
// finds it full merges (always in the order of the positions), empties the slot and goes on to the next level.  The partner's
// first word has been sent before its second one: it is what the exchange returned, or is about to take the place of this share's own
// one (the sign bit of the sum tells the two apart), a wait for memory and for no other workgroup.  One trip to memory per level (1.1 us);
// maximum and sum stay two f32, so that a share's weight is exact whatever the size of the scores.  ({value, log of the
// weights' sum} in one word: weights that are off by |score| 2^-24.  The second word sent when the first has arrived: 0.4 us more.
// Partials through agent-scope stores, an arrival counter and a last workgroup that reads them back: three trips, 5 us.)
// Chunks of 128 positions and a launch that merges them (attn_chunk_kernel) -> this: 32 heads over 8 of 128, 16 sequences of 2048
// positions 27.2 + 4.8 -> 25.4 us (5.3 TB/s; a step of 32 layers 2757 -> 2571), 8 sequences 2205 -> 2117 a step.  With fewer than 64
// (sequence, kv head) pairs a workgroup has to take in more than it can at 50 .. 60 GB/s, or the merge gets deep: 4 sequences of 1000
// positions 1697 -> 1739 a step, 2 of 2048 1547 -> 1602 (2 of 100: 1497 -> 1425).  16 heads over 2 of 64, where one workgroup per head
// and sequence walked all positions: 16 sequences of 2000 positions 1573 -> 963 us a step of 24 layers, 4 of 1000 950 -> 782, 16 of 360
// 974 -> 905, 2 of 100 no change.
#include <mutex>

#include "common.hpp"
#include "decoder.hpp"
#include "int4_common.hpp"
#include "rope.hpp"

namespace yscv {

namespace {

constexpr int AD_WAVES = 8, AD_THREADS = 64 * AD_WAVES, AD_Q = 16;
constexpr int kAttMin = 512;  // positions below which a share is not cut further: two blocks per wave (256: 0.5 % slower, 1024: up to 10 %)
constexpr uint64_t kEmpty = ~(uint64_t)0;  // a word nobody has been to (no pair is stored with this NaN in it)

typedef float float2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float2_t word_pair(uint64_t w) { return float2_t{__uint_as_float((uint32_t)w), __uint_as_float((uint32_t)(w >> 32))}; }
// mark: into the sign bit of y, which then is no negative number
__device__ __forceinline__ uint64_t swap_pair(uint64_t *slot, float x, float y, uint32_t mark = 0) {
  const uint32_t hi = (y == y ? __float_as_uint(y) : 0x7fc00000u) | mark << 31;
  return __hip_atomic_exchange(slot, ((uint64_t)hi << 32) | __float_as_uint(x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct AttnDecodeArgs {
  const _Float16 *qkv;  // [batch][(hq + 2 hkv) HD]
  _Float16 *kc, *vc;    // K [batch][kv head][max_ctx][HD], V [batch][kv head][max_ctx / 8][HD][8]
  const int32_t *pos;   // position of the token
  uint64_t *meet;       // [batch][kv head][head block][node][heads of a block * HD], kEmpty between launches
  _Float16 *qrot;       // rotated query heads for a reader of the activations; null: qkv is rotated and the cache holds the row
  _Float16 *out;        // [batch][hq HD]
  int hq, hkv, max_ctx, splits;
  const float *angles;  // cos, then sin of the HD / 2 pairs at the position (the embedding launch leaves them)
  float scale;
};

template <int HD>
__global__ void __launch_bounds__(AD_THREADS, 2) attn_decode_kernel(AttnDecodeArgs a) {
  constexpr int KK = HD / 32, DT = HD / 16, HALF = HD / 2;
  constexpr int P = 2;        // blocks in flight per wave
  constexpr int OP = HD + 4;          // pitch of the merge buffer
  extern __shared__ __attribute__((aligned(16))) float o_s[];  // [AD_WAVES][heads][OP]
  __shared__ __attribute__((aligned(16))) _Float16 q_s[AD_Q][HD + 8], k_new[HD], v_new[HD];
  __shared__ float m_s[AD_WAVES][AD_Q], l_s[AD_WAVES][AD_Q];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const int group = a.hq / a.hkv, qblocks = (group + AD_Q - 1) / AD_Q;
  const int kvh = (int)blockIdx.x / qblocks, qb = (int)blockIdx.x % qblocks, b = blockIdx.y, split = blockIdx.z;
  const int nq = min(AD_Q, group - qb * AD_Q), head0 = kvh * group + qb * AD_Q;
  const int pos = *a.pos, n_ctx = pos + 1;
  const int per = max(kAttMin, ((n_ctx + a.splits - 1) / a.splits + 31) & ~31), live = (n_ctx + per - 1) / per;
  if (split >= live) return;  // uniform in the workgroup, before any barrier
  const int begin = split * per, blocks = (min(n_ctx, begin + per) - begin + 31) / 32;
  const int mine = (blocks - wave + AD_WAVES - 1) / AD_WAVES;  // blocks wave, wave + 8, ... of the share; 0 or less: none
  const bool owner = split == live - 1;                         // the token's position is in this share

  _Float16 *kbase = a.kc + ((size_t)b * a.hkv + kvh) * a.max_ctx * HD;
  _Float16 *vbase = a.vc + ((size_t)b * a.hkv + kvh) * a.max_ctx * HD;
  struct Block {
    half8_t k[2][KK], v[DT];
  };
  const int k_row = 8 * (r >> 2) + (r & 3);
  auto load = [&](Block &x, int i) {
    const int p0 = begin + 32 * (wave + AD_WAVES * i);
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const _Float16 *src = kbase + (size_t)min(p0 + k_row + 4 * u, pos) * HD + (HD / 4) * c;  // rows past the end repeat the last one
#pragma unroll
      for (int kk = 0; kk < KK; kk++) x.k[u][kk] = *reinterpret_cast<const half8_t *>(src + 8 * kk);
    }
    const _Float16 *src = vbase + ((size_t)min((p0 >> 3) + c, pos >> 3) * HD + r) * 8;
#pragma unroll
    for (int t = 0; t < DT; t++) x.v[t] = __builtin_nontemporal_load(reinterpret_cast<const half8_t *>(src + 128 * t));
  };
  // loads return in order: the row of the token in front of the blocks, whatever a thread will do with it
  const _Float16 *row = a.qkv + (size_t)b * (a.hq + 2 * a.hkv) * HD;
  const int new_t = AD_THREADS - 1 - tid;  // element of the new cache row: the threads that have least to rotate
  _Float16 q0, q1, n0, n1;
  float q_cs = 0.0f, q_sn = 0.0f, n_cs = 0.0f, n_sn = 0.0f;
  {
    const int j = min(tid, nq * HALF - 1), t = min(new_t, HALF + HD - 1);
    const _Float16 *src = row + (size_t)(head0 + j / HALF) * HD + j % HALF;
    q0 = src[0];
    q1 = src[HALF];
    src = row + (size_t)(t < HALF ? a.hq + kvh : a.hq + a.hkv + kvh) * HD + (t < HALF ? t : t - HALF);
    n0 = src[0];
    n1 = src[t < HALF ? HALF : 0];
    if (a.qrot) {
      q_cs = a.angles[j % HALF];
      q_sn = a.angles[HALF + j % HALF];
      n_cs = a.angles[min(t, HALF - 1)];
      n_sn = a.angles[HALF + min(t, HALF - 1)];
    }
  }
  Block ring[P];
  if (mine > 0) {
#pragma unroll
    for (int i = 0; i < P; i++) load(ring[i], min(i, mine - 1));
  }

  // ---- the query heads of this workgroup, rotated, and the new row of the cache
  if (a.qrot) {
    for (int idx = tid; idx < nq * HALF; idx += AD_THREADS) {
      const int h = idx / HALF, i = idx % HALF;
      if (idx != tid) {
        const _Float16 *src = row + (size_t)(head0 + h) * HD;
        q0 = src[i];
        q1 = src[i + HALF];
        q_cs = a.angles[i];
        q_sn = a.angles[HALF + i];
      }
      _Float16 y0, y1;
      rope_pair((float)q0, (float)q1, q_cs, q_sn, y0, y1);
      q_s[h][i] = y0;
      q_s[h][i + HALF] = y1;
      if (split == 0) {
        _Float16 *dst = a.qrot + ((size_t)b * a.hq + head0 + h) * HD;
        dst[i] = y0;
        dst[i + HALF] = y1;
      }
    }
    if (owner) {  // (several head blocks work out the same row; the first one appends it)
      const int t = new_t;
      if (t < HALF) {
        _Float16 y0, y1;
        rope_pair((float)n0, (float)n1, n_cs, n_sn, y0, y1);
        k_new[t] = y0;
        k_new[t + HALF] = y1;
        if (qb == 0) {
          kbase[(size_t)pos * HD + t] = y0;
          kbase[(size_t)pos * HD + t + HALF] = y1;
        }
      } else if (t < HALF + HD) {
        const int d = t - HALF;
        v_new[d] = n0;
        if (qb == 0) vbase[((size_t)(pos >> 3) * HD + d) * 8 + (pos & 7)] = n0;
      }
    }
  } else {
    for (int idx = tid; idx < nq * (HD / 8); idx += AD_THREADS) {
      const int h = idx / (HD / 8), i = idx % (HD / 8) * 8;
      *reinterpret_cast<half8_t *>(&q_s[h][i]) = *reinterpret_cast<const half8_t *>(row + (size_t)(head0 + h) * HD + i);
    }
  }
  lds_barrier();  // (the blocks requested above stay in flight)
  half8_t q[KK];
#pragma unroll
  for (int kk = 0; kk < KK; kk++) {
    const half8_t v = *reinterpret_cast<const half8_t *>(&q_s[min(r, nq - 1)][(HD / 4) * c + 8 * kk]);
    q[kk] = r < nq ? v : half8_t{0, 0, 0, 0, 0, 0, 0, 0};
  }

  float m_run = -INFINITY, l_run = 0.0f;  // of query r; l_run: this lane's positions only
  float4_t o[DT];
#pragma unroll
  for (int t = 0; t < DT; t++) o[t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  auto attend = [&](Block &x, int i) {
    const int p0 = begin + 32 * (wave + AD_WAVES * i);
    const bool tail = p0 + 32 >= n_ctx;  // uniform: the block of the token, or the one that ends with it
    if (tail) {
      const int rel = pos - p0;
      if (a.qrot) {  // the row appended in this launch: the loads saw what the cache held before
#pragma unroll
        for (int u = 0; u < 2; u++)
          if (k_row + 4 * u == rel) {
#pragma unroll
            for (int kk = 0; kk < KK; kk++) x.k[u][kk] = *reinterpret_cast<const half8_t *>(&k_new[(HD / 4) * c + 8 * kk]);
          }
      }
      // positions past the end have weight 0, but 0 * NaN would poison the sum: whatever the slab holds there is blanked
      uint32_t keep[4], put[4];  // of a lane's eight positions, two to a word
#pragma unroll
      for (int w = 0; w < 4; w++) {
        const int left = rel - 8 * c - 2 * w;  // positions of the word in front of the token
        const uint32_t at = left == 0 ? 0xffffu : (left == 1 ? 0xffff0000u : 0u);
        keep[w] = (left >= 2 ? 0xffffffffu : (left == 1 ? 0xffffu : 0u)) | (a.qrot ? 0u : at);
        put[w] = a.qrot ? at : 0u;
      }
#pragma unroll
      for (int t = 0; t < DT; t++) {
        union {
          half8_t h;
          uint32_t w[4];
        } v;
        v.h = x.v[t];
        const uint32_t nv = (uint32_t)*reinterpret_cast<const uint16_t *>(&v_new[16 * t + r]) * 0x10001u;
#pragma unroll
        for (int w = 0; w < 4; w++) v.w[w] = (v.w[w] & keep[w]) | (nv & put[w]);
        x.v[t] = v.h;
      }
    }
    float4_t s[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      s[u] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kk = 0; kk < KK; kk++) s[u] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.k[u][kk], q[kk], s[u], 0, 0, 0);
    }
    // lane (r, c): query r, positions p0 + 8 c + 4 u + e
    float w[8], mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      w[e] = s[e >> 2][e & 3] * a.scale;
      if (tail && p0 + 8 * c + e > pos) w[e] = -INFINITY;
      mx = fmaxf(mx, w[e]);
    }
    mx = max_xor16_xor32(mx);
    if (__any(mx > m_run)) {  // (a factor of exactly one otherwise)
      const float m_new = fmaxf(m_run, mx);
      const float f = m_run == -INFINITY ? 0.0f : __expf(m_run - m_new);
      l_run *= f;
#pragma unroll
      for (int t = 0; t < DT; t++) o[t] = o[t] * f;
      m_run = m_new;
    }
    half8_t pw;
#pragma unroll
    for (int e = 0; e < 8; e++) {
      const float v = w[e] == -INFINITY ? 0.0f : __expf(w[e] - m_run);
      l_run += v;
      pw[e] = (_Float16)v;
    }
#pragma unroll
    for (int t = 0; t < DT; t++) o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x.v[t], pw, o[t], 0, 0, 0);
  };
  if (mine > 0) {
    int i = 0;
    for (; i + P < mine; i += P) {
#pragma unroll
      for (int u = 0; u < P; u++) {
        attend(ring[u], i + u);
        load(ring[u], min(i + u + P, mine - 1));
      }
    }
#pragma unroll
    for (int u = 0; u < P; u++)
      if (i + u < mine) attend(ring[u], i + u);
  }

  // ---- the eight waves: lane (r, c) holds O^T[16 t + 4 c + e][query r]
  l_run = sum_xor16_xor32(l_run);
  if (c == 0) {
    m_s[wave][r] = m_run;
    l_s[wave][r] = l_run;
  }
  const int pair = ((int)b * a.hkv + kvh) * qblocks + qb;
  uint64_t *nodes = a.meet + (size_t)pair * (size_t)a.splits * min(AD_Q, group) * HD;  // (the last block of heads may be smaller)
  const size_t node = (size_t)nq * HD;
  const int second_word = nq * HALF;  // a node's first words, then its second ones: lanes side by side (in turn: 0.4 us a launch more)
  const bool meets = live > 1 && (split ^ 1) < live;  // at the first level (the last share of an odd number goes on by itself)
  // a thread's two channels of a head: the share's maximum and sum
  float m, l, f[AD_WAVES];
  auto sums = [&](int h) {
    m = -INFINITY;
    l = 0.0f;
#pragma unroll
    for (int w = 0; w < AD_WAVES; w++) m = fmaxf(m, m_s[w][h]);
#pragma unroll
    for (int w = 0; w < AD_WAVES; w++) {
      f[w] = m_s[w][h] == -INFINITY ? 0.0f : __expf(m_s[w][h] - m);
      l += l_s[w][h] * f[w];
    }
  };
  if (r < nq) {
#pragma unroll
    for (int t = 0; t < DT; t++) *reinterpret_cast<float4_t *>(&o_s[(wave * nq + r) * OP + 16 * t + 4 * c]) = o[t];
  }
  lds_barrier();
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): no block's load is pending, so that the compiler need not wait for the exchange with them
  uint64_t ml = kEmpty;
  if (tid < nq * HALF) {
    sums(tid / HALF);
    // (on its way while the waves' outputs are added up; sent a barrier earlier, in front of their way through LDS, it gains nothing:
    // eight steps of 16 sequences at 2048 positions 20 818 and 20 809 us, this way 20 793 and 20 857)
    if (meets) ml = swap_pair(nodes + tid + (size_t)(split >> 1) * node, m, l, split & 1);
  }
  auto meet = [&](int idx) __attribute__((always_inline)) {
    const int h = idx / HALF, d = idx % HALF * 2;
    uint64_t *level = nodes + idx;
    float2_t o = {0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < AD_WAVES; w++) o += *reinterpret_cast<const float2_t *>(&o_s[(w * nq + h) * OP + d]) * f[w];
    bool top = true;
    if (live > 1) {
      int met = 0;  // bit i: merged at level i
      for (int at = split, count = live, width = a.splits, bit = 1; count > 1; at >>= 1, count = (count + 1) >> 1, width >>= 1, bit <<= 1) {
        uint64_t *slot = level + (size_t)(at >> 1) * node;
        level += (size_t)(width >> 1) * node;
        if ((at ^ 1) >= count) continue;
        if (bit > 1) ml = swap_pair(slot, m, l, at & 1);
        const uint64_t ov = swap_pair(slot + second_word, o[0], o[1]);
        if (ov == kEmpty) {
          top = false;
          break;
        }
        met |= bit;
        // the first word empty and the second one full: the partner's first word, sent before its second, takes the place of this share's
        while (ml == kEmpty || (uint32_t)(ml >> 63) == (uint32_t)(at & 1)) ml = __hip_atomic_load(slot, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const float2_t om = word_pair(ov), other = word_pair(ml & ~((uint64_t)1 << 63));
        const float mo = other[0], lo = other[1], mx = fmaxf(m, mo);
        const float own = m == mx ? 1.0f : __expf(m - mx), theirs = mo == mx ? 1.0f : __expf(mo - mx);
        const bool second = (at & 1) != 0;  // always added in the order of the positions
        const float f0 = second ? theirs : own, f1 = second ? own : theirs;
        const float2_t o0 = second ? om : o, o1 = second ? o : om;
        l = (second ? lo : l) * f0 + (second ? l : lo) * f1;
        o = o0 * f0 + o1 * f1;
        m = mx;
      }
      // the slots are emptied at the end: a store in front of the next exchange would be waited for with it
      level = nodes + idx;
      for (int at = split, width = a.splits; met != 0; at >>= 1, width >>= 1, met >>= 1) {
        uint64_t *slot = level + (size_t)(at >> 1) * node;
        if (met & 1) {
          __hip_atomic_store(slot, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(slot + second_word, kEmpty, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        level += (size_t)(width >> 1) * node;
      }
    }
    if (top) {
      const float2_t v = l > 0.0f ? float2_t{o[0] / l, o[1] / l} : o * 0.0f;  // (a NaN stays one)
      *reinterpret_cast<half2_t *>(a.out + ((size_t)b * a.hq + head0 + h) * HD + d) = half2_t{(_Float16)v[0], (_Float16)v[1]};
    }
  };
  // (not as the first turn of the loop: its registers might be those of an exchange of the turn before, and it would start with a wait)
  if (tid < nq * HALF) meet(tid);
  for (int idx = tid + AD_THREADS; idx < nq * HALF; idx += AD_THREADS) {
    sums(idx / HALF);
    if (meets) ml = swap_pair(nodes + idx + (size_t)(split >> 1) * node, m, l, split & 1);
    meet(idx);
  }
}

int head_blocks(int hq, int hkv) { return (hq / hkv + AD_Q - 1) / AD_Q; }

// shares of a kv head's positions: a power of two (no level of the merge for a single share), no more than the CUs hold at once or
// the longest context can use
int shares(int batch, int hq, int hkv, int max_ctx, int num_cus) {
  const int pairs = batch * hkv * head_blocks(hq, hkv), most = (max_ctx + kAttMin - 1) / kAttMin;
  const int n = (num_cus > 0 ? num_cus : 256) / pairs;
  int k = 1;
  while (2 * k <= n && 2 * k <= most) k *= 2;
  return k;
}

template <int HD>
int32_t go(const AttnDecodeArgs &a, int batch, hipStream_t s) {
  const int group = a.hq / a.hkv, nq = group < AD_Q ? group : AD_Q;
  constexpr int kMostLds = AD_WAVES * AD_Q * (HD + 4) * 4;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_decode_kernel<HD>), hipFuncAttributeMaxDynamicSharedMemorySize, kMostLds);
  });
  if (attr_err != hipSuccess) return set_error(YSCV_HIP_ERR_DEVICE, "cannot reserve LDS for the attention merge: %s", hipGetErrorString(attr_err));
  hipLaunchKernelGGL((attn_decode_kernel<HD>), dim3((unsigned)(a.hkv * head_blocks(a.hq, a.hkv)), (unsigned)batch, (unsigned)a.splits),
                     dim3(AD_THREADS), (size_t)AD_WAVES * nq * (HD + 4) * 4, s, a);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

}  // namespace

size_t attention_decode_meet_bytes(int max_batch, int hq, int hkv, int hd, int max_ctx, int num_cus) {
  size_t most = 0;
  const size_t group = (size_t)(hq / hkv), nq = group < AD_Q ? group : AD_Q;
  for (int b = 1; b <= max_batch; b++) {
    const size_t n = (size_t)b * hkv * head_blocks(hq, hkv) * shares(b, hq, hkv, max_ctx, num_cus) * nq * hd;
    if (n > most) most = n;
  }
  return most * sizeof(uint64_t);
}

int32_t launch_attention_decode(const _Float16 *qkv, _Float16 *kc, _Float16 *vc, const int32_t *pos, int batch, int hq, int hkv, int hd,
                                const float *angles, int max_ctx, int num_cus, uint64_t *meet, _Float16 *qrot, _Float16 *out, hipStream_t s) {
  AttnDecodeArgs a;
  a.qkv = qkv;
  a.kc = kc;
  a.vc = vc;
  a.pos = pos;
  a.meet = meet;
  a.qrot = qrot;
  a.out = out;
  a.hq = hq;
  a.hkv = hkv;
  a.max_ctx = max_ctx;
  a.splits = shares(batch, hq, hkv, max_ctx, num_cus);
  a.scale = 1.0f / sqrtf((float)hd);
  a.angles = angles;
  switch (hd) {
    case 32: return go<32>(a, batch, s);
    case 64: return go<64>(a, batch, s);
    case 96: return go<96>(a, batch, s);
    case 128: return go<128>(a, batch, s);
    default: return set_error(YSCV_HIP_ERR_UNSUPPORTED, "attention: head width %d (supported: 32, 64, 96, 128)", hd);
  }
}

}  // namespace yscv
