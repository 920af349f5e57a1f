// One token through all layers of a decoder with head width 128 and one CU per 16 rows of its residual stream (batch 1), in
// one launch: the step of the loop of apps/llm-bench/src/main.rs:525-548 between the embedding lookup and the final norm.
//
// A layer of the 7B shape (d_model 4096, 32 heads over 8, d_ff 14336) is 123 MB of weights, 18 us at the rate a read stream
// sustains.  A step, position 2000: 1033 us; as kernels of a graph, each with its launch and a ramp that moves little, 1376
// (1619 before int4_gemv.hip); decode_persistent.hip, whose six hand-overs of a layer take 4.5 us each, 1454.  16 layers of d_model
// 2560, d_ff 8960: 409 against 663; 3072, 8192: 431 against 558 and 638.  There is no supported shape or context (64 .. 16000) at
// which another path is the faster one.
//   * G = d_model / 16 workgroups of eight waves, one per CU.  Workgroup w owns the 16-row blocks w (and w + G) of q/k/v, w of o
//     and down, and a run of gate/up blocks; its waves split K in slices of 512, the unit of int4_gemv.hip: sixteen 32-k blocks
//     that stand in the sixteen rows of the MFMA's activation operand, so that one operand of four registers serves a slice
//     whatever the number of row blocks.
//   * Weights go from memory to registers, three to six slices (18 registers each) ahead in the order they are used, across the
//     hand-overs: while a stage's input is on the way the next slices stream in.  A poll's answer comes behind the loads
//     requested before it, whichever wave asked, so where each slice is requested is a balance: about 70 KB of a CU pass while a
//     hand-over takes its 2 us anyway.  (Four slices ahead throughout: 1215 us a step; the next stage's first slices requested
//     inside gate/up's first blocks: 1066, behind its fourth and fifth: 1033.)
//   * The first slice of a stage is decoded while the stage's input is on the way.
//   * A stage's input arrives as tagged entries (decode_exchange.hpp); a wave polls what its own slices need, in operand order
//     where an entry holds two fp16 values.  The sum of squares of a norm is formed by the consumers.
//   * Attention: the positions are cut into at most G / kv_heads equal pieces per kv head, multiples of 32; a wave takes 32 at a
//     time, its keys and values requested two stages ahead.  One wave per workgroup merges the pieces of sixteen channels.
// An entry buffer is written again one layer later, and between the two lies a stage whose input comes from every workgroup
// behind its last read, as in decode_layers.hip.  Every wait is bounded; one that gives up sets *give_up, all others then
// return at once and the host reports it.  The host lets one such launch run at a time (Resident in decoder.hip).
//
// A layer at position 2000 takes 31 us: six hand-overs of 2 .. 4 from the last wave's sums to the first product, gate/up 7 of
// arithmetic and stream, down 2.5, q/k/v 1, attention 1, o 0.4, and 0.3 .. 2 until the slowest wave of a stage arrives.
//
// Arithmetic: exact (q - 8) in fp16 against fp16 activations, f32 accumulation, group scale in f32 per 32 k.  Behind a norm the
// activation is fp16(h * gamma) with the largest of a wave's 512 values brought to 2^14 .. 2^15; the powers of two and the
// norm's factor follow the f32 sums: the same product as RMSNorm in front, with the rounding before the row factor.
#include <hip/hip_runtime.h>

#include "decode_exchange.hpp"

namespace yscv {

namespace {

constexpr int WAVES = 8;
constexpr int HD = 128;
constexpr int MAX_GU = 7;           // blocks of gate/up rows of a workgroup
constexpr int MAX_DOWN = 4;         // slices of the FFN's width of a wave
constexpr int MAX_PIECES = 32;      // pieces of a kv head's positions
constexpr int HEAD_REC = 144;       // entries of one head's partials of a piece: o[128], max, sum; whole lines
constexpr int MERGER = WAVES - 1;

struct Quad {  // 16 rows x 512 k: lane (r, c) holds four words of each of four 128-k tiles, and the scales of row r in tile c
  uint4_t w[4];
  half4_t s;
};
struct Decoded {
  half8_t w[4][4];
};

}  // namespace

__global__ void __launch_bounds__(64 * WAVES, 2) decode_wide_kernel(LayersModel m) {
  __shared__ __attribute__((aligned(16))) _Float16 xs[WAVES][512];            // a wave's activations behind a norm
  __shared__ __attribute__((aligned(16))) float part[2][MAX_GU * 16][WAVES];  // per row the sums of the waves
  __shared__ __attribute__((aligned(16))) float wave_ss[2][WAVES];
  __shared__ __attribute__((aligned(16))) float rot[2][HD / 2];               // cos, sin of pair (i, i + 64) at this position
  __shared__ __attribute__((aligned(16))) _Float16 q_lds[WAVES][4][HD], p_lds[WAVES][4][32], knew[HD], vnew[HD];
  __shared__ float w_m[WAVES][4], w_l[WAVES][4];
  __shared__ float w_o[WAVES][4][HD];
  int tid = threadIdx.x, lane = tid & 63;
  int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int r = lane & 15, c = lane >> 4;
  const int wg = blockIdx.x, G = m.G, L = m.n_layers, D = m.d;
  const int HQ = m.heads, HKV = m.kv_heads, GROUP = HQ / HKV;
  const int nt_q = (HQ + 2 * HKV) * HD / 16, nt_g = 2 * m.ff / 16;
  const int ks_d = D / 512, ks_o = HQ * HD / 512, ks_f = (m.ff + 511) / 512;  // slices of K
  const int gu_base = nt_g / G, gu_rem = nt_g % G;
  const int gu_first = wg * gu_base + min(wg, gu_rem), gu_n = gu_base + (wg < gu_rem ? 1 : 0);
  const int pos_now = *m.pos;
  // piece ch of kv head kvh belongs to workgroup ch * HKV + kvh
  const int pieces_max = min(G / HKV, MAX_PIECES);
  const int piece = ((pos_now + pieces_max) / pieces_max + 31) & ~31, pieces = pos_now / piece + 1;
  const int kvh = wg % HKV, ch = wg / HKV;
  const bool attends = ch < pieces;  // uniform in the workgroup
  const uint32_t tag0 = *m.steps * (uint32_t)(L + 1) + 1u;
  Patience pt{POLL_LIMIT, m.give_up};
  NibbleConsts nc;
  nc.init();
  uint32_t magic_hi = 0x54005400u;
  asm volatile("" : "+v"(magic_hi));

  // blocks and slices past the end are loaded again from the last one and not used
  auto load_quad = [&](const LayerAt &ly, int kind, int nt, int nts, int sl, int sls) {
    nt = nt < nts ? nt : nts - 1;
    sl = sl < sls ? sl : sls - 1;
    const size_t t = (size_t)nt * m.ktp[kind] + 4 * sl;
    Quad o;
    const uint8_t *p = ly.tiles[kind] + t * 1024 + lane * 16;
#pragma unroll
    for (int i = 0; i < 4; i++) o.w[i] = *reinterpret_cast<const uint4_t *>(p + i * 1024);
    o.s = *reinterpret_cast<const half4_t *>(ly.scales[kind] + ((t + c) * 16 + r) * 4);
    return o;
  };
  auto load_q = [&](const LayerAt &ly, int b) { return load_quad(ly, 0, wg + G * b, nt_q, wave, ks_d); };
  auto load_o = [&](const LayerAt &ly) { return load_quad(ly, 1, wg, G, wave, ks_o); };
  auto load_g = [&](const LayerAt &ly, int b) { return load_quad(ly, 2, gu_first + min(b, gu_n - 1), nt_g, wave, ks_d); };
  auto load_d = [&](const LayerAt &ly, int i) { return load_quad(ly, 3, wg, G, wave + WAVES * i, ks_f); };
  float2 gam[4];  // norm weights of this wave's slice
  auto load_gamma = [&](const LayerAt &ly, int which) {
    const float *g = ly.gamma[which] + (wave < ks_d ? wave : 0) * 512 + 2 * lane;
#pragma unroll
    for (int i = 0; i < 4; i++) gam[i] = *reinterpret_cast<const float2 *>(g + 128 * i);
  };

  // keys of positions p0 + 16 pb + r, channels 32 c + 8 j; values of positions p0 + 8 c .. + 7, channel 16 t + r
  half8_t kf[2][4], vf[8];
  auto load_kv = [&](const LayerAt &ly, int p0) {
#pragma unroll
    for (int pb = 0; pb < 2; pb++) {
      const int at = min(p0 + 16 * pb + r, m.max_ctx - 1);
      const _Float16 *k = ly.kc + ((size_t)kvh * m.max_ctx + at) * HD + 32 * c;
#pragma unroll
      for (int j = 0; j < 4; j++) kf[pb][j] = *reinterpret_cast<const half8_t *>(k + 8 * j);
    }
    const int slab = min(p0 / 8 + c, m.max_ctx / 8 - 1);
    const _Float16 *v = ly.vc + (((size_t)kvh * (m.max_ctx / 8) + slab) * HD + r) * 8;
#pragma unroll
    for (int t = 0; t < 8; t++) vf[t] = *reinterpret_cast<const half8_t *>(v + 128 * t);
  };

  // the first slice of a stage is decoded while the stage's input is on the way
  auto decode = [&](const Quad &v) {
    Decoded o;
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        o.w[t][q] = decode_q8(v.w[t][q], nc, magic_hi);
        asm volatile("" : "+v"(o.w[t][q]));  // here, not behind the wait
      }
    return o;
  };
  // a lane's part (tile c) of the sums of 16 rows over the 512 k
  auto mul_with = [&](auto weights, const half4_t &sc, half8_t x) {
    const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
    float sel[4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const float4_t dd = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, weights(t, q), zero, 0, 0, 0);
        sel[q] = t == 0 ? dd[q] : (c == t ? dd[q] : sel[q]);
      }
    float acc = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; q++) acc = fmaf((float)sc[q], sel[q], acc);
    return acc;
  };
  auto mul = [&](const Quad &v, half8_t x) { return mul_with([&](int t, int q) { return decode_q8(v.w[t][q], nc, magic_hi); }, v.s, x); };
  auto mul_decoded = [&](const Decoded &d, const Quad &v, half8_t x) { return mul_with([&](int t, int q) { return d.w[t][q]; }, v.s, x); };
  int pb_now = 0;  // which of the two sets of partial sums this stage uses
  auto put_part = [&](int b, float v) {
    v = sum_xor16_xor32(v);
    if (lane < 16) part[pb_now][16 * b + lane][wave] = v;
  };
  auto sum8 = [](const float *p) {
    const float4_t a = *reinterpret_cast<const float4_t *>(p), b = *reinterpret_cast<const float4_t *>(p + 4);
    return ((a[0] + a[1]) + (a[2] + a[3])) + ((b[0] + b[1]) + (b[2] + b[3]));
  };
  auto row_sum = [&]() { return sum8(part[pb_now][tid]); };  // thread t: row t & 15 of block t >> 4
  auto row_rstd = [&]() { return __builtin_amdgcn_rsqf(sum8(wave_ss[pb_now]) / (float)D + m.eps); };

  // Input of a projection behind a norm: fp16(h * gamma * 2^e) of this wave's slice, 2^e from the largest of the 512 values,
  // 2^-e for the wave's sums.  The other factor of the norm, common to all waves, follows the sums too.
  float down = 0.0f;
  auto take_normed = [&](const u64 *buf, uint32_t tag) {
    half8_t x = {0, 0, 0, 0, 0, 0, 0, 0};
    down = 0.0f;
    if (wave >= ks_d) {
      if (lane == 0) wave_ss[pb_now][wave] = 0.0f;
      return x;
    }
    uint4_t v[4];
    while (true) {
      bool ok = true;
#pragma unroll
      for (int i = 0; i < 4; i++) v[i] = get2(buf + wave * 512 + 128 * i + 2 * lane);
      landed(v);
#pragma unroll
      for (int i = 0; i < 4; i++) ok = ok && both(v[i], tag);
      if (__all(ok)) break;
      if (!pt.again()) break;
    }
    float y[8], mx = 0.0f, ss = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const float h0 = as_f(v[i][0]), h1 = as_f(v[i][2]);
      y[2 * i] = h0 * gam[i].x;
      y[2 * i + 1] = h1 * gam[i].y;
      mx = fmaxf(mx, fmaxf(fabsf(y[2 * i]), fabsf(y[2 * i + 1])));
      ss += h0 * h0 + h1 * h1;
    }
    const uint32_t top = (__float_as_uint(wave_max(mx)) >> 23) & 255u;
    const uint32_t f = min(268u - top, 253u);  // the largest value becomes 2^14 .. 2^15
    const float up = as_f(f << 23);
    down = as_f((254u - f) << 23);
#pragma unroll
    for (int i = 0; i < 4; i++)
      *reinterpret_cast<uint32_t *>(&xs[wave][128 * i + 2 * lane]) = pack2(narrow(y[2 * i] * up), narrow(y[2 * i + 1] * up));
    ss = wave_sum(ss);
    if (lane == 0) wave_ss[pb_now][wave] = ss;
    wave_lds_sync();
    x = *reinterpret_cast<const half8_t *>(&xs[wave][32 * r + 8 * c]);
    return x;
  };
  // eight fp16 values from two loads of two entries
  auto eight = [&](const uint4_t &a, const uint4_t &b) {
    union {
      uint4_t u;
      half8_t h;
    } v;
    v.u = uint4_t{a[0], a[2], b[0], b[2]};
    return v.h;
  };

  // residual stream: thread t < 16 owns row 16 wg + t
  const int own_row = 16 * wg + (tid & 15);
  float h = 0.0f;
  auto publish_h = [&](u64 *buf, uint32_t tag) {
    if (tid < 16) put_entry(buf + own_row, __float_as_uint(h), tag);
  };

  int token = m.tokens[0];
  token = token < 0 ? 0 : (token >= m.vocab ? m.vocab - 1 : token);
  h = (float)m.emb[(size_t)token * D + own_row];
  publish_h(m.x + m.at_attn, tag0);
  const bool two_q = wg + G < nt_q;  // uniform in the workgroup
  const int p_first = ch * piece + 32 * wave;
  const bool kv_used = attends && 32 * wave < piece && p_first <= pos_now;  // uniform in the wave
  Quad q0, q1;
  load_gamma(m.layers[0], 0);
  q0 = load_q(m.layers[0], 0);
  q1 = load_q(m.layers[0], 1);
  if (kv_used) load_kv(m.layers[0], p_first);
  if (tid < HD / 2) {
    const float inv_freq = 1.0f / powf(m.theta, (float)(2 * tid) / (float)HD);
    sincosf(inv_freq * (float)pos_now, &rot[1][tid], &rot[0][tid]);
  }
  lds_barrier();
  // where this lane's eight values of slice wave + 8 i of the SwiGLU output begin
  int act_at[MAX_DOWN];
#pragma unroll
  for (int i = 0; i < MAX_DOWN; i++) {
    const int b = 64 * (wave + WAVES * i) + 4 * r + c;
    act_at[i] = b < nt_g ? m.at_act + act_entry(b, gu_base, gu_rem) : -1;
  }

#pragma unroll 1
  for (int l = 0; l < L; l++) {
    const uint32_t tag = tag0 + (uint32_t)l;
    const bool last = l + 1 == L;
    const LayerAt &ly = m.layers[l], &nx = m.layers[last ? l : l + 1];
    asm volatile("" : "+v"(tid), "+s"(wave));  // opaque in every layer: nothing made from them is kept over the loop
    lane = tid & 63;
    r = lane & 15;
    c = lane >> 4;
    Quad o, g0, g1, g2, g3, g4, g5, g6, d0, d1, d2, d3;
    // ---- q / k / v ---------------------------------------------------------------------------------------------------
    {
      const Decoded w = decode(q0);
      const half8_t x = take_normed(m.x + m.at_attn, tag);
      put_part(0, mul_decoded(w, q0, x) * down);
      if (two_q) put_part(1, mul(q1, x) * down);
    }
    lds_barrier();
    if (tid < 32) {
      const int nt = wg + G * (tid >> 4), row = 16 * nt + (tid & 15);
      if (nt < nt_q) {
        _Float16 v = narrow(row_sum() * row_rstd());
        const _Float16 *bias = ly.qkv_bias;
        if (bias) v = (_Float16)((float)v + (float)bias[row]);
        const float nxt = dpp_move<DPP_NEXT1>((float)v);
        if (!(tid & 1)) put_entry(m.x + m.at_qkv + qkv_entry(row), pack2(v, (_Float16)nxt), tag);
      }
    }
    pb_now ^= 1;
    o = load_o(ly);
    g0 = load_g(ly, 0);
    // ---- attention ---------------------------------------------------------------------------------------------------
    if (attends) {
      float m_h = -INFINITY, l_h = 0.0f, o_acc[8];  // head c, channels 16 t + r
#pragma unroll
      for (int t = 0; t < 8; t++) o_acc[t] = 0.0f;
      int pos = pos_now;
      asm volatile("" : "+s"(pos));
      if (kv_used) {  // uniform in the wave
        const int rel = pos - ch * piece;  // the token's position counted from the piece's first
        const bool own = rel < piece && (rel >> 5) % WAVES == wave;  // this wave has it: its k and v come with q
        {
          const int hh = min(lane >> 4, GROUP - 1), i4 = 4 * (lane & 15);
          const u64 *qe = m.x + m.at_qkv + qkv_entry((kvh * GROUP + hh) * HD + i4);
          const u64 *ke = m.x + m.at_qkv + qkv_entry((HQ + kvh) * HD + i4);
          const u64 *ve = m.x + m.at_qkv + qkv_entry((HQ + HKV + kvh) * HD + 4 * (lane & 31));
          uint4_t v[8];  // q and its other half, k and its other half, v
#pragma unroll
          for (int i = 2; i < 8; i++) v[i] = uint4_t{0u, tag, 0u, tag};
          while (true) {
            v[0] = get2(qe);
            v[1] = get2(qe + 64);  // 64 channels further: four blocks
            if (own) {
              v[2] = get2(ke);
              v[3] = get2(ke + 64);
              v[4] = get2(ve);
            }
            landed(v);
            bool ok = true;
#pragma unroll
            for (int i = 0; i < 5; i++) ok = ok && both(v[i], tag);
            if (__all(ok)) break;
            if (!pt.again()) break;
          }
          const float4_t cs = *reinterpret_cast<const float4_t *>(&rot[0][i4]), sn = *reinterpret_cast<const float4_t *>(&rot[1][i4]);
          auto rotate = [&](const uint4_t &lo, const uint4_t &hi, _Float16 *dst) {
            half4_t y0, y1;
#pragma unroll
            for (int u = 0; u < 4; u++) {
              U32H2 a, b;
              a.u = lo[2 * (u >> 1)];
              b.u = hi[2 * (u >> 1)];
              const float x0 = (float)a.h[u & 1], x1 = (float)b.h[u & 1];
              y0[u] = narrow(fmaf(x0, cs[u], -(x1 * sn[u])));
              y1[u] = narrow(fmaf(x0, sn[u], x1 * cs[u]));
            }
            *reinterpret_cast<half4_t *>(dst + i4) = y0;
            *reinterpret_cast<half4_t *>(dst + 64 + i4) = y1;
          };
          if ((lane >> 4) < GROUP) rotate(v[0], v[1], q_lds[wave][lane >> 4]);
          if (own) {
            if (lane < 16) rotate(v[2], v[3], knew);
            if (lane < 32) {
              typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
              *reinterpret_cast<u32x2 *>(&vnew[4 * lane]) = u32x2{v[4][0], v[4][2]};
            }
          }
          wave_lds_sync();
        }
        half8_t qa[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const half8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
          qa[j] = ((r & 3) == 0 && (r >> 2) < GROUP) ? *reinterpret_cast<const half8_t *>(&q_lds[wave][r >> 2][32 * c + 8 * j]) : z;
        }
#pragma unroll 1
        for (int p0 = p_first; p0 < ch * piece + piece && p0 <= pos; p0 += 32 * WAVES) {
          if (p0 != p_first) load_kv(ly, p0);
          const int at = pos - p0;
          if (own && at >= 0 && at < 32) {
#pragma unroll
            for (int pb = 0; pb < 2; pb++)
              if (at == pb * 16 + r) {
#pragma unroll
                for (int j = 0; j < 4; j++) kf[pb][j] = *reinterpret_cast<const half8_t *>(&knew[32 * c + 8 * j]);
              }
#pragma unroll
            for (int t = 0; t < 8; t++) {
              const _Float16 nv = vnew[t * 16 + r];
#pragma unroll
              for (int e = 0; e < 8; e++) vf[t][e] = 8 * c + e < at ? vf[t][e] : (8 * c + e == at ? nv : (_Float16)0.0f);
            }
          }
          float s[2];
#pragma unroll
          for (int pb = 0; pb < 2; pb++) {
            float4_t dd = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int j = 0; j < 4; j++) dd = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[j], kf[pb][j], dd, 0, 0, 0);
            s[pb] = p0 + pb * 16 + r <= pos ? dd[0] * 0.08838834764831845f : -INFINITY;
          }
          const float mx = fmaxf(m_h, row_max16(fmaxf(s[0], s[1])));
          const float e0 = s[0] == -INFINITY ? 0.0f : __expf(s[0] - mx), e1 = s[1] == -INFINITY ? 0.0f : __expf(s[1] - mx);
          const float old = m_h == -INFINITY ? 0.0f : __expf(m_h - mx);
          l_h = l_h * old + row_sum16(e0 + e1);
          m_h = mx;
          p_lds[wave][c][r] = (_Float16)e0;
          p_lds[wave][c][16 + r] = (_Float16)e1;
          wave_lds_sync();
          half8_t pa = {0, 0, 0, 0, 0, 0, 0, 0};
          if ((r & 3) == 0 && (r >> 2) < GROUP) pa = *reinterpret_cast<const half8_t *>(&p_lds[wave][r >> 2][8 * c]);
#pragma unroll
          for (int t = 0; t < 8; t++) {
            float4_t dd = {0.0f, 0.0f, 0.0f, 0.0f};
            dd = __builtin_amdgcn_mfma_f32_16x16x32_f16(pa, vf[t], dd, 0, 0, 0);
            o_acc[t] = o_acc[t] * old + dd[0];
          }
          wave_lds_sync();
        }
        if (own) {  // the token's row of the cache
          if (lane < 32) *reinterpret_cast<half4_t *>(ly.kc + ((size_t)kvh * m.max_ctx + pos) * HD + 4 * lane) = *reinterpret_cast<const half4_t *>(&knew[4 * lane]);
#pragma unroll
          for (int u = 0; u < 2; u++)
            ly.vc[(((size_t)kvh * (m.max_ctx / 8) + pos / 8) * HD + 64 * u + lane) * 8 + (pos & 7)] = vnew[64 * u + lane];
        }
      }
      if (r == 0) {
        w_m[wave][c] = m_h;
        w_l[wave][c] = l_h;
      }
#pragma unroll
      for (int t = 0; t < 8; t++) w_o[wave][c][16 * t + r] = o_acc[t];
      lds_barrier();
      if (tid < GROUP * HD) {
        const int hh = tid >> 7, d = tid & 127;
        float mw[WAVES], M = -INFINITY, ls = 0.0f, os = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
          mw[w] = w_m[w][hh];
          M = fmaxf(M, mw[w]);
        }
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
          const float f = mw[w] == -INFINITY ? 0.0f : __expf(mw[w] - M);
          ls += w_l[w][hh] * f;
          os += w_o[w][hh][d] * f;
        }
        u64 *rec = m.x + m.at_part + ((size_t)(kvh * GROUP + hh) * MAX_PIECES + ch) * HEAD_REC;
        put_entry(rec + d, __float_as_uint(os), tag);
        if (d < 2) put_entry(rec + HD + d, __float_as_uint(d ? ls : M), tag);
      }
    }
    g1 = load_g(ly, 1);
    // ---- merge of sixteen channels: lane (g, p) takes channels 2 p, 2 p + 1 of every eighth piece ------------------------
    if (wave == MERGER && wg < HQ * HD / 16) {
      const int head = wg >> 3, p = lane & 7, g = lane >> 3;
      const u64 *rec = m.x + m.at_part + (size_t)head * MAX_PIECES * HEAD_REC;
      uint4_t v[8];
      while (true) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < 4; i++) {  // pieces past the end repeat the last one
          const u64 *q = rec + min(g + 8 * i, pieces - 1) * HEAD_REC;
          v[2 * i] = get2(q + HD);
          v[2 * i + 1] = get2(q + 16 * (wg & 7) + 2 * p);
        }
        landed(v);
#pragma unroll
        for (int i = 0; i < 8; i++) ok = ok && both(v[i], tag);
        if (__all(ok)) break;
        if (!pt.again()) break;
      }
      float M = -INFINITY, ls = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (g + 8 * i < pieces) M = fmaxf(M, as_f(v[2 * i][0]));
      M = fmaxf(M, dpp_move<DPP_ROR8>(M));
      M = max_xor16_xor32(M);
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (g + 8 * i < pieces) {
          const float mc = as_f(v[2 * i][0]), f = mc == -INFINITY ? 0.0f : __expf(mc - M);
          ls += as_f(v[2 * i][2]) * f;
          o0 += as_f(v[2 * i + 1][0]) * f;
          o1 += as_f(v[2 * i + 1][2]) * f;
        }
      auto over_g = [](float t) {
        t += dpp_move<DPP_ROR8>(t);
        return sum_xor16_xor32(t);
      };
      ls = over_g(ls);
      o0 = over_g(o0);
      o1 = over_g(o1);
      const float inv = ls > 0.0f ? 1.0f / ls : 0.0f;
      if (lane < 8) put_entry(m.x + m.at_ao + 16 * wg + lane, pack2(narrow(o0 * inv), narrow(o1 * inv)), tag);
    }
    // ---- output projection ---------------------------------------------------------------------------------------------
    {
      const Decoded w = decode(o);
      g2 = load_g(ly, 2);
      load_gamma(ly, 1);
      half8_t x = {0, 0, 0, 0, 0, 0, 0, 0};
      if (wave < ks_o) {
        const u64 *e = m.x + m.at_ao + (32 * wave + 2 * r + (c >> 1)) * 16 + 4 * (c & 1);
        uint4_t v[2];
        while (true) {
          v[0] = get2(e);
          v[1] = get2(e + 2);
          landed(v);
          if (__all(both(v[0], tag) && both(v[1], tag))) break;
          if (!pt.again()) break;
        }
        x = eight(v[0], v[1]);
      }
      put_part(0, mul_decoded(w, o, x));
      g3 = load_g(ly, 3);
    }
    lds_barrier();
    if (tid < 16) h += row_sum();
    publish_h(m.x + m.at_ffn, tag);
    pb_now ^= 1;
    // ---- gate / up + SwiGLU: -------------------------------------------------------------------------------
    {
      const Decoded w = decode(g0);
      g4 = load_g(ly, 4);
      const half8_t x = take_normed(m.x + m.at_ffn, tag);
      put_part(0, mul_decoded(w, g0, x) * down);
      g5 = load_g(ly, 5);
      auto block = [&](int b, const Quad &q) {
        if (b < gu_n) put_part(b, mul(q, x) * down);
      };
      block(1, g1);
      g6 = load_g(ly, 6);
      block(2, g2);
      block(3, g3);
      block(4, g4);
      d0 = load_d(ly, 0);
      block(5, g5);
      d1 = load_d(ly, 1);
      block(6, g6);
    }
    lds_barrier();
    if (tid < 16 * gu_n) {
      const float v = row_sum() * row_rstd();
      const _Float16 a = narrow(silu(v) * dpp_move<DPP_NEXT1>(v));  // even rows are gates, odd ones ups
      const float a2 = dpp_move<DPP_NEXT2>((float)a);
      if (!(tid & 3)) put_entry(m.x + m.at_act + wg * kLayersActSlots + (tid >> 2), pack2(a, (_Float16)a2), tag);
    }
    pb_now ^= 1;
    d2 = load_d(ly, 2);
    d3 = load_d(ly, 3);
    // ---- down --------------------------------------------------------------------------------------------------
    {
      const Decoded w = decode(d0);
      half8_t x[MAX_DOWN];
      uint4_t v[8];
      while (true) {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < MAX_DOWN; i++) {
          const u64 *e = m.x + (act_at[i] >= 0 ? act_at[i] : m.at_act);
          v[2 * i] = get2(e);
          v[2 * i + 1] = get2(e + 2);
        }
        landed(v);
#pragma unroll
        for (int i = 0; i < MAX_DOWN; i++) ok = ok && (act_at[i] < 0 || (both(v[2 * i], tag) && both(v[2 * i + 1], tag)));
        if (__all(ok)) break;
        if (!pt.again()) break;
      }
#pragma unroll
      for (int i = 0; i < MAX_DOWN; i++) {
        const half8_t z = {0, 0, 0, 0, 0, 0, 0, 0};
        x[i] = act_at[i] >= 0 ? eight(v[2 * i], v[2 * i + 1]) : z;
      }
      load_gamma(nx, 0);
      float acc = mul_decoded(w, d0, x[0]);
      q0 = load_q(nx, 0);
      if (wave + WAVES < ks_f) acc += mul(d1, x[1]);
      q1 = load_q(nx, 1);
      if (wave + 2 * WAVES < ks_f) acc += mul(d2, x[2]);
      if (wave + 3 * WAVES < ks_f) acc += mul(d3, x[3]);
      put_part(0, acc);
    }
    lds_barrier();
    if (tid < 16) h += row_sum();
    if (!last) publish_h(m.x + m.at_attn, tag + 1);
    else if (tid < 16) m.h[own_row] = h;
    // nothing is left in these (a wave that loads no keys would else carry them round the loop)
#pragma unroll
    for (int t = 0; t < 8; t++) {
      asm volatile("" : "=v"(kf[t >> 2][t & 3]));
      asm volatile("" : "=v"(vf[t]));
    }
    if (kv_used) load_kv(nx, p_first);
    pb_now ^= 1;
  }
  if (wg == 0 && tid == 0) *m.steps += 1;  // every workgroup has read it before it published anything
}

// What the multi-kernel path leaves in its activation buffers, for the last layer of the last step, from the entries of that
// step (read_activation only).  One workgroup.
__global__ void __launch_bounds__(512) wide_report_kernel(LayersModel m, int pos, _Float16 *qkv, _Float16 *qrot, _Float16 *ao, _Float16 *act) {
  const int HQ = m.heads, HKV = m.kv_heads, G = m.G, tid = threadIdx.x;
  const int base = (2 * m.ff / 16) / G, rem = (2 * m.ff / 16) % G;
  const u64 *xq = m.x + m.at_qkv, *xa = m.x + m.at_act, *xo = m.x + m.at_ao;
  auto half_of = [](u64 e, int which) {
    U32H2 u;
    u.u = (uint32_t)e;
    return u.h[which];
  };
  for (int i = tid; i < (HQ + 2 * HKV) * HD; i += 512) qkv[i] = half_of(xq[qkv_entry(i & ~1)], i & 1);
  for (int i = tid; i < HQ * HD / 2; i += 512) {
    const int at = i / (HD / 2) * HD + i % (HD / 2), p = i % (HD / 2);
    const float inv_freq = 1.0f / powf(m.theta, (float)(2 * p) / (float)HD);
    float sn, cs;
    sincosf(inv_freq * (float)pos, &sn, &cs);
    const float x0 = (float)half_of(xq[qkv_entry(at & ~1)], at & 1), x1 = (float)half_of(xq[qkv_entry((at + HD / 2) & ~1)], at & 1);
    qrot[at] = narrow(fmaf(x0, cs, -(x1 * sn)));
    qrot[at + HD / 2] = narrow(fmaf(x0, sn, x1 * cs));
  }
  for (int i = tid; i < HQ * HD; i += 512) ao[i] = half_of(xo[(i >> 4) * 16 + ((i & 15) >> 1)], i & 1);
  for (int i = tid; i < m.ff; i += 512) act[i] = half_of(xa[act_entry(i / 8, base, rem) + (i & 7) / 2], i & 1);
}

// ---- host side -------------------------------------------------------------------------------------------------------
bool wide_supported(const yscv_hip_decoder_config &c, int num_cus) {
  if (c.head_dim != HD || c.group_size != 32 || c.n_heads % c.n_kv_heads != 0 || c.n_heads / c.n_kv_heads > 4) return false;
  const int G = c.d_model / 16, width = c.n_heads * HD;
  if (c.d_model % 512 != 0 || G > num_cus || 2 * G <= num_cus) return false;
  if (c.d_model > 512 * WAVES || width % 512 != 0 || width > 512 * WAVES || width > c.d_model) return false;
  if (c.d_ff % 128 != 0 || c.d_ff > 512 * WAVES * MAX_DOWN || c.n_kv_heads > G) return false;
  if ((c.n_heads + 2 * c.n_kv_heads) * HD / 16 > 2 * G) return false;
  const int gu = 2 * c.d_ff / 16;
  return gu <= MAX_GU * G && gu >= G;
}

void wide_exchange_entries(const yscv_hip_decoder_config &c, size_t out[6]) {
  const size_t G = c.d_model / 16;
  out[0] = out[1] = (size_t)c.d_model;
  out[2] = (size_t)(c.n_heads + 2 * c.n_kv_heads) * HD;
  out[3] = G * kLayersActSlots;
  out[4] = (size_t)c.n_heads * MAX_PIECES * HEAD_REC;
  out[5] = (size_t)c.n_heads * HD;
}

int32_t launch_decode_wide(const LayersModel &m, hipStream_t s) {
  hipLaunchKernelGGL(decode_wide_kernel, dim3(m.G), dim3(64 * WAVES), 0, s, m);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

int32_t launch_wide_report(const LayersModel &m, int pos, _Float16 *qkv, _Float16 *qrot, _Float16 *ao, _Float16 *act, hipStream_t s) {
  hipLaunchKernelGGL(wide_report_kernel, dim3(1), dim3(512), 0, s, m, pos, qkv, qrot, ao, act);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

}  // namespace yscv
