// One token through all layers of a small decoder (batch 1, head width 64, d_model <= 1024) in one launch: the step of
// the loop of apps/llm-bench/src/main.rs:525-548 between the embedding lookup and the final norm.
//
// A layer of such a model is 6 MB of weights, a microsecond of memory time, cut into five dependent stages (q/k/v, attention,
// o, gate/up, down).  As kernels of a graph each stage costs 2.5-5 us whatever it moves; here the workgroups stay resident
// and hand small vectors to each other.  24 layers of d_model 1024, 16 heads over 2, d_ff 2816: a step 690 -> 305 us at position
// 64, 945 -> 331 at 1000; 2715 -> 483 at 8128, 11155 -> 1270 at 32704 (these two with the LM head on the skinny kernel, 10 us more;
// the other path's attention has one workgroup per head).  With its norms folded and the one-row kernel in its projections the
// other path takes 500 at 100: there is no context at which it is the faster one.
//   * G = d_model / 16 workgroups of eight waves.  Workgroup w owns 16-row blocks of every projection, its eight waves split K
//     in tiles of 128, one 1 KiB load per (block, tile) in the layout the other int4 kernels use.  A wave's weights for a whole
//     layer fit its registers (2 + 1 + 6 + 3 tiles of 4 registers, and scales): the tiles of a stage are requested one or two
//     stages ahead and decoded while its input is on the way (decoded behind the input: 384 us a step instead of 345).
//   * A stage's input arrives as 8-byte {payload, tag} entries in global memory, written with agent-scope stores and
//     polled with coherent loads (the exchange of decode_persistent.hip).  A wave polls only the 128 values of its own tile:
//     one or two loads.  An exchange of 1024 values between 64 workgroups takes 0.97 us on its own, on one XCD as well as over
//     all eight, and 2.3 us where the workgroups also write entries into lines they share: so no line here has two writers, a
//     workgroup's entries of a line leave in one store where they can, and the sum of squares of a norm is not exchanged but
//     formed by the consumers, each wave its tile's part.
//   * Partial sums of the eight waves meet in LDS behind one barrier per stage (two buffers in turn).
//   * Attention: one workgroup takes 256 positions of one kv head (a wave 32), all its query heads as columns of the MFMA;
//     scores come out in the operand layout of the second product.  The waves of the output projection merge the chunks of
//     their two heads themselves: no stage in between.  (Every wave publishing its own 32 positions, without the merge in LDS:
//     378 instead of 332 us, the stores are more than the merge.)
// A layer takes 11 us: five exchanges of 1.0, 1.2 for the attention's arithmetic and merge, and per projection 0.2-0.6 of
// arithmetic, 0.1-0.5 until the slowest wave arrives and 0.3 for the sum and its epilogue.
// An entry buffer is written again one layer later.  Between the two lies a stage whose input comes from every
// workgroup behind its last read (layers_supported asks for what that takes: every workgroup owns rows of the residual and of
// gate/up), so no reader is overtaken.  Every wait is bounded; one that gives up sets *give_up, all others then return at
// once and the host reports it.  The host lets one launch of this kind run at a
// time (Resident in decoder.hip).
//
// Arithmetic: exact (q - 8) in fp16 against fp16 activations, f32 accumulation, group scale in f32 per 32 k, as the
// multi-kernel path does up to the order of sums.  Behind a norm the activation is fp16(h * gamma) with the largest of a
// wave's 128 values brought to 2^14 .. 2^15, the powers of two and the norm's factor follow the f32 sums: the same product
// as RMSNorm in front, with the rounding before the row factor.  Of the MFMA's 16 activation rows all carry the same row.
#include <hip/hip_runtime.h>

#include "decode_exchange.hpp"

namespace yscv {

namespace {

constexpr int WAVES = 8;
constexpr int MAX_QKV = 2, MAX_GU = 6, MAX_DOWN = 3;  // tiles a wave holds of q/k/v, gate/up (one K tile) and down
constexpr int HD = 64;

struct Tile {
  uint4_t w;   // 16 rows x 128 k, four 32-k words per lane
  half4_t s;   // scales of row lane & 15
};
struct Decoded {
  half8_t w[4];
};

}  // namespace

__global__ void __launch_bounds__(64 * WAVES, 2) decode_layers_kernel(LayersModel m) {
  __shared__ __attribute__((aligned(16))) _Float16 xs[WAVES][MAX_DOWN][128];  // a wave's activations, per tile
  __shared__ __attribute__((aligned(16))) float part[2][MAX_GU * 16][WAVES];  // per row the sums of the eight waves
  __shared__ __attribute__((aligned(16))) float wave_ss[2][WAVES];
  __shared__ float w_m[16][WAVES], w_l[16][WAVES];
  __shared__ float w_o[WAVES][16][HD];
  __shared__ __attribute__((aligned(16))) float rot[2][HD / 2];  // cos, sin of pair (i, i + 32) at this position
  int tid = threadIdx.x, lane = tid & 63;
  int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int r = lane & 15, c = lane >> 4;
  const int wg = blockIdx.x, G = m.G, L = m.n_layers, D = m.d;
  const int HQ = m.heads, HKV = m.kv_heads, GROUP = HQ / HKV;
  const int nt_q = (HQ + 2 * HKV) * HD / 16, nt_g = 2 * m.ff / 16;
  const int kt_d = D / 128, kt_o = HQ * HD / 128, kt_f = m.ff / 128;
  const int gu_base = nt_g / G, gu_rem = nt_g % G;
  const int gu_first = wg * gu_base + min(wg, gu_rem), gu_n = gu_base + (wg < gu_rem ? 1 : 0);
  const int pos_now = *m.pos;
  const int chunks = pos_now / kLayersChunk + 1;
  const int items = HKV * chunks;  // attention work items; item i runs on workgroup G - 1 - i mod G
  const int rec_step = GROUP * kLayersHeadRec, kv_step = layers_chunks(m.max_ctx) * rec_step;  // per chunk, per kv head
  const int item0 = G - 1 - wg;
  const uint32_t tag0 = *m.steps * (uint32_t)(L + 1) + 1u;
  Patience pt{POLL_LIMIT, m.give_up};
  NibbleConsts nc;
  nc.init();
  uint32_t magic_hi = 0x54005400u;
  asm volatile("" : "+v"(magic_hi));

  // blocks and tiles past the end are loaded again from the last one and not used
  auto load_tile = [&](const LayerAt &ly, int kind, int nt, int nts, int kt, int kts) {
    nt = nt < nts ? nt : nts - 1;
    kt = kt < kts ? kt : kts - 1;
    const size_t t = (size_t)nt * m.ktp[kind] + kt;
    Tile o;
    o.w = *reinterpret_cast<const uint4_t *>(ly.tiles[kind] + t * 1024 + lane * 16);
    o.s = *reinterpret_cast<const half4_t *>(ly.scales[kind] + (t * 16 + r) * 4);
    return o;
  };
  Tile tq[MAX_QKV], to, tg[MAX_GU], td[MAX_DOWN];
  float2 ga, gf;  // norm weights of this wave's tile, two per lane
  const int g_at = (wave < kt_d ? wave : 0) * 128 + 2 * lane;
  auto load_qkv = [&](const LayerAt &ly) {
#pragma unroll
    for (int b = 0; b < MAX_QKV; b++) tq[b] = load_tile(ly, 0, wg + G * b, nt_q, wave, kt_d);
    ga = *reinterpret_cast<const float2 *>(ly.gamma[0] + g_at);
  };
  auto load_o = [&](const LayerAt &ly) { to = load_tile(ly, 1, wg, G, wave, kt_o); };
  auto load_gu = [&](const LayerAt &ly) {
#pragma unroll
    for (int b = 0; b < MAX_GU; b++) tg[b] = load_tile(ly, 2, gu_first + min(b, gu_n - 1), nt_g, wave, kt_d);
    gf = *reinterpret_cast<const float2 *>(ly.gamma[1] + g_at);
  };
  auto load_down = [&](const LayerAt &ly) {
#pragma unroll
    for (int i = 0; i < MAX_DOWN; i++) td[i] = load_tile(ly, 3, wg, G, wave + WAVES * i, kt_f);
  };

  // Cached keys and values of 32 positions of an item: K rows as the A operand of the scores, in the order (row r of half pb
  // is position 8 (r / 4) + 4 pb + r % 4) that leaves a lane with the scores of positions 8c .. 8c + 7, which is one 16-byte
  // piece of V, the B operand of the second product.
  struct KvAt {
    uint32_t k[2], v;  // bytes
  };
  auto kv_at = [&](int item) {
    const int kvh = item % HKV, p0 = item / HKV * kLayersChunk + wave * 32;
    KvAt a;
#pragma unroll
    for (int pb = 0; pb < 2; pb++)
      a.k[pb] = (uint32_t)((kvh * m.max_ctx + min(p0 + 8 * (r >> 2) + 4 * pb + (r & 3), m.max_ctx - 1)) * HD + 8 * c) * 2u;
    a.v = (uint32_t)((kvh * (m.max_ctx / 8) + min((p0 >> 3) + c, m.max_ctx / 8 - 1)) * HD + r) * 16u;
    return a;
  };
  half8_t kf[2][2], vf[4];
  auto load_kv = [&](const LayerAt &ly, const KvAt &a) {
    const char *kc = reinterpret_cast<const char *>(ly.kc), *vc = reinterpret_cast<const char *>(ly.vc);
#pragma unroll
    for (int pb = 0; pb < 2; pb++)
#pragma unroll
      for (int j = 0; j < 2; j++) kf[pb][j] = *reinterpret_cast<const half8_t *>(kc + a.k[pb] + 64 * j);
#pragma unroll
    for (int t = 0; t < 4; t++) vf[t] = *reinterpret_cast<const half8_t *>(vc + a.v + 256 * t);
  };

  // weights of a stage are decoded while its input is on the way
  auto decode = [&](const Tile &t) {
    Decoded o;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      o.w[j] = decode_q8(t.w[j], nc, magic_hi);
      asm volatile("" : "+v"(o.w[j]));  // here, not behind the wait
    }
    return o;
  };
  // activations of tile i of this wave from LDS
  half8_t xa[4];
  auto read_x = [&](int i) {
#pragma unroll
    for (int j = 0; j < 4; j++) xa[j] = *reinterpret_cast<const half8_t *>(&xs[wave][i][32 * j + 8 * c]);
  };
  auto mul = [&](const Decoded &w, const half4_t &sc, float acc) {
    const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float4_t dd = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[j], w.w[j], zero, 0, 0, 0);
      acc = fmaf((float)sc[j], dd[0], acc);
    }
    return acc;
  };
  int pb_now = 0;  // which of the two sets of partial sums this stage uses
  auto put_part = [&](int b, float v) {
    if (lane < 16) part[pb_now][16 * b + lane][wave] = v;
  };
  auto sum8 = [](const float *p) {
    const float4_t a = *reinterpret_cast<const float4_t *>(p), b = *reinterpret_cast<const float4_t *>(p + 4);
    return ((a[0] + a[1]) + (a[2] + a[3])) + ((b[0] + b[1]) + (b[2] + b[3]));
  };
  auto row_sum = [&]() { return sum8(part[pb_now][tid]); };  // thread t: row t & 15 of block t >> 4
  auto row_rstd = [&]() { return __builtin_amdgcn_rsqf(sum8(wave_ss[pb_now]) / (float)D + m.eps); };

  // Input of a projection behind a norm: fp16(h * gamma * 2^e) of this wave's tile to LDS, 2^e from the largest of the 128
  // values, 2^-e (returned) for the wave's sums.  The other factor of the norm, common to all waves, follows the sums too:
  // the wave's part of the sum of squares meets the other seven there.
  auto take_normed = [&](const u64 *buf, uint32_t tag, const float2 &gamma) {
    if (wave >= kt_d) {
      if (lane == 0) wave_ss[pb_now][wave] = 0.0f;
      return 0.0f;
    }
    uint4_t v[1];
    while (true) {
      v[0] = get2(buf + wave * 128 + 2 * lane);
      landed(v);
      if (__all(both(v[0], tag))) break;
      if (!pt.again()) break;
    }
    const float h0 = as_f(v[0][0]), h1 = as_f(v[0][2]);
    const float x0 = h0 * gamma.x, x1 = h1 * gamma.y;
    const uint32_t top = (__float_as_uint(wave_max(fmaxf(fabsf(x0), fabsf(x1)))) >> 23) & 255u;
    const uint32_t f = min(268u - top, 253u);  // the largest value becomes 2^14 .. 2^15
    const float up = as_f(f << 23), down = as_f((254u - f) << 23);
    *reinterpret_cast<uint32_t *>(&xs[wave][0][2 * lane]) = pack2(narrow(x0 * up), narrow(x1 * up));
    const float ss = wave_sum(h0 * h0 + h1 * h1);
    if (lane == 0) wave_ss[pb_now][wave] = ss;
    wave_lds_sync();
    return down;
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
  publish_h((m.x + m.at_attn), tag0);
  load_qkv(m.layers[0]);
  load_o(m.layers[0]);
  const bool attends = item0 < items;  // uniform in the workgroup
  const bool kv_used = attends && item0 / HKV * kLayersChunk + wave * 32 <= pos_now;  // uniform in the wave
  const KvAt kv0 = kv_at(attends ? item0 : 0);
  if (kv_used) load_kv(m.layers[0], kv0);
  if (attends) {
    if (tid < HD / 2) {
      const float inv_freq = 1.0f / powf(m.theta, (float)(2 * tid) / (float)HD);
      sincosf(inv_freq * (float)pos_now, &rot[1][tid], &rot[0][tid]);
    }
    lds_barrier();
  }
  // where this lane finds its two entries of tiles wave + 8 hi and wave + 16 of the SwiGLU output (a load takes two tiles)
  const int hi = lane >> 5, e2 = 2 * (lane & 31);
  const bool act_a = wave + WAVES * hi < kt_f, act_b = hi == 0 && wave + 2 * WAVES < kt_f;
  const u64 *act_pa = (m.x + m.at_act) + (act_a ? act_entry((wave + WAVES * hi) * 16 + (e2 >> 2), gu_base, gu_rem) + (e2 & 3) : 0);
  const u64 *act_pb = (m.x + m.at_act) + (act_b ? act_entry((wave + 2 * WAVES) * 16 + (e2 >> 2), gu_base, gu_rem) + (e2 & 3) : 0);

#pragma unroll 1
  for (int l = 0; l < L; l++) {
    const uint32_t tag = tag0 + (uint32_t)l;
    const bool last = l + 1 == L;
    // Lane and wave numbers are opaque in every layer: comparisons and offsets made from them would else be kept over the
    // loop in more registers than there are, and moving them in and out costs more than making them again.
    asm volatile("" : "+v"(tid), "+s"(wave));
    lane = tid & 63;
    r = lane & 15;
    c = lane >> 4;
    // ---- q / k / v ---------------------------------------------------------------------------------------------------
    {
      Decoded w[MAX_QKV];
#pragma unroll
      for (int b = 0; b < MAX_QKV; b++) w[b] = decode(tq[b]);
      const float down = take_normed((m.x + m.at_attn), tag, ga);
      read_x(0);
#pragma unroll
      for (int b = 0; b < MAX_QKV; b++)
        if (wg + G * b < nt_q) put_part(b, wave < kt_d ? mul(w[b], tq[b].s, 0.0f) * down : 0.0f);
    }
    lds_barrier();
    if (tid < 16 * MAX_QKV) {
      const int nt = wg + G * (tid >> 4), row = 16 * nt + (tid & 15);
      if (nt < nt_q) {
        _Float16 v = narrow(row_sum() * row_rstd());
        const _Float16 *bias = m.layers[l].qkv_bias;
        if (bias) v = (_Float16)((float)v + (float)bias[row]);
        const float nxt = dpp_move<DPP_NEXT1>((float)v);
        if (!(tid & 1)) put_entry((m.x + m.at_qkv) + qkv_entry(row), pack2(v, (_Float16)nxt), tag);
      }
    }
    pb_now ^= 1;
    // ---- attention ---------------------------------------------------------------------------------------------------
#pragma unroll 1
    for (int item = item0; item < items; item += G) {
      int pos = pos_now;
      asm volatile("" : "+s"(pos));
      const int kvh = item % HKV, ch = item / HKV, p0 = ch * kLayersChunk + wave * 32;
      if (item != item0 && p0 <= pos) load_kv(m.layers[l], kv_at(item));
      const bool here = pos >= p0 && pos < p0 + 32;  // this wave has the position of the token: its k and v come with q
      const int rel = pos - p0;                      // 0 .. 31 then
      half8_t kn[2];
      _Float16 vn[4];
      float mx = -INFINITY, sum = 0.0f;
      float4_t o[4];
#pragma unroll
      for (int t = 0; t < 4; t++) o[t] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
      if (p0 <= pos) {  // uniform in the wave
        const u64 *qe = (m.x + m.at_qkv) + qkv_entry((kvh * GROUP + min(r, GROUP - 1)) * HD + 8 * c);
        const u64 *ke = (m.x + m.at_qkv) + qkv_entry((HQ + kvh) * HD + 8 * c);
        const u64 *ve = (m.x + m.at_qkv) + qkv_entry((HQ + HKV + kvh) * HD + (r & ~3));
        uint4_t vq[4], vk[8];  // vk: k, then v of channels 16 t + r
#pragma unroll
        for (int i = 0; i < 8; i++) vk[i] = uint4_t{0u, tag, 0u, tag};
        while (true) {
          // eight channels of both halves of a head: a half is two blocks of 16 rows further
          vq[0] = get2(qe);
          vq[1] = get2(qe + 2);
          vq[2] = get2(qe + 32);
          vq[3] = get2(qe + 34);
          if (here) {
            vk[0] = get2(ke);
            vk[1] = get2(ke + 2);
            vk[2] = get2(ke + 32);
            vk[3] = get2(ke + 34);
#pragma unroll
            for (int t = 0; t < 4; t++) vk[4 + t] = get2(ve + 16 * t);
          }
          landed(vk);
          landed(vq);
          bool ok = true;
#pragma unroll
          for (int i = 0; i < 4; i++) ok = ok && both(vq[i], tag) && both(vk[i], tag) && both(vk[4 + i], tag);
          if (__all(ok)) break;
          if (!pt.again()) break;
        }
        float cs[8], sn[8];
#pragma unroll
        for (int e = 0; e < 8; e++) {
          cs[e] = rot[0][8 * c + e];
          sn[e] = rot[1][8 * c + e];
        }
        auto rotate = [&](const uint4_t *v, half8_t (&out)[2]) {
#pragma unroll
          for (int i = 0; i < 4; i++) {
            U32H2 a, b;
            a.u = v[i >> 1][2 * (i & 1)];
            b.u = v[2 + (i >> 1)][2 * (i & 1)];
#pragma unroll
            for (int u = 0; u < 2; u++) {
              const float x0 = (float)a.h[u], x1 = (float)b.h[u];
              out[0][2 * i + u] = narrow(fmaf(x0, cs[2 * i + u], -(x1 * sn[2 * i + u])));
              out[1][2 * i + u] = narrow(fmaf(x0, sn[2 * i + u], x1 * cs[2 * i + u]));
            }
          }
        };
        half8_t qf[2];
        rotate(vq, qf);
        if (here) {
          rotate(vk, kn);
          const bool mine = (r >> 2) == (rel >> 3) && (r & 3) == (rel & 3);
#pragma unroll
          for (int pb = 0; pb < 2; pb++)
            if (pb == ((rel >> 2) & 1)) {  // uniform
#pragma unroll
              for (int j = 0; j < 2; j++) kf[pb][j] = mine ? kn[j] : kf[pb][j];
            }
          // the token's v, and 0 behind it (what the cache holds there may be anything, and 0 * inf would not be 0)
#pragma unroll
          for (int t = 0; t < 4; t++) {
            U32H2 u;
            u.u = (r & 2) ? vk[4 + t][2] : vk[4 + t][0];
            vn[t] = (r & 1) ? u.h[1] : u.h[0];
#pragma unroll
            for (int e = 0; e < 8; e++) vf[t][e] = 8 * c + e < rel ? vf[t][e] : (8 * c + e == rel ? vn[t] : (_Float16)0.0f);
          }
        }
        // lane (r, c): score of head r at positions p0 + 8c + e
        float sv[8], pe[8];
#pragma unroll
        for (int pb = 0; pb < 2; pb++) {
          float4_t s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int j = 0; j < 2; j++) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[pb][j], qf[j], s, 0, 0, 0);
#pragma unroll
          for (int q = 0; q < 4; q++) sv[4 * pb + q] = s[q] * 0.125f;
        }
        if (here) {
#pragma unroll
          for (int e = 0; e < 8; e++) sv[e] = 8 * c + e <= rel ? sv[e] : -INFINITY;
        }
#pragma unroll
        for (int e = 0; e < 8; e++) mx = fmaxf(mx, sv[e]);
        mx = max_xor16_xor32(mx);
        half8_t pf;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          pe[e] = sv[e] == -INFINITY ? 0.0f : __expf(sv[e] - mx);
          sum += pe[e];
          pf[e] = (_Float16)pe[e];
        }
        sum = sum_xor16_xor32(sum);
#pragma unroll
        for (int t = 0; t < 4; t++) {
          o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(pf, vf[t], o[t], 0, 0, 0);  // lane (r, c): head 4c + q at 16 t + r
        }
      }
      if (lane < 16) {
        w_m[lane][wave] = mx;
        w_l[lane][wave] = sum;
      }
#pragma unroll
      for (int t = 0; t < 4; t++)
#pragma unroll
        for (int q = 0; q < 4; q++)
          if (4 * c + q < GROUP) w_o[wave][4 * c + q][16 * t + r] = o[t][q];
      lds_barrier();
      u64 *rec = (m.x + m.at_part) + (size_t)kvh * kv_step + ch * rec_step;
      for (int hh = wave; hh < GROUP; hh += WAVES) {  // a wave merges a head: lane = channel
        const float mw = w_m[hh][lane & 7], M = row_max16(mw);
        const float fw = mw == -INFINITY ? 0.0f : __expf(mw - M);
        const float ls = 0.5f * row_sum16(w_l[hh][lane & 7] * fw);  // (a row of 16 lanes holds the eight waves twice)
        float os = 0.0f;
#pragma unroll
        for (int w = 0; w < WAVES; w++)
          os += w_o[w][hh][lane] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(fw), w));
        put_entry(rec + hh * kLayersHeadRec + lane, __float_as_uint(os), tag);
        if (lane < 2) put_entry(rec + hh * kLayersHeadRec + HD + lane, __float_as_uint(lane ? ls : M), tag);
      }
      if (here) {  // the token's row of the cache
        _Float16 *kc = m.layers[l].kc, *vc = m.layers[l].vc;
        if ((r >> 2) == (rel >> 3) && (r & 3) == (rel & 3)) {
          _Float16 *kd = kc + ((size_t)kvh * m.max_ctx + pos) * HD + 8 * c;
          *reinterpret_cast<half8_t *>(kd) = kn[0];
          *reinterpret_cast<half8_t *>(kd + 32) = kn[1];
        }
        if (c == 0) {
#pragma unroll
          for (int t = 0; t < 4; t++) vc[(((size_t)kvh * (m.max_ctx / 8) + pos / 8) * HD + 16 * t + r) * 8 + (pos & 7)] = vn[t];
        }
      }
      lds_barrier();  // the states are written again by the next item
    }
    // ---- output projection: this wave's tile is the two heads 2 wave, 2 wave + 1, lane pairs of channels -----------------
    load_gu(m.layers[l]);
    {
      const Decoded w = decode(to);
      if (wave < kt_o) {
        const int head = 2 * wave + (lane >> 5), kvh = head / GROUP;
        const u64 *rec0 = (m.x + m.at_part) + (size_t)kvh * kv_step;
        const int at_m = head % GROUP * kLayersHeadRec + HD, at_o = at_m - HD + 2 * (lane & 31);
        float M = -INFINITY, ls = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll 1
        for (int c0 = 0; c0 < chunks; c0 += 4) {
          uint4_t v[8];
          while (true) {
            bool ok = true;
#pragma unroll
            for (int i = 0; i < 4; i++) {  // chunks past the end repeat the last one
              const u64 *rec = rec0 + (size_t)min(c0 + i, chunks - 1) * rec_step;
              v[2 * i] = get2(rec + at_m);
              v[2 * i + 1] = get2(rec + at_o);
            }
            landed(v);
#pragma unroll
            for (int i = 0; i < 8; i++) ok = ok && both(v[i], tag);
            if (__all(ok)) break;
            if (!pt.again()) break;
          }
#pragma unroll
          for (int i = 0; i < 4; i++)
            if (c0 + i < chunks) {  // uniform
              const float mc = as_f(v[2 * i][0]), Mn = fmaxf(M, mc);
              const float fa = M == -INFINITY ? 0.0f : __expf(M - Mn), fb = mc == -INFINITY ? 0.0f : __expf(mc - Mn);
              ls = ls * fa + as_f(v[2 * i][2]) * fb;
              o0 = o0 * fa + as_f(v[2 * i + 1][0]) * fb;
              o1 = o1 * fa + as_f(v[2 * i + 1][2]) * fb;
              M = Mn;
            }
        }
        const float inv = ls > 0.0f ? 1.0f / ls : 0.0f;
        const uint32_t x2 = pack2(narrow(o0 * inv), narrow(o1 * inv));
        *reinterpret_cast<uint32_t *>(&xs[wave][0][2 * lane]) = x2;
        wave_lds_sync();
      }
      read_x(0);
      put_part(0, wave < kt_o ? mul(w, to.s, 0.0f) : 0.0f);
    }
    lds_barrier();
    if (tid < 16) h += row_sum();
    publish_h((m.x + m.at_ffn), tag);
    pb_now ^= 1;
    // ---- gate / up + SwiGLU --------------------------------------------------------------------------------------------
    load_down(m.layers[l]);
    {
      Decoded w[MAX_GU];
#pragma unroll
      for (int b = 0; b < MAX_GU; b++) w[b] = decode(tg[b]);
      const float down = take_normed((m.x + m.at_ffn), tag, gf);
      read_x(0);
#pragma unroll
      for (int b = 0; b < MAX_GU; b++)
        if (b < gu_n) put_part(b, wave < kt_d ? mul(w[b], tg[b].s, 0.0f) * down : 0.0f);
    }
    lds_barrier();
    if (tid < 16 * gu_n) {
      const float v = row_sum() * row_rstd();
      const _Float16 a = narrow(silu(v) * dpp_move<DPP_NEXT1>(v));  // even rows are gates, odd ones ups
      const float a2 = dpp_move<DPP_NEXT2>((float)a);
      if (!(tid & 3)) put_entry((m.x + m.at_act) + wg * kLayersActSlots + (tid >> 2), pack2(a, (_Float16)a2), tag);
    }
    pb_now ^= 1;
    // ---- down ----------------------------------------------------------------------------------------------------------
    if (!last) {
      load_qkv(m.layers[l + 1]);
      if (kv_used) load_kv(m.layers[l + 1], kv0);
    }
    {
      Decoded w[MAX_DOWN];
#pragma unroll
      for (int i = 0; i < MAX_DOWN; i++) w[i] = decode(td[i]);
      uint4_t v[2];
      while (true) {
        v[0] = get2(act_pa);
        v[1] = get2(act_pb);
        landed(v);
        if (__all((!act_a || both(v[0], tag)) && (!act_b || both(v[1], tag)))) break;
        if (!pt.again()) break;
      }
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      if (act_a) *reinterpret_cast<u32x2 *>(&xs[wave][hi][2 * e2]) = u32x2{v[0][0], v[0][2]};
      if (act_b) *reinterpret_cast<u32x2 *>(&xs[wave][2][2 * e2]) = u32x2{v[1][0], v[1][2]};
      wave_lds_sync();
      float acc = 0.0f;
#pragma unroll
      for (int i = 0; i < MAX_DOWN; i++)
        if (wave + WAVES * i < kt_f) {  // uniform
          read_x(i);
          acc = mul(w[i], td[i].s, acc);
        }
      put_part(0, acc);
    }
    lds_barrier();
    if (tid < 16) h += row_sum();
    if (!last) publish_h((m.x + m.at_attn), tag + 1);
    else if (tid < 16) m.h[own_row] = h;
    if (!last) load_o(m.layers[l + 1]);
    pb_now ^= 1;
  }
  if (wg == 0 && tid == 0) *m.steps += 1;  // every workgroup has read it before it published anything
}

// What the multi-kernel path leaves in its activation buffers, for the last layer of the last step, from the entries of that
// step (read_activation only).  One workgroup.
__global__ void __launch_bounds__(512) layers_report_kernel(LayersModel m, int pos, _Float16 *qkv, _Float16 *qrot, _Float16 *ao,
                                                            _Float16 *act) {
  const int HQ = m.heads, HKV = m.kv_heads, GROUP = HQ / HKV, G = m.G, tid = threadIdx.x;
  const int base = (2 * m.ff / 16) / G, rem = (2 * m.ff / 16) % G;
  const u64 *xq = m.x + m.at_qkv, *xa = m.x + m.at_act, *xp = m.x + m.at_part;
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
  for (int i = tid; i < m.ff; i += 512) act[i] = half_of(xa[act_entry(i / 8, base, rem) + (i & 7) / 2], i & 1);
  const int rec_step = GROUP * kLayersHeadRec, kv_step = layers_chunks(m.max_ctx) * rec_step;
  const int chunks = pos / kLayersChunk + 1;
  for (int i = tid; i < HQ * HD; i += 512) {
    const int head = i / HD;
    const u64 *rec = xp + (size_t)(head / GROUP) * kv_step;
    const int at_m = head % GROUP * kLayersHeadRec + HD, at_o = at_m - HD + i % HD;
    float M = -INFINITY, ls = 0.0f, o = 0.0f;
    for (int k = 0; k < chunks; k++, rec += rec_step) {
      const float mc = as_f((uint32_t)rec[at_m]), Mn = fmaxf(M, mc);
      const float fa = M == -INFINITY ? 0.0f : __expf(M - Mn), fb = mc == -INFINITY ? 0.0f : __expf(mc - Mn);
      ls = ls * fa + as_f((uint32_t)rec[at_m + 1]) * fb;
      o = o * fa + as_f((uint32_t)rec[at_o]) * fb;
      M = Mn;
    }
    ao[i] = narrow(o * (ls > 0.0f ? 1.0f / ls : 0.0f));
  }
}

// ---- host side -------------------------------------------------------------------------------------------------------
bool layers_supported(const yscv_hip_decoder_config &c, int num_cus) {
  if (c.head_dim != HD || c.group_size != 32 || c.n_heads % c.n_kv_heads != 0 || c.n_heads / c.n_kv_heads > 16) return false;
  if (c.d_model % 128 != 0 || c.d_model > 1024 || c.d_ff % 128 != 0 || (c.n_heads * HD) % 128 != 0) return false;
  const int G = c.d_model / 16;
  if (G > num_cus) return false;
  // one K tile per wave behind the norms and the attention, up to three of the FFN's width
  if (c.n_heads * HD > 128 * WAVES || c.d_ff > 128 * WAVES * MAX_DOWN) return false;
  if ((c.n_heads + 2 * c.n_kv_heads) * HD / 16 > MAX_QKV * G) return false;
  const int gu = 2 * c.d_ff / 16;
  if (gu > MAX_GU * G || gu < G) return false;
  return (int64_t)c.n_kv_heads * c.max_ctx * HD * 2 < (1ll << 31);  // byte offsets into a layer's cache
}

void layers_exchange_entries(const yscv_hip_decoder_config &c, size_t out[5]) {
  const size_t G = c.d_model / 16;
  out[0] = out[1] = (size_t)c.d_model;
  out[2] = (size_t)(c.n_heads + 2 * c.n_kv_heads) * HD;
  out[3] = G * kLayersActSlots;
  out[4] = (size_t)c.n_kv_heads * layers_chunks(c.max_ctx) * (c.n_heads / c.n_kv_heads) * kLayersHeadRec;
}

int32_t launch_decode_layers(const LayersModel &m, hipStream_t s) {
  hipLaunchKernelGGL(decode_layers_kernel, dim3(m.G), dim3(64 * WAVES), 0, s, m);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

int32_t launch_layers_report(const LayersModel &m, int pos, _Float16 *qkv, _Float16 *qrot, _Float16 *ao, _Float16 *act, hipStream_t s) {
  hipLaunchKernelGGL(layers_report_kernel, dim3(1), dim3(512), 0, s, m, pos, qkv, qrot, ao, act);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

}  // namespace yscv
