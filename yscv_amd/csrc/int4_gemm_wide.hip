// Packed-int4 matmul for many rows (fp16-prepared activations): y[m][n] = sum_k x[m][k] * W[n][k] in tiles of 256 or 128 rows x 256 or
// 192 columns.  Replaces packed_int4_gemm_dispatch (crates/yscv-kernels/src/ops/int4_matmul.rs:548-605) where int4_plan
// (int4_gemm_plan.hpp) finds such tiles faster than the LDS-ring GEMM's.
//
// Bound by the matrix cores and by the power they take: the card holds its power, and the clock falls to 1.5 .. 1.75 GHz with all CUs in
// this loop.  What is left to win is work beside the MFMAs, so each weight is decoded once: four waves, one per SIMD, stand side by
// side in columns and each takes ALL rows of the tile.  A wave owns 16 MT rows x 16 NT columns (256 x 64: its accumulators are the
// accumulation half of the register file), reads a packed word once per 128 k and decodes it in registers, where it feeds MT MFMAs.
// Per 32 k a 256 x 256 tile moves 16 KB of activations and 4 KB of packed weights into LDS and 64 + 4 KB of fragments out, in 1024 cycles.
// With one wave per SIMD nobody else fills a gap, and a SIMD issues an instruction every four cycles, an MFMA being two of them and the
// matrix pipe taking one every 16 cycles: two more instructions of ANY kind fit behind each MFMA, a third makes the pipe wait.  So the
// loop is laid out by hand: MFMAs and the 13 instructions that make eight weights are asm statements in their order, fragments are
// waited for in pairs, loads (m0 in front of an MFMA, the load behind it) leave one to a row tile.
// Everything arrives by LDS-direct loads whose count each wave knows: activations in three slots of 64 k (XOR-swizzled as in
// the LDS-ring GEMM), weights and scales in two of 128 k, used only by the wave that asked for them.  One barrier per 64 k.
// Power is also why a row of tiles goes through its columns forwards and the next one backwards: between two MFMAs one operand stays
// (registers only, all CUs, fp16 rows of a normal distribution and scaled int4 weights, clock settled: 2014 -> 2060 TFLOP/s; with
// 32 x 32 x 16 MFMAs 1725, operands in the other order 1965).  Whole op, 2048 x 14336 x 4096 with zero points, bf16: 194.8 -> 191.9 us.
// The group scale is folded into fp16 weights as in the LDS-ring GEMM, products are added in the same order: same results.
// A 64-k stage of a 256 x 256 tile: 2500 cycles (2048 of MFMAs; 2150 without the decode, 2170 without the fragment reads).  Eight waves of
// 128 x 64, which decode every weight twice and which the compiler schedules: 3100.  Registers spent otherwise do not help: the same
// tile with the MFMAs left to the compiler copies accumulators between the halves of the register file.
// us of the whole op, eight waves -> this: m x n x k, fp16 rows, replayed (clock settled): 2048 x 14336 x 4096 197 -> 179, with zero
// points in 128-groups 208 -> 188, 2048 x 8192 x 4096 113 -> 100, 2048 x 8192 x 8192 210 -> 190, 2048 x 14336 x 1024 66 -> 56.  The 128-row
// tiles against the LDS-ring GEMM: 2048 x 4096 x 4096 71 -> 58, 512 x 14336 x 4096 66 -> 53.
#include <mutex>
#include <type_traits>

#include "int4_common.hpp"
#include "int4_gemm_plan.hpp"
#include "kernels.hpp"

namespace yscv {

namespace {

constexpr int WG_WAVES = 4, WG_THREADS = 64 * WG_WAVES;
constexpr int WG_XSLOTS = 3;  // activations of 64 k; packed weights and scales of 128 k have two slots

struct WideArgs {
  const uint8_t *tiles;
  const void *tscales;
  const uint8_t *tzps;
  const _Float16 *xh;
  const float *row_scale;  // null: 1
  void *y;
  int m, n, col0;  // rows; end and begin of the column range (col0 a multiple of 16)
  int ldy;         // columns of the whole product
  int nt, kt, ktp, chunks, chunk_div;
  int ldx, stages;  // row stride of xh; 64-k stages that hold data
  int16_t y_dtype, epi;
  int tiles_m, tiles_n;
  int kt_per, parts;  // K split: 128-k tiles of a part; y is f32 [parts][m][ldy] then
};
static_assert(sizeof(WideArgs) <= kCheapArgs, "arguments of a launch");

// Scales (and zero points) of a wave's NT blocks and 128 k
template <int GM, bool SF16, bool HAS_ZP, int NT>
struct WideScale {
  static constexpr int SPT = GM == GM32 ? 4 : (GM == GM64 ? 2 : 1);
  static constexpr int BLOCK = 16 * SPT * (SF16 ? 2 : 4);     // bytes of one 16-column block
  static constexpr int LOADS = (NT * BLOCK + 255) / 256;      // 4-byte-per-lane loads of a wave's blocks
  static constexpr int ZBLOCK = 16 * SPT;
  static constexpr int ZLOADS = HAS_ZP ? (NT * ZBLOCK + 255) / 256 : 0;
  static constexpr int BYTES = (LOADS + ZLOADS) * 256;        // LDS per wave and slot
  typedef typename std::conditional<SF16, _Float16, float>::type elem_t;
  typedef elem_t vec_t __attribute__((ext_vector_type(SPT)));
};

// A tile of MT x 4 NT blocks of 16
template <int GM, bool SF16, bool HAS_ZP, int MT, int NT>
struct WideTile {
  static constexpr int BM = 16 * MT, BN = 16 * NT * WG_WAVES;
  static constexpr int XSLOT = BM * 128, WSLOT = NT * WG_WAVES * 1024;
  static constexpr int LOOP = WG_XSLOTS * XSLOT + 2 * WSLOT + WG_WAVES * 2 * WideScale<GM, SF16, HAS_ZP, NT>::BYTES;
  static constexpr int HALF = BM / 2 * (BN * 4 + 16), LDS = LOOP > HALF ? LOOP : HALF;  // (the epilogue: half of the rows in f32)
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

template <int N>
__device__ __forceinline__ void wide_barrier() {
  // this wave's loads of the stage have landed and its fragment reads of the last one have returned; then everyone's
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int GM, bool SF16, bool HAS_ZP, int MT, int NT>
__global__ void __launch_bounds__(WG_THREADS, 1) int4_gemm_wide_kernel(WideArgs p) {
  using S = WideScale<GM, SF16, HAS_ZP, NT>;
  using T = WideTile<GM, SF16, HAS_ZP, MT, NT>;
  constexpr int XL = MT / 2, WL = NT, SL = S::LOADS + S::ZLOADS;  // loads per wave
  // (Half the rows with zero points per 32 or 64 k are bound by what decodes them, not by power: 811 x 7811 x 8096, bf16 and zero points per 32,
  // 117.4 us there and back, 114.9 in order; without zero points 102.9 and 103.7)
  constexpr bool BACK = MT > 8 || !HAS_ZP || GM == GM128;
  constexpr int PM = MT / 2, AHEAD = 3;  // pairs of row tiles; fragments of x are read that many pairs ahead, into four pairs of registers
  static_assert(PM % 4 == 0, "a pair's registers are known at compile time");
  extern __shared__ __attribute__((aligned(1024))) uint8_t wide_lds[];
  // Tiles are numbered down bands of eight row tiles, column by column; an XCD (workgroup ids equal modulo 8) takes an eighth
  // of them in a row: 32 neighbours share row and column panels in its L2, and no XCD has more than its share (super-blocks of
  // 32 tiles gave four XCDs a second one at three row tiles x 85 columns: 700 x 24000 x 2048 140 us against 98)
  const int tiles = p.tiles_m * p.tiles_n, share = (tiles * p.parts + 7) >> 3;
  int t = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || t >= tiles * p.parts) return;
  const int part = t / tiles, kt0 = part * p.kt_per, stages = min(p.stages - 2 * kt0, 2 * p.kt_per);
  t -= part * tiles;
  const int band = t / (8 * p.tiles_n), in_band = t - band * 8 * p.tiles_n, rows = min(8, p.tiles_m - 8 * band);
  const int tn = in_band / rows, tm = 8 * band + in_band % rows;
  const int m0 = tm * T::BM, n0 = p.col0 + tn * T::BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4, first = NT * wave, nb0 = n0 / 16 + first;
  NibbleConsts nc;
  nc.init();

  const uint32_t lds0 = (uint32_t)(size_t)wide_lds;
  uint8_t *w_lds = wide_lds + WG_XSLOTS * T::XSLOT;
  uint8_t *s_lds = w_lds + 2 * T::WSLOT + wave * 2 * S::BYTES;
  const uint32_t w_off = lds0 + WG_XSLOTS * T::XSLOT, s_off = w_off + 2 * T::WSLOT + (uint32_t)(wave * 2 * S::BYTES);

  // ---- load addresses: uniform base + 32-bit lane offsets.  x piece q of a stage: rows 8 q .. 8 q + 7, 128 bytes each
  uint32_t xoff[XL];
#pragma unroll
  for (int u = 0; u < XL; u++) {
    const int q = wave * XL + u, row8 = lane >> 3, row = min(m0 + 8 * q + row8, p.m - 1);
    xoff[u] = (uint32_t)(((size_t)row * p.ldx + ((lane & 7) ^ (4 * (q & 1) + (row8 >> 1))) * 8) * 2);
  }
  // (blocks past the matrix repeat the last one)
  const int blk0 = min(nb0, p.nt - 1);
  uint32_t woff[WL];
#pragma unroll
  for (int u = 0; u < WL; u++) woff[u] = lane * 16 + (uint32_t)(min(nb0 + u, p.nt - 1) - blk0) * (uint32_t)p.ktp * kTileBytes;
  // scales (zero points) of the wave's blocks: byte 4 lane + 256 u of them
  uint32_t scoff[S::LOADS], zpoff[S::ZLOADS > 0 ? S::ZLOADS : 1];
#pragma unroll
  for (int u = 0; u < S::LOADS; u++) {
    const int byte = (u * 256 + lane * 4) % (NT * S::BLOCK), blk = min(nb0 + byte / S::BLOCK, p.nt - 1);
    scoff[u] = (uint32_t)blk * (uint32_t)(p.chunks * S::BLOCK) + (uint32_t)(byte % S::BLOCK);
  }
#pragma unroll
  for (int u = 0; u < S::ZLOADS; u++) {
    const int byte = (u * 256 + lane * 4) % (NT * S::ZBLOCK), blk = min(nb0 + byte / S::ZBLOCK, p.nt - 1);
    zpoff[u] = (uint32_t)blk * (uint32_t)(p.chunks * S::ZBLOCK) + (uint32_t)(byte % S::ZBLOCK);
  }
  // A group of loads: first W = WL + SL of a 128-k tile (or none), then XL of a stage.  Where they come from and go to:
  const char *x_base, *w_base, *s_base, *z_base;
  uint32_t x_m0, w_m0, s_m0;
  auto aim_x = [&](int st, uint32_t slot) __attribute__((always_inline)) {
    x_base = reinterpret_cast<const char *>(p.xh) + (size_t)(2 * kt0 + min(st, stages - 1)) * 128;
    x_m0 = lds0 + slot + (uint32_t)(wave * XL * 1024);
  };
  auto aim_w = [&](int kt) __attribute__((always_inline)) {
    const uint32_t slot = (uint32_t)(kt & 1);
    kt = kt0 + min(kt, (stages - 1) >> 1);
    const int chunk = GM == GM128 ? kt / p.chunk_div : kt;
    w_base = reinterpret_cast<const char *>(p.tiles) + ((size_t)blk0 * p.ktp + kt) * kTileBytes;
    s_base = reinterpret_cast<const char *>(p.tscales) + (size_t)chunk * S::BLOCK;
    if (HAS_ZP) z_base = reinterpret_cast<const char *>(p.tzps) + (size_t)chunk * S::ZBLOCK;
    w_m0 = w_off + slot * T::WSLOT + (uint32_t)(first * 1024);
    s_m0 = s_off + slot * S::BYTES;
  };
  // load l of a group: where it goes (one instruction at least in front of the load), and the load
  auto load_to = [&](int l, int W) __attribute__((always_inline)) {
    const uint32_t to = l >= W ? x_m0 + (l - W) * 1024 : (l < WL ? w_m0 + l * 1024 : s_m0 + (l - WL) * 256);
    asm volatile("s_mov_b32 m0, %0" ::"s"(to));
  };
  auto load = [&](int l, int W) __attribute__((always_inline)) {
    if (l >= W) asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(xoff[l - W < XL ? l - W : 0]), "s"(x_base));
    else if (l < WL) asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(woff[l]), "s"(w_base));
    else if (l < WL + S::LOADS) asm volatile("global_load_lds_dword %0, %1" ::"v"(scoff[l - WL]), "s"(s_base));
    else asm volatile("global_load_lds_dword %0, %1" ::"v"(zpoff[l - WL - S::LOADS]), "s"(z_base));
  };
  auto load_all = [&](int l0, int l1, int W) __attribute__((always_inline)) {
#pragma unroll
    for (int l = l0; l < l1; l++) {
      load_to(l, W);
      asm volatile("s_nop 0");
      load(l, W);
    }
  };

  // ---- LDS -> registers
  typedef uint32_t word_pair_t __attribute__((ext_vector_type(2)));
  word_pair_t wq[2][NT];  // words of a stage's two k-steps: of even and of odd stages
  auto read_w = [&](int kt, int half) {
    const uint8_t *src = w_lds + (kt & 1) * T::WSLOT + first * 1024 + lane * 16 + half * 8;
#pragma unroll
    for (int j = 0; j < NT; j++) wq[half][j] = *reinterpret_cast<const word_pair_t *>(src + j * 1024);
  };
  constexpr int SR = GM == GM32 ? 2 : 1;  // registers of a block's scales of 128 k, as fp16 pairs (f32 scales are rounded as the weights are)
  half2_t sv[NT][SR];
  uint32_t zv[HAS_ZP ? NT : 1];
  auto read_s = [&](int kt) {
    const uint8_t *ss = s_lds + (kt & 1) * S::BYTES;
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const typename S::vec_t v = *reinterpret_cast<const typename S::vec_t *>(ss + j * S::BLOCK + r * (S::BLOCK / 16));
#pragma unroll
      for (int e = 0; e < S::SPT; e++) sv[j][e >> 1][e & 1] = (_Float16)v[e];
      if constexpr (HAS_ZP) {
        const uint8_t *z = ss + S::LOADS * 256 + j * S::ZBLOCK + r * S::SPT;
        if constexpr (GM == GM32) zv[j] = *reinterpret_cast<const uint32_t *>(z);
        else if constexpr (GM == GM64) zv[j] = *reinterpret_cast<const uint16_t *>(z);
        else zv[j] = *z;
      }
    }
  };
  // what is added to 1024 + q and to 64 + q: minus (offset + zero point)
  half2_t c1[HAS_ZP ? NT : 1], c2[HAS_ZP ? NT : 1];
  if constexpr (!HAS_ZP) {
    c1[0] = half2_t{(_Float16)-1032.0f, (_Float16)-1032.0f};
    c2[0] = half2_t{(_Float16)-72.0f, (_Float16)-72.0f};
  }
  auto offsets = [&](int ks) {  // of the group that k-step ks of a tile begins
    if constexpr (HAS_ZP) {
      if (GM == GM64 ? (ks & 1) != 0 : (GM == GM128 && ks != 0)) return;
      const int e = GM == GM32 ? ks : (GM == GM64 ? ks >> 1 : 0);
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const _Float16 z = (_Float16)(float)((zv[j] >> (8 * e)) & 0xFFu), z1 = (_Float16)(-1024.0f) - z, z2 = (_Float16)(-64.0f) - z;
        c1[j] = half2_t{z1, z1};
        c2[j] = half2_t{z2, z2};
      }
    }
  };
  // Instruction o of the 13 that make eight fp16 weights of block j for k-step ks: decode8_exact times the group's scale.  They are
  // statements of their own because their places between the MFMAs matter (below).
  constexpr int OPS = 13;
  const uint32_t sixteenth = 0x2C002C00u;
  uint32_t dq[4], dq2;
  union Frag {
    half8_t h;
    uint32_t u[4];
  };
  Frag b[2][NT];
  auto decode_op = [&](int o, int j, auto KS) __attribute__((always_inline)) {
    constexpr int ks = decltype(KS)::value, e = GM == GM32 ? ks : (GM == GM64 ? ks >> 1 : 0);
    const uint32_t w = wq[ks >> 1][j][ks & 1];
    const half2_t off1 = c1[HAS_ZP ? j : 0], off2 = c2[HAS_ZP ? j : 0], sc = sv[j][e >> 1];
    Frag &out = b[ks & 1][j];
    if (o == 0) asm volatile("v_lshrrev_b32 %0, 8, %1" : "=v"(dq2) : "v"(w));
    else if (o == 1 || o == 3) asm volatile("v_and_or_b32 %0, %1, %2, %3" : "=v"(dq[o - 1]) : "v"(o == 1 ? w : dq2), "s"(nc.lo), "v"(nc.magic));
    else if (o == 2 || o == 4) asm volatile("v_and_or_b32 %0, %1, %2, %3" : "=v"(dq[o - 1]) : "v"(o == 2 ? w : dq2), "s"(nc.hi), "v"(nc.magic));
    else if (o == 5 || o == 7) asm volatile("v_pk_add_f16 %0, %0, %1" : "+v"(dq[o - 5]) : "v"(off1));
    else if (o == 6 || o == 8) asm volatile("v_pk_fma_f16 %0, %0, %1, %2" : "+v"(dq[o - 5]) : "s"(sixteenth), "v"(off2));
    else if ((e & 1) == 0) asm volatile("v_pk_mul_f16 %0, %1, %2 op_sel_hi:[1,0]" : "=v"(out.u[o - 9]) : "v"(dq[o - 9]), "v"(sc));
    else asm volatile("v_pk_mul_f16 %0, %1, %2 op_sel:[0,1]" : "=v"(out.u[o - 9]) : "v"(dq[o - 9]), "v"(sc));
  };
  const uint32_t g = 4u * (r >> 3) + ((r & 7) >> 1);
  const uint32_t rd0 = (uint32_t)((r >> 3) * 1024) + (((r & 7) * 8 + (c ^ g)) * 16);  // k-step 1: ^ 64
  auto read_a = [&](int i, uint32_t slot, int h) { return *reinterpret_cast<const half8_t *>(wide_lds + slot + i * 2048 + (rd0 ^ (64u * h))); };

  float4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  half8_t a[8];
  // In place and in order: the accumulators fill the accumulation registers, any copy of one would cost more than it could give.
  auto mfma = [&](int i, int j, const Frag &bb) __attribute__((always_inline)) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(bb.h), "v"(a[i % 8]));
  };

  uint32_t slot = 0;  // of the stage at hand
  auto next_slot = [&](uint32_t s) { return s + T::XSLOT == WG_XSLOTS * T::XSLOT ? 0u : s + T::XSLOT; };
  auto read_pair = [&](int q, int half, uint32_t from) __attribute__((always_inline)) {  // one fragment of pair q of a stage
    const int i = 2 * (q % PM) + half;
    a[2 * (q % 4) + half] = read_a(i, from, q / PM % 2);
  };
  const std::integral_constant<int, 0> K0;
  const std::integral_constant<int, 1> K1;
  // The matrix pipe takes an MFMA every 16 cycles, two vector instructions of the SIMD fit in between and a third makes it wait
  // (measured: 7.2, 7.3, 7.5, 9.1, 11.1 ns per MFMA with 0 .. 4 of them).  So the decode is dealt out evenly: the instructions
  // whose turn it is behind MFMA `at` of a k-step, counted from MFMA FROM on.
  auto deal = [&](int at, auto FROM, auto KS) __attribute__((always_inline)) {
    constexpr int from = decltype(FROM)::value, slots = MT * NT - from - 2, ops = OPS * NT;  // (the last MFMAs are two wait states)
    const int q = at - from;
    if (q < 0 || q >= slots) return;
#pragma unroll
    for (int o = (q * ops + slots - 1) / slots; o < ((q + 1) * ops + slots - 1) / slots; o++) decode_op(o % OPS, o / OPS, KS);
  };

  constexpr int WGRP = WL + SL;
  constexpr int BAR = 2 * PM - 2;  // pair of a stage in front of which its barrier stands, two pairs behind its last fragment read
  aim_w(0);
  load_all(0, WGRP, WGRP);
  aim_w(1);
  load_all(0, WGRP, WGRP);
  aim_x(0, 0);
  load_all(0, XL, 0);
  aim_x(1, T::XSLOT);
  load_all(0, XL, 0);
  wide_barrier<XL>();
  aim_x(2, 2 * T::XSLOT);
  load_all(0, 4, 0);
  read_w(0, 0);
  read_s(0);
  offsets(0);
#pragma unroll
  for (int q = 0; q < AHEAD; q++) {
    read_pair(q, 0, 0);
    read_pair(q, 1, 0);
  }
#pragma unroll
  for (int o = 0; o < OPS * NT; o++) decode_op(o % OPS, o / OPS, K0);
  asm volatile("s_nop 3" ::: "memory");  // vector writes in front of an MFMA that reads them

  // A pair of row tiles of a stage: its MFMAs and what is issued between them.  The group of loads that leaves behind a stage's
  // barrier goes one to a row tile, through the rest of the stage and into the next one (LG: the group left by the stage before).
  auto pair = [&](auto Q, auto H2, int kt, uint32_t ns) __attribute__((always_inline)) {
    constexpr int q = decltype(Q)::value, h2 = decltype(H2)::value, step = q / PM;
    constexpr bool behind = q >= BAR;  // the barrier
    constexpr int W = (behind ? h2 : 1 - h2) == 0 ? WGRP : 0, l0 = behind ? 2 * (q - BAR) : 4 + 2 * q;
    if constexpr (q == BAR) {
      // the next stage: behind its activations in this wave's queue are those of the stage after it, and in front of an even
      // stage the weights requested with those; then every wave is done with the stage at hand
      if constexpr (h2 == 0) wide_barrier<XL>();
      else wide_barrier<XL + WGRP>();
      // every wave is done with the stage at hand: its slot takes the third stage from here (and behind a tile's first stage,
      // which ends with the last words of the tile in registers, the weight slot takes the tile after next)
      if constexpr (h2 == 0) aim_w(kt + 2);
      aim_x(2 * kt + h2 + 3, slot);
    }
    asm volatile("" : "+v"(a[2 * (q % 4)]), "+v"(a[2 * (q % 4) + 1]));  // one wait for both
#pragma unroll
    for (int t = 0; t < 2 * NT; t++) {
      const int i = 2 * (q % PM) + t / NT, j = t % NT, l = l0 + t / NT;
      const int jj = BACK && i % 2 ? NT - 1 - j : j;  // there and back: from one MFMA to the next only one operand changes
      if (j == 1 && l < W + XL) load_to(l, W);
      mfma(i, jj, b[step][jj]);
      if (j == 1 && l < W + XL) load(l, W);
      constexpr int ks = step == 0 ? 2 * h2 + 1 : (h2 == 0 ? 2 : 0);  // whose weights are decoded meanwhile
      // (the second step waits for the words and scales it decodes)
      deal(i * NT + j, std::integral_constant<int, step == 0 ? 0 : (h2 == 0 ? 4 : 8)>{}, std::integral_constant<int, ks>{});
      if (q + AHEAD < 2 * PM) {
        if (j == 0) read_pair(q + AHEAD, t / NT, slot);
      } else if (q == BAR) {
        if (j < 2) read_pair(j, t / NT, ns);  // pairs 0 and 1 of the next stage
      } else if (q > BAR) {
        if (j == 0) read_pair(2, t / NT, ns);
      }
    }
  };
  auto pairs = [&](auto H2, auto FROM, auto &self, int kt, uint32_t ns, auto TO) __attribute__((always_inline)) -> void {
    constexpr int q = decltype(FROM)::value, to = decltype(TO)::value;
    if constexpr (q < to) {
      pair(FROM, H2, kt, ns);
      self(H2, std::integral_constant<int, q + 1>{}, self, kt, ns, TO);
    }
  };
  const std::integral_constant<int, PM> KPM;
  const std::integral_constant<int, 2 * PM> KEND;
  auto first_step = [&](auto H2, int kt) __attribute__((always_inline)) {
    constexpr int h2 = decltype(H2)::value;
    if (GM == GM32) offsets(2 * h2 + 1);
    pairs(H2, K0, pairs, kt, 0u, KPM);
    read_w(kt + h2, h2 ^ 1);  // (the next tile's words have landed: their loads are older than this stage's activations)
  };
  auto second_step = [&](auto H2, int kt) __attribute__((always_inline)) {
    constexpr int h2 = decltype(H2)::value;
    const uint32_t ns = next_slot(slot);
    if (h2 == 1) read_s(kt + 1);
    offsets(2 - 2 * h2);
    pairs(H2, KPM, pairs, kt, ns, KEND);
    slot = ns;
  };
  const int whole = stages >> 1;
  for (int kt = 0; kt < whole; kt++) {
    first_step(K0, kt);
    second_step(K0, kt);
    first_step(K1, kt);
    second_step(K1, kt);
  }
  if (stages & 1) {  // a K that ends in the middle of 128
    first_step(K0, whole);
#pragma unroll
    for (int q = PM; q < 2 * PM; q++) {
      if (q + AHEAD < 2 * PM) {
        read_pair(q + AHEAD, 0, slot);
        read_pair(q + AHEAD, 1, slot);
      }
#pragma unroll
      for (int t = 0; t < 2 * NT; t++) mfma(2 * (q - PM) + t / NT, t % NT, b[1][t % NT]);
    }
  }
  // nothing is in flight to the slots any more, and the last MFMAs have written
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier\n\ts_nop 15\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) asm volatile("" : "+a"(acc[i][j]));

  // ---- the tile leaves through LDS as whole rows, 16 bytes per lane whatever the rows' alignment (global stores need none), in few
  // instructions: with one wave per SIMD their number is the time (a row at a time by each wave, with an address and a test per
  // store: 26 000 cycles for a tile of fp16, 71 000 where rows end off a vector)
  float rs[MT];
#pragma unroll
  for (int i = 0; i < MT; i++) rs[i] = 1.0f;
  if (p.row_scale) {
#pragma unroll
    for (int i = 0; i < MT; i++) rs[i] = p.row_scale[min(m0 + 16 * i + r, p.m - 1)];
  }
  auto leave = [&](auto EPI, auto DTYPE) __attribute__((always_inline)) {
    constexpr int epi = decltype(EPI)::value, dtype = decltype(DTYPE)::value, OB = dtype == YSCV_HIP_F32 ? 4 : 2, EPC = 16 / OB;
    constexpr int OCOLS = epi == EPI_SWIGLU ? T::BN / 2 : T::BN, PITCH = OCOLS * OB + 16, CPR = OCOLS / EPC;
    constexpr int PASSES = T::BM * PITCH <= T::LDS ? 1 : 2, ROWS = T::BM / PASSES;
    static_assert(ROWS * PITCH <= T::LDS, "a pass fits the LDS of the main loop");
    constexpr int SLOTS = CPR > 32 ? 64 : (CPR > 16 ? 32 : 16), STEP = WG_THREADS / SLOTS;  // chunks of a row, rows per instruction
    typedef uint32_t chunk_t __attribute__((ext_vector_type(4)));
    typedef chunk_t loose_t __attribute__((aligned(2)));
    typedef float4_t loose4_t __attribute__((aligned(4)));
    int me = tid;
    asm volatile("" : "+v"(me));  // (or the offsets of all seven forms would be worked out side by side)
    const int ch = me % SLOTS, rr = me / SLOTS, r = me & 15, c = me >> 4 & 3;
    const int ldo = epi == EPI_SWIGLU ? p.ldy >> 1 : p.ldy, oc0 = epi == EPI_SWIGLU ? n0 >> 1 : n0;
    const int left = min((epi == EPI_SWIGLU ? p.n >> 1 : p.n) - oc0, OCOLS) - ch * EPC;  // columns from this lane's chunk on
    const uint32_t off = (uint32_t)(rr * ldo + ch * EPC) * OB;
#pragma unroll
    for (int pass = 0; pass < PASSES; pass++) {
      if (pass > 0) __syncthreads();  // (in front of the first one, every wave is behind the main loop)
#pragma unroll
      for (int i = 0; i < MT / PASSES; i++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const float4_t v = acc[pass * (MT / PASSES) + i][j] * rs[pass * (MT / PASSES) + i];
          uint8_t *dst = wide_lds + (16 * i + r) * PITCH;
          const int col = 16 * (first + j) + 4 * c;
          if constexpr (epi == EPI_SWIGLU) {  // columns 4 c .. 4 c + 3 are gate, up, gate, up of two channels
            const float y0 = silu(v[0]) * v[1], y1 = silu(v[2]) * v[3];
            if constexpr (OB == 4) *reinterpret_cast<float2 *>(dst + col / 2 * OB) = float2{y0, y1};
            else {
              store_out(dst, col / 2, y0, dtype);
              store_out(dst, col / 2 + 1, y1, dtype);
            }
          } else if constexpr (OB == 4) {
            *reinterpret_cast<float4_t *>(dst + col * OB) = v;
          } else {
            store_cols4(dst, dtype, EPI_STORE, 0, 1 << 30, 0, col, true, v);
          }
        }
      __syncthreads();
      const int row0 = m0 + pass * ROWS, rows_left = min(p.m - row0, ROWS);
      char *base = reinterpret_cast<char *>(p.y) + (((size_t)part * p.m + row0) * ldo + oc0) * OB;
      const size_t stride = (size_t)STEP * ldo * OB;
      const uint8_t *src = wide_lds + rr * PITCH + ch * 16;
      constexpr int BATCH = ROWS / STEP < 8 ? ROWS / STEP : 8;
      int it = 0;
      if (left >= EPC) {
        for (; (it + BATCH) * STEP <= rows_left; it += BATCH) {
          chunk_t v[BATCH];
          float4_t old[epi == EPI_ADD_F32 ? BATCH : 1];
#pragma unroll
          for (int e = 0; e < BATCH; e++) {
            v[e] = *reinterpret_cast<const chunk_t *>(src + (it + e) * STEP * PITCH);
            if constexpr (epi == EPI_ADD_F32) old[e] = *reinterpret_cast<const loose4_t *>(base + e * stride + off);
          }
#pragma unroll
          for (int e = 0; e < BATCH; e++) {
            if constexpr (epi == EPI_ADD_F32) *reinterpret_cast<loose4_t *>(base + off) = old[e] + __builtin_bit_cast(float4_t, v[e]);
            else *reinterpret_cast<loose_t *>(base + off) = v[e];
            base += stride;
          }
        }
      }
      // the rows behind the last whole batch, and a chunk that the last column cuts
      if (left > 0) {
        const int from = left >= EPC ? it : 0;
        char *at = reinterpret_cast<char *>(p.y) + (((size_t)part * p.m + row0) * ldo + oc0) * OB + (size_t)from * stride + off;
        for (int q = from; q * STEP + rr < rows_left; q++, at += stride) {
          const uint8_t *s1 = src + q * STEP * PITCH;
          for (int e = 0; e < min(left, EPC); e++) {
            if constexpr (epi == EPI_ADD_F32) reinterpret_cast<float *>(at)[e] += reinterpret_cast<const float *>(s1)[e];
            else if constexpr (OB == 4) reinterpret_cast<float *>(at)[e] = reinterpret_cast<const float *>(s1)[e];
            else reinterpret_cast<uint16_t *>(at)[e] = reinterpret_cast<const uint16_t *>(s1)[e];
          }
        }
      }
    }
  };
  const std::integral_constant<int, YSCV_HIP_F32> F32;
  const std::integral_constant<int, YSCV_HIP_F16> F16;
  const std::integral_constant<int, YSCV_HIP_BF16> BF16;
  const std::integral_constant<int, EPI_STORE> STORE;
  const std::integral_constant<int, EPI_SWIGLU> SWIGLU;
  if (p.epi == EPI_ADD_F32) leave(std::integral_constant<int, EPI_ADD_F32>{}, F32);
  else if (p.epi == EPI_SWIGLU && p.y_dtype == YSCV_HIP_F16) leave(SWIGLU, F16);
  else if (p.epi == EPI_SWIGLU && p.y_dtype == YSCV_HIP_F32) leave(SWIGLU, F32);
  else if (p.epi == EPI_SWIGLU) leave(SWIGLU, BF16);
  else if (p.y_dtype == YSCV_HIP_F16) leave(STORE, F16);
  else if (p.y_dtype == YSCV_HIP_F32) leave(STORE, F32);
  else leave(STORE, BF16);
}

template <int GM, bool SF16, bool HAS_ZP, int MT, int NT>
int32_t wide_launch_one(WideArgs a, hipStream_t s) {
  using T = WideTile<GM, SF16, HAS_ZP, MT, NT>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kern = int4_gemm_wide_kernel<GM, SF16, HAS_ZP, MT, NT>;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS); });
  if (attr_err != hipSuccess) return set_error(YSCV_HIP_ERR_DEVICE, "cannot reserve %d bytes of LDS: %s", T::LDS, hipGetErrorString(attr_err));
  a.tiles_m = (a.m + T::BM - 1) / T::BM;
  a.tiles_n = (a.n - a.col0 + T::BN - 1) / T::BN;
  hipLaunchKernelGGL(kern, dim3((unsigned)((a.tiles_m * a.tiles_n * a.parts + 7) / 8 * 8)), dim3(WG_THREADS), T::LDS, s, a);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

template <int GM, bool SF16, bool HAS_ZP>
int32_t wide_launch_tile(const WideArgs &a, int tile, hipStream_t s) {
  switch (tile) {
    case WIDE_256x256: return wide_launch_one<GM, SF16, HAS_ZP, 16, 4>(a, s);
    case WIDE_256x192: return wide_launch_one<GM, SF16, HAS_ZP, 16, 3>(a, s);
    case WIDE_128x256: return wide_launch_one<GM, SF16, HAS_ZP, 8, 4>(a, s);
    default: return wide_launch_one<GM, SF16, HAS_ZP, 8, 3>(a, s);
  }
}
template <int GM, bool SF16>
int32_t wide_launch_zp(const WideArgs &a, int tile, hipStream_t s) {
  return a.tzps ? wide_launch_tile<GM, SF16, true>(a, tile, s) : wide_launch_tile<GM, SF16, false>(a, tile, s);
}

}  // namespace

int32_t launch_int4_gemm_wide(const yscv_hip_int4_weight *w, const _Float16 *xh, const float *row_scale, size_t ldx, void *y, int y_dtype,
                              size_t m, size_t col0, size_t col1, int tile, hipStream_t s, int epi, int parts, int kt_per, float *partial) {
  WideArgs a;
  a.tiles = w->tiles;
  a.tscales = w->tscales;
  a.tzps = w->has_zp ? w->tzps : nullptr;
  a.xh = xh;
  a.row_scale = row_scale;
  a.y = parts > 1 ? partial : y;
  a.m = (int)m;
  a.n = (int)col1;
  a.col0 = (int)col0;
  a.ldy = (int)w->n;
  a.nt = (int)w->nt;
  a.kt = (int)w->kt;
  a.ktp = (int)w->ktp;
  a.chunks = (int)w->chunks;
  a.chunk_div = w->gm == GM128 ? (int)(w->g / 128) : 1;
  a.ldx = (int)ldx;
  a.stages = (int)ceil_div(w->k, (size_t)64);
  a.y_dtype = (int16_t)(parts > 1 ? YSCV_HIP_F32 : y_dtype);
  a.epi = (int16_t)(parts > 1 ? EPI_STORE : epi);
  a.parts = parts;
  a.kt_per = parts > 1 ? kt_per : (int)w->kt;
  const bool sf16 = w->scale_dtype == YSCV_HIP_F16;
  auto launch = [&] {
    if (w->gm == GM32) return sf16 ? wide_launch_zp<GM32, true>(a, tile, s) : wide_launch_zp<GM32, false>(a, tile, s);
    if (w->gm == GM64) return sf16 ? wide_launch_zp<GM64, true>(a, tile, s) : wide_launch_zp<GM64, false>(a, tile, s);
    return sf16 ? wide_launch_zp<GM128, true>(a, tile, s) : wide_launch_zp<GM128, false>(a, tile, s);
  };
  YSCV_TRY(launch());
  return parts > 1 ? launch_int4_partial_sum(partial, parts, (int)m, (int)w->n, y, y_dtype, epi, s) : YSCV_HIP_OK;
}

}  // namespace yscv
