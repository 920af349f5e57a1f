// int8 x int8 -> int32 GEMM in tiles of 128 x 256 or 64 x 128: zero-point correction and requantising epilogue as in i8_gemm.hip.  Replaces
// int8_matmul_dispatch / int8_matmul_prepacked_dispatch (crates/yscv-kernels/src/ops/int8_matmul.rs:2407-2425) for shapes with more tiles
// than i8_ksplit.hip serves well.
//
// Four waves stand side by side in columns and each takes ALL rows of the tile, so nobody but one wave needs a block of B: B goes from
// memory to the registers of that wave (it is packed as the MFMA takes it) and only A passes through LDS.  (Waves 2 x 2 with both operands
// in LDS, four more waves to load them: 12 KB written to LDS and 24 KB read per 64 k of a 64 x 128 tile took 184 ns.)
//   64 x 128:  eight waves, two rows of four that take alternate pairs of k-steps; their sums meet in LDS at the end.  One wave per SIMD
//              is bound by the instructions it can issue (70 in a k-step, five cycles each), two fill each other's gaps.  A k-step takes
//              in its 12 KB in 128 ns (512 rows, N 4096, K 1024 8.3 us, 4096 14.4): 96 GB/s per CU with all of them at it, where loads
//              to LDS alone reach 70 .. 76 (yscv_hip_measure_fill).  The other 6.2 us are launch, first operands and what the end takes.
//   128 x 256: four waves, the accumulators in the other half of the register file.  Half the bytes per MFMA; bound by issue: a SIMD takes
//              an instruction every four cycles and an MFMA every sixteen, two more fit behind each.  So the loop is laid out by hand as in
//              int4_gemm_wide.hip: MFMAs are statements in their order, fragments of A are read a k-step ahead and made signed two row
//              tiles ahead, loads go one to an MFMA, and what only the end of K needs is left to code of its own (masks and tests in
//              the loop: 8192 x 8192, 2048 rows 125 -> 120 us; ways out of its middle, which have the accumulators copied: 136).
// A arrives by LDS-direct loads in S + 1 slots (XOR-swizzled as in i8_ksplit.hip), one barrier a stage; the compiler waits for B's, which are
// plain loads.  It does not know of A's, whose count only makes it wait for more than it must.
// us of the whole op, the kernel before -> this (m x n x k, to int32): 512 x 4096 x 4096 16.6 -> 15.1, 512 x 4096 x 1024 8.4 -> 7.7, 1024 x 2048 x
// 2048 11.0 -> 10.2, 1500 x 3000 x 5056 46.7 -> 33.9, 2048 x 4096 x 4096 45 -> 34.5, 2048 x 8192 x 8192 165 -> 120 (2.3 POP/s); requantised: 500 x 4000 x
// 4096 17.1 -> 14.4, 130 x 8192 x 8192 25 -> 20.7.
#include <mutex>
#include <type_traits>

#include "i8_common.hpp"

namespace yscv {

namespace {

// A tile of MT x 4 NT blocks of 16.  Four waves stand side by side in columns, WK such rows of waves share the K of a stage; B of S
// stages is in flight; one stage: all of K.
// A stage is KS k-steps of 64 for each of a wave's rows.
template <int MT, int NT, int WK, int S, int KS>
struct IwTile {
  static constexpr int BM = 16 * MT, BN = 64 * NT, THREADS = 256 * WK;
  static constexpr int STAGE = BM * 64 * KS * WK, SLOTS = S + 1;
  static constexpr int RS = BN + 4;  // row stride of a tile of sums in LDS, in ints (16 bytes of padding)
  static constexpr int LOOP = SLOTS * STAGE, SUMS = WK * BM * RS * 4, LDS = LOOP > SUMS ? LOOP : SUMS, ALL = LDS + 12 * BN;
  static_assert(ALL <= 160 * 1024, "LDS of a CU");
};

template <int N>
__device__ __forceinline__ void iw_barrier() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int MT, int NT, int WK, int S, int KS>
__global__ void __launch_bounds__(256 * WK, WK) i8_gemm_wide_kernel(I8Args p, int tiles_m, int tiles_n) {
  using T = IwTile<MT, NT, WK, S, KS>;
  static_assert(MT % 4 == 0 && NT >= 2 && MT >= NT && S >= 1 && S <= 4, "");
  constexpr int AL = MT / 4;  // A loads of a wave and k-step
  extern __shared__ __attribute__((aligned(1024))) uint8_t iw_lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4, wn = wave & 3, wk = wave >> 2;
  // Tiles are numbered down bands of eight row tiles, column by column; an XCD (workgroup ids equal modulo 8) takes an eighth
  // of them in a row: the neighbours that it runs together share row panels of A and column panels of B in its L2, and no
  // XCD has more than its share.
  const int tiles = tiles_m * tiles_n, share = (tiles + 7) >> 3, t = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= share || t >= tiles) return;
  const int band = t / (8 * tiles_n), in_band = t - band * 8 * tiles_n, band_rows = min(8, tiles_m - 8 * band);
  const int tn = in_band / band_rows, tm = 8 * band + in_band % band_rows;
  const int m0 = tm * T::BM, nb0 = tn * 4 * NT + wn * NT, nb_last = (p.n + 15) / 16 - 1;
  const int nst = (p.ksteps + KS * WK - 1) / (KS * WK);
  // (a single k-step is the first half of a pair at byte 0 whose second half is multiplied as zeros)
  const bool one = S == 1 && p.ksteps == 1;
  const int odd = one ? 0 : p.ksteps & 1;
  const uint32_t lds0 = (uint32_t)(size_t)iw_lds;

  // the per-column terms of the epilogue, requested ahead of the loop, wait in LDS behind the ring
  int32_t *terms = reinterpret_cast<int32_t *>(iw_lds + T::LDS);
  const int tcol = min(tn * T::BN + min(tid, T::BN - 1), p.n - 1);
  const int32_t t_sum = p.col_sum[tcol], t_corr = p.corr ? p.corr[tcol] : 0;
  const float t_comp = p.composite_v ? p.composite_v[tcol] : p.composite;

  // ---- loads.  A pair is two k-steps, 128 bytes of every row.  A: pieces [row tile][pair][half] of a stage, 1 KiB each; a wave fetches
  // those of AL row tiles and its own pairs.  Lane i of half h fetches 16-byte chunk (i & 7) ^ g of row 8 h + i / 8, g = 4 h + (i / 8) / 2, so
  // that the sixteen rows of a fragment read fall into sixteen different slots.  An odd count of k-steps: the last pair begins a
  // k-step early, and its first half, which the pair in front has had, is multiplied as zeros.  One k-step: the second half is fetched from
  // where the first one is.
  uint32_t aoff[AL][2];
#pragma unroll
  for (int i = 0; i < AL; i++)
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const int row8 = lane >> 3, row = min(m0 + 16 * (AL * wn + i) + 8 * h + row8, p.m - 1);
      aoff[i][h] = (uint32_t)row * (uint32_t)p.lda + (uint32_t)((((lane & 7) ^ (4 * h + (row8 >> 1))) & (one ? 3 : 7)) * 16);
    }
  uint32_t boff[NT];  // (column blocks past the end repeat the last one)
#pragma unroll
  for (int j = 0; j < NT; j++) boff[j] = (uint32_t)(min(nb0 + j, nb_last) - min(nb0, nb_last)) * (uint32_t)p.ksteps * 1024 + lane * 16;
  int8_t *const frag0 = const_cast<int8_t *>(p.frag) + (size_t)min(nb0, nb_last) * p.ksteps * 1024;
  const uint64_t a_ptr = (uint64_t)p.a;
  constexpr int kAll = 0x7FFFFFFF, kNone = 0, kRaw = 0x00020000;  // bytes of a buffer (none: loads read nothing), its format
  const int last_k = one ? 0 : p.ksteps - 2;
  auto pair_k = [&](int q) { return min(2 * q, last_k); };  // first k-step of pair q
  // A load l of k-step ks of a stage, whose pair begins at byte k of the rows
  const int4_t a_rsrc = {(int)(uint32_t)a_ptr, (int)(uint32_t)(a_ptr >> 32), kAll, kRaw};
  const uint32_t a_lds = lds0 + (uint32_t)(KS * (AL * wn * WK + wk) * 1024);
  auto load_a = [&](int k, int ks, int l, uint32_t slot) __attribute__((always_inline)) {
    const uint32_t to = a_lds + slot + (uint32_t)((KS * WK * l + ks) * 1024);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(aoff[l][ks & 1]), "s"(a_rsrc), "s"(k) : "memory");
  };
  int4_t b[S][KS][NT];
  auto load_b = [&](int k, int j, auto SLOT, auto STEP, int records) __attribute__((always_inline)) {  // of a pair that begins at byte k of a block
    constexpr int ks = decltype(STEP)::value;
    typedef int v4 __attribute__((ext_vector_type(4)));
    const v4 v = __builtin_amdgcn_raw_buffer_load_b128(__builtin_amdgcn_make_buffer_rsrc(frag0, 0, records, kRaw), boff[j] + (ks & 1) * 1024, k, 0);
    b[decltype(SLOT)::value][ks][j] = v;
  };

  // ---- fragments of A, one k-step ahead
  const uint32_t g = 4u * (r >> 3) + ((r & 7) >> 1);
  const uint32_t rd0 = (uint32_t)(wk * KS * 1024 + (r >> 3) * 1024) + (((r & 7) * 8 + (c ^ g)) * 16);  // odd k-steps: ^ 64
  int4_t a[2][MT];
  uint32_t rd[2] = {rd0, rd0 ^ 64u};  // (of the slot that is read)
  auto read_a = [&](int i, auto STEP) __attribute__((always_inline)) {
    constexpr int ks = decltype(STEP)::value;
    a[ks & 1][i] = *reinterpret_cast<const int4_t *>(iw_lds + rd[ks & 1] + i * 1024 * KS * WK + (ks >> 1) * 2048);
  };
  // signed bytes (a ^ 0x80 or a), 0 in the place of a k-step that there is not
  const int a_xor = p.a_xor;
  auto convert = [&](int4_t &v, int e) __attribute__((always_inline)) {
    int w = v[e];
    asm volatile("v_xor_b32 %0, %1, %0" : "+v"(w) : "s"(a_xor));
    v[e] = w;
  };
  auto convert_if = [&](int4_t &v, int e, int mask) __attribute__((always_inline)) {
    int w = v[e];
    asm volatile("v_bitop3_b32 %0, %0, %1, %2 bitop3:0x28" : "+v"(w) : "s"(a_xor), "v"(mask));  // (w ^ a_xor) & mask
    v[e] = w;
  };
  auto mask_of = [&](int st, int ks) __attribute__((always_inline)) {
    const int k = (st * WK + wk) * KS + ks;
    const int end = k == p.ksteps ? (odd ? 0 : 1) : (k >= p.ksteps - odd ? 1 : 0);
    return end - 1;
  };

  int4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = int4_t{0, 0, 0, 0};
  // one wave per SIMD: the accumulators are the other half of the register file; two: there is one half for all
  auto mfma = [&](int4_t &d, const int4_t &bb, const int4_t &aa) __attribute__((always_inline)) {
    if constexpr (WK == 1) asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+a"(d) : "v"(bb), "v"(aa));
    else asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(d) : "v"(bb), "v"(aa));
  };

  const std::integral_constant<int, 0> K0;
  const std::integral_constant<int, 1> K1;
  const std::integral_constant<int, 2 % KS> K2;
  const std::integral_constant<int, 3 % KS> K3;
  uint32_t slot = 0, fill = S * T::STAGE;  // of the stage at hand, and of the one whose A is requested meanwhile
  auto next_slot = [&](uint32_t s) { return s + T::STAGE == T::SLOTS * T::STAGE ? 0u : s + T::STAGE; };
  auto wave_pair = [&](int st, int which) { return pair_k((st * WK + wk) * (KS / 2) + which); };

  // k-step STEP of stage st, whose B is in slot U.  Meanwhile: fragments come out of LDS, those two row tiles ahead are converted, A of stage
  // st + S is requested, and B of that stage into the registers that are done.  TAIL >= 0: one of the last stages, with nothing to load
  // and k-steps that there are not.
  auto kstep = [&](int st, auto U, auto TAIL, auto STEP, int records) __attribute__((always_inline)) {
    constexpr int u = decltype(U)::value, ks = decltype(STEP)::value, rk = (ks + 1) % KS, tail = decltype(TAIL)::value;
    constexpr bool loads = tail < 0;
    if constexpr (ks == KS - 1) {
      // this wave's A of the next stage has landed: behind it came B of S - 2 stages and of this one's k-steps at least
      iw_barrier<loads ? (S - 2) * KS * NT + (KS - 1) * NT : (S - 2 - tail > 0 ? S - 2 - tail : 0) * KS * NT>();
      slot = next_slot(slot);
      rd[0] = rd0 + slot;
      rd[1] = (rd0 ^ 64u) + slot;
    }
    const int k = wave_pair(st + S, ks / 2);
    const int mask0 = loads ? -1 : mask_of(st, ks), mask1 = !loads || ks == KS - 1 ? mask_of(ks == KS - 1 ? st + 1 : st, rk) : -1;
#pragma unroll
    for (int i = 0; i < MT; i++) {
      const int cf = i / 2 * 2 + 2;  // the pair of fragments that is converted
      const bool of_next = cf >= MT;
      int4_t &c0 = a[of_next ? rk & 1 : ks & 1][cf % MT], &c1 = a[of_next ? rk & 1 : ks & 1][(cf + 1) % MT];
      if (i % 2 == 0) asm volatile("" : "+v"(c0), "+v"(c1));  // one wait for both
      const bool load = loads && i >= MT / 2 && i - MT / 2 < AL;
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const int jj = i % 2 ? NT - 1 - j : j, at = (i % 2) * NT + j;
        mfma(acc[i][jj], b[u][ks][jj], a[ks & 1][i]);
        if (j == 0 && i < MT / 2) read_a(2 * i, std::integral_constant<int, rk>{});
        if (j == 1 && i < MT / 2) read_a(2 * i + 1, std::integral_constant<int, rk>{});
        if (load && j == 0) {
          if (records != kNone) load_a(k * 64, ks, i - MT / 2, fill);  // uniform
        }
        if (loads && i == MT - 1) load_b(k * 1024, jj, U, STEP, records);
#pragma unroll
        for (int e = 0; e < 8 / (2 * NT); e++) {
          const int o = at * (8 / (2 * NT)) + e;
          if (loads && !(of_next && ks == KS - 1)) convert(o < 4 ? c0 : c1, o & 3);
          else convert_if(o < 4 ? c0 : c1, o & 3, of_next ? mask1 : mask0);
        }
      }
    }
    if constexpr (ks == KS - 1) fill = next_slot(fill);
  };
  auto stage = [&](int st, auto U, auto TAIL) __attribute__((always_inline)) {
    const int records = st + S < nst ? kAll : kNone;
    kstep(st, U, TAIL, K0, records);
    kstep(st, U, TAIL, K1, records);
    if constexpr (KS == 4) {
      kstep(st, U, TAIL, K2, records);
      kstep(st, U, TAIL, K3, records);
    }
  };

  auto first = [&](auto U, auto &self) __attribute__((always_inline)) -> void {
    constexpr int u = decltype(U)::value;
    if constexpr (u < S) {
      const int records = u < nst ? kAll : kNone, second = one ? kNone : records;
      if (u < nst) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
          for (int l = 0; l < AL; l++) load_a(wave_pair(u, ks / 2) * 64, ks, l, u * T::STAGE);
      }
#pragma unroll
      for (int j = 0; j < NT; j++) {
        load_b(wave_pair(u, 0) * 1024, j, U, K0, records);
        load_b(wave_pair(u, 0) * 1024, j, U, K1, second);
        if constexpr (KS == 4) {
          load_b(wave_pair(u, 1) * 1024, j, U, K2, records);
          load_b(wave_pair(u, 1) * 1024, j, U, K3, second);
        }
      }
      self(std::integral_constant<int, u + 1>{}, self);
    }
  };
  first(K0, first);
  // Every accumulator has its own zeros from here on, while the first operands are on their way: left to the compiler, which sees no MFMA in an
  // asm statement, it copied them from the first one's, between MFMAs that had written it.  (Behind the wait for the operands they are
  // 32 .. 128 instructions in front of the first MFMA: 197 x 3072 x 768 requantised 5.99 us, 5.97 so,
  // 2048 x 4096 x 1024 with ties to even 15.3 and 14.9.)
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) {
      if constexpr (WK == 1) asm volatile("" : "+a"(acc[i][j]));
      else asm volatile("" : "+v"(acc[i][j]));
    }
  if (tid < T::BN) {
    terms[tid] = t_sum;
    terms[T::BN + tid] = t_corr;
    terms[2 * T::BN + tid] = __float_as_int(t_comp);
  }
  iw_barrier<S * KS * NT>();
#pragma unroll
  for (int i = 0; i < MT; i++) read_a(i, K0);
  {
    const int mask = mask_of(0, 0);
#pragma unroll
    for (int e = 0; e < 4; e++) {
      convert_if(a[0][0], e, mask);
      convert_if(a[0][1], e, mask);
    }
  }
  asm volatile("s_nop 1");
  const std::integral_constant<int, -1> LOADS;
  const std::integral_constant<int, 2 % S> U2;
  const std::integral_constant<int, 3 % S> U3;
  const int full = p.ksteps / (KS * WK);  // stages without a k-step that there is not
  int st = 0;
  if constexpr (S > 1) {
    for (; st + S <= full; st += S) {
      stage(st, K0, LOADS);
      stage(st + 1, K1, LOADS);
      if constexpr (S > 2) stage(st + 2, U2, LOADS);
      if constexpr (S > 3) stage(st + 3, U3, LOADS);
    }
  }
  // no more than S stages are left and nothing to load (ways out of the loop's middle would have the accumulators copied in every round)
  if (st < nst) stage(st, K0, K0);
  if constexpr (S > 1) {
    if (st + 1 < nst) stage(st + 1, K1, K1);
  }
  if constexpr (S > 2) {
    if (st + 2 < nst) stage(st + 2, U2, U2);
  }
  if constexpr (S > 3) {
    if (st + 3 < nst) stage(st + 3, U3, U3);
  }
  // nothing is in flight to the slots any more, every wave is done with them, and the last MFMAs have written
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier\n\ts_nop 15\n\ts_nop 7" ::: "memory");
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) {
      if constexpr (WK == 1) asm volatile("" : "+a"(acc[i][j]));
      else asm volatile("" : "+v"(acc[i][j]));
    }

  // ---- the tile leaves through LDS (lane (c, r) holds C[16 i + r][16 j + 4 c + 0..3] of its wave's part) as whole rows
  int32_t *sums = reinterpret_cast<int32_t *>(iw_lds);
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) *reinterpret_cast<int4_t *>(sums + (wk * T::BM + 16 * i + r) * T::RS + (wn * NT + j) * 16 + 4 * c) = acc[i][j];
  lds_barrier();
  const float lo = (float)p.lo, hi = (float)p.hi;
  const int zp_mul = p.a_zp_dev ? 128 - (int)p.a_zp_dev[0] : p.zp_mul;
  constexpr int CPR = T::BN / 4, STEP = T::THREADS / CPR;  // pieces of four columns in a row; rows between those of a thread
  static_assert(T::THREADS % CPR == 0 && T::BM % STEP == 0, "a thread keeps its columns from row to row");
  const int col = tn * T::BN + tid % CPR * 4;
  if (col >= p.n) return;
  const int32_t *mine = terms + tid % CPR * 4;
  const int4_t corr = *reinterpret_cast<const int4_t *>(mine + T::BN);
  uint4_t zc = *reinterpret_cast<const uint4_t *>(mine) * (uint32_t)zp_mul;
  if (p.mode() == 1) zc += __builtin_bit_cast(uint4_t, corr);
  const float4_t comp = *reinterpret_cast<const float4_t *>(mine + 2 * T::BN);
  auto leave = [&](auto MODE, auto AWAY) __attribute__((always_inline)) {
    constexpr int mode = decltype(MODE)::value, OB = mode == 1 ? 1 : 4, ITERS = T::BM / STEP, BATCH = ITERS < 4 ? ITERS : 4;
    const bool whole = col + 4 <= p.n;
    typedef uint32_t loose_t __attribute__((aligned(1)));
    typedef int4_t loose4_t __attribute__((aligned(4)));
    const int rr = tid / CPR, rows = p.m - m0 - rr;  // rows from this thread's first one on
    const int32_t *src = sums + rr * T::RS + tid % CPR * 4;
    char *out = reinterpret_cast<char *>(p.out) + ((size_t)(m0 + rr) * p.n + col) * OB;
    const size_t step = (size_t)STEP * p.n * OB;
    for (int it = 0; it < ITERS && it * STEP < rows; it += BATCH) {
      int4_t v[BATCH];
#pragma unroll
      for (int x = 0; x < BATCH; x++) {
        v[x] = *reinterpret_cast<const int4_t *>(src + (it + x) * STEP * T::RS);
        if constexpr (WK == 2) v[x] += *reinterpret_cast<const int4_t *>(src + (T::BM + (it + x) * STEP) * T::RS);
      }
#pragma unroll
      for (int x = 0; x < BATCH; x++) {
        int4_t f;
        uint32_t packed = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) {
          const int32_t w = (int32_t)((uint32_t)v[x][e] + zc[e]);
          if constexpr (mode == 0) f[e] = w;
          else if constexpr (mode == 3) f[e] = __float_as_int((float)w);
          else if constexpr (mode == 2) f[e] = requant_dequant_bits(w, corr[e], comp[e], p.y_zp, p.round_mode(), lo, hi, p.dq_scale);
          else if constexpr (mode == 4) f[e] = requant_f32_bits(w, corr[e], comp[e], p.y_zp, p.round_mode(), lo, hi);
          else packed |= (uint32_t)(uint8_t)requant_int<decltype(AWAY)::value>(w, comp[e], p.y_zp, lo, hi) << (8 * e);
        }
        if ((it + x) * STEP < rows) {
          if (whole) {  // (global stores need no alignment)
            if constexpr (mode == 1) *reinterpret_cast<loose_t *>(out) = packed;
            else *reinterpret_cast<loose4_t *>(out) = f;
          } else {
            for (int e = 0; e < 4; e++) {
              if (col + e >= p.n) break;
              if constexpr (mode == 1) reinterpret_cast<uint8_t *>(out)[e] = (uint8_t)(packed >> (8 * e));
              else reinterpret_cast<int32_t *>(out)[e] = f[e];
            }
          }
        }
        out += step;
      }
    }
  };
  const std::true_type away;
  const std::false_type even;
  if (p.mode() == 0) leave(std::integral_constant<int, 0>{}, away);
  else if (p.mode() == 1 && p.round_mode() == YSCV_HIP_ROUND_HALF_AWAY) leave(std::integral_constant<int, 1>{}, away);
  else if (p.mode() == 1) leave(std::integral_constant<int, 1>{}, even);
  else if (p.mode() == 2) leave(std::integral_constant<int, 2>{}, away);
  else if (p.mode() == 3) leave(std::integral_constant<int, 3>{}, away);
  else leave(std::integral_constant<int, 4>{}, away);
}

template <int MT, int NT, int WK, int S, int KS>
int32_t iw_launch(const I8Args &p, hipStream_t s) {
  using T = IwTile<MT, NT, WK, S, KS>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kern = i8_gemm_wide_kernel<MT, NT, WK, S, KS>;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, T::ALL); });
  if (attr_err != hipSuccess) return set_error(YSCV_HIP_ERR_DEVICE, "cannot reserve %d bytes of LDS: %s", T::ALL, hipGetErrorString(attr_err));
  const int tiles_m = (p.m + T::BM - 1) / T::BM, tiles_n = (p.n + T::BN - 1) / T::BN;
  hipLaunchKernelGGL(kern, dim3((unsigned)((tiles_m * tiles_n + 7) / 8 * 8)), dim3(T::THREADS), T::ALL, s, p, tiles_m, tiles_n);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

}  // namespace

// us of a launch: whole rounds over the CUs, and a last one that fills a part of them; 64 x 128 tiles run two to a CU, which their rounds
// count as one after the other.  Fitted to 200 shapes of the same ranges as i8_ksplit.hip's (with those: the choice is 1.1 % slower than
// the fastest of all on average, 8.5 % faster than before there were these tiles).
double i8_wide_us(int tile, size_t m, size_t n, size_t ksteps, int mode, size_t cus) {
  const bool big = tile == IW_128x256;
  // A thread of the big tile requantises 128 values with nothing else to do: bytes (mode 1), dequantised (2) and f32 carriers (4), whose rounding
  // is the longer one.  us, big and small tiles: 4009 x 2880 x 512 dequantised 37.9 and 28.1, as carriers 40.6 and 28.5, 3994 x 3968 x 1344
  // 56.8 and 52.5, 59.3 and 52.4, 3058 x 5248 x 3648 88.8 and 101, 91.7 and 99.8.
  const double k = (double)ksteps, requant = !big ? 0.0 : mode == 1 ? 2.5 : mode == 2 ? 4.8 : mode == 4 ? 6.2 : 0.0;
  const double full = big ? 1.0 + 0.43 * k + requant : 0.6 + 0.155 * k, fast = big ? 0.30 * k + requant : 0.145 * k;
  // The small tile's last requantisation, and a single k-step, for which the line is too low.  With a K of 64 and 128 either is what decides against
  // i8_ksplit.hip: 509 x 880 x 64 to bytes 5.0 us and 4.2, as carriers 5.8 and 5.0, sums 4.4 and 4.1, 332 x 1200 x 128 to bytes 4.9 and 4.3.
  const double ends = big ? 6.0 : 4.1 + (mode == 1 || mode == 2 || mode == 4 ? 0.3 : 0.0) + (ksteps == 1 ? 0.2 : 0.0);
  const size_t tiles = ceil_div(m, (size_t)(big ? 128 : 64)) * ceil_div(n, (size_t)(big ? 256 : 128)), rest = tiles % cus;
  const double part = full * (double)rest / (double)cus;
  return ends + (double)(tiles / cus) * full + (rest == 0 ? 0.0 : (part > fast ? part : fast));
}

int32_t launch_i8_gemm_wide(const I8Args &p, int tile, hipStream_t s) {
  // A K of one stage has a form of its own: the others ask for as many stages as they keep in flight, whether there are any or not, and with
  // a K of 64 and tiles in several rounds i8_ksplit.hip gives a wave in four something to do.  us to int32, either of these before -> this: 20000 x
  // 64 x 64 33.5 -> 5.6, 2048 x 8192 x 64 53.7 -> 19.0, 8192 x 512 x 128 8.0 -> 7.3, 512 x 4096 x 256 5.8 -> 5.3.
  if (p.ksteps <= 4) return tile == IW_128x256 ? iw_launch<8, 4, 1, 1, 4>(p, s) : iw_launch<4, 2, 2, 1, 2>(p, s);
  return tile == IW_128x256 ? iw_launch<8, 4, 1, 2, 4>(p, s) : iw_launch<4, 2, 2, 3, 2>(p, s);
}

}  // namespace yscv
