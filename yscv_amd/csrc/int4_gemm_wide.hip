// Packed-int4 matmul for many rows (fp16-prepared activations): y[m][n] = sum_k x[m][k] * W[n][k] in tiles of 256 x 256.
// Replaces packed_int4_gemm_dispatch (crates/yscv-kernels/src/ops/int4_matmul.rs:548-605) where such tiles fill the CUs.
//
// The LDS-ring GEMM's tiles are bound by LDS bandwidth: per 32 k its 256 x 128 tile moves 72 KB through LDS (activations and
// decoded weights in, fragments out) in the 512 cycles its MFMAs take, 144 bytes per cycle where LDS moves 128.  Here only
// packed weights pass through LDS: a wave owns 128 rows x 64 columns, reads a weight word once per 128 k and decodes it in
// registers, where it feeds eight MFMAs.  Eight waves (2 x 4) make a tile of 256 x 256, two waves per SIMD: per 32 k 16 KB of
// activations and 4 KB of packed weights in, 64 + 8 KB of fragments out, in 1024 cycles of MFMAs: 90 bytes per cycle.  The
// decode (about 60 vector instructions per k-step and wave) is issued between the wave's MFMAs and those of the other wave.
// Everything arrives by LDS-direct loads whose count each wave knows: activations in three slots of 64 k (XOR-swizzled as in
// the LDS-ring GEMM), weights and scales in two of 128 k.  One barrier per 64 k; half a k-step's MFMAs are issued behind it
// and cover the first fragment reads of the next stage.
// The group scale is folded into fp16 weights as in the LDS-ring GEMM, products are added in the same order: same results.
// us of the whole op, planned without -> with this kernel (m x n x k, fp16 rows), in bursts of six calls 50 ms apart | replayed
// for 1.5 s, the clock settled: 2048 x 8192 x 4096 137 -> 120 | 134 -> 114, 2048 x 14336 x 4096 248 -> 228 | 240 -> 210, 2048 x
// 28672 x 4096 525 -> 472 | 456 -> 408, 700 x 24000 x 2048 95 -> 84 | 90 -> 79.  With zero points (two more instructions per
// pair of weights, and the bf16 rows prepared first: 9 us of it) the decode takes back most of it: 2048 x 14336 x 4096 in
// 128-groups 254 -> 266 | 242 -> 233: slower while the clock is still coming up behind an idle stretch, faster once it is there.
// Tiles of 14 and 12 column blocks (224, 192 columns) where they fill the CUs in whole rounds and 256 columns leave the last
// one short: 2048 x 7168 x 4096 101 us (a round of 256 columns 113), 2048 x 6144 x 4096 105 -> 91, with zero points 103 -> 96;
// 2048 x 14336 x 4096 with zero points 220 -> 207, without 207 -> 202, 2048 x 28672 x 4096 no change (settled clock: CUs left
// idle by a short round leave the others a higher clock, so a round saved is worth less than its share).
// A stage takes 1.43 us (1.09 without the decode) where its MFMAs take 1.05 at the rate a registers-only loop reaches.
#include <mutex>
#include <type_traits>

#include "int4_common.hpp"
#include "kernels.hpp"

namespace yscv {

namespace {

constexpr int WG_MT = 8, WG_NT = 4, WG_WM = 2, WG_WN = 4;  // MFMA tiles of a wave (the widest tile), waves of a workgroup
constexpr int WG_BM = 16 * WG_MT * WG_WM, WG_BLOCKS = WG_NT * WG_WN, WG_THREADS = 64 * WG_WM * WG_WN;
constexpr int WG_XSLOT = WG_BM * 128, WG_XSLOTS = 3;  // activations of 64 k
constexpr int WG_WSLOT = WG_BLOCKS * 1024;            // packed weights of 128 k, two slots
constexpr int WG_RS = 16 * WG_NT + 4;                 // floats per row of the epilogue's LDS tile
constexpr int WG_ERED = 8 * WG_MT * WG_RS * 4;        // a wave's LDS there: half of its rows

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
  int y_dtype, epi;
};

template <int GM, bool SF16, bool HAS_ZP>
struct WideScale {
  static constexpr int SPT = GM == GM32 ? 4 : (GM == GM64 ? 2 : 1);
  static constexpr int BLOCK = 16 * SPT * (SF16 ? 2 : 4);        // bytes of one 16-column block and 128 k
  static constexpr int LOADS = (WG_NT * BLOCK + 255) / 256;      // 4-byte-per-lane loads of a wave's blocks
  static constexpr int ZBLOCK = 16 * SPT;
  static constexpr int ZLOADS = HAS_ZP ? (WG_NT * ZBLOCK + 255) / 256 : 0;
  static constexpr int BYTES = (LOADS + ZLOADS) * 256;           // LDS per wave and slot
  typedef typename std::conditional<SF16, _Float16, float>::type elem_t;
  typedef elem_t vec_t __attribute__((ext_vector_type(SPT)));
};

template <int N>
__device__ __forceinline__ void wide_barrier() {
  // this wave's loads of the stage have landed and its fragment reads of the last one have returned; then everyone's
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// One wave's share of a tile: 128 rows of the half wave & 1, the NT column blocks from block OFF + NT (wave / 2) of the tile's on.
template <int GM, bool SF16, bool HAS_ZP, int NT, int OFF>
__device__ __forceinline__ void wide_wave(const WideArgs &p, int m0, int n0) {
  using S = WideScale<GM, SF16, HAS_ZP>;
  constexpr int MT = WG_MT, XL = WG_BM / 64, WL = WG_BLOCKS / 8, SL = S::LOADS + S::ZLOADS;  // loads per wave
  extern __shared__ __attribute__((aligned(1024))) uint8_t wide_lds[];
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // (offsets shared by the two forms of a 14-block tile would be kept beside the accumulators)
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4, wm = wave & 1, first = OFF + NT * (wave >> 1), nb0 = n0 / 16;
  NibbleConsts nc;
  nc.init();

  const uint32_t lds0 = (uint32_t)(size_t)wide_lds;
  uint8_t *w_lds = wide_lds + WG_XSLOTS * WG_XSLOT;
  uint8_t *s_lds = w_lds + 2 * WG_WSLOT + wave * 2 * S::BYTES;
  const uint32_t w_off = lds0 + WG_XSLOTS * WG_XSLOT, s_off = w_off + 2 * WG_WSLOT + (uint32_t)(wave * 2 * S::BYTES);

  // ---- load addresses: uniform base + 32-bit lane offsets.  x piece q of a stage: rows 8 q .. 8 q + 7, 128 bytes each
  uint32_t xoff[XL];
#pragma unroll
  for (int u = 0; u < XL; u++) {
    const int q = wave * XL + u, row8 = lane >> 3, row = min(m0 + 8 * q + row8, p.m - 1);
    xoff[u] = (uint32_t)(((size_t)row * p.ldx + ((lane & 7) ^ (4 * (q & 1) + (row8 >> 1))) * 8) * 2);
  }
  auto load_x = [&](int st, uint32_t slot) {
    const char *base = reinterpret_cast<const char *>(p.xh) + (size_t)min(st, p.stages - 1) * 128;
#pragma unroll
    for (int u = 0; u < XL; u++)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds0 + slot + (uint32_t)((wave * XL + u) * 1024)), "v"(xoff[u]), "s"(base) : "memory");
  };
  const uint32_t woff = lane * 16;
  // scales (zero points) of the wave's four blocks: byte 4 lane + 256 u of them, blocks past the matrix repeat the last one
  uint32_t scoff[S::LOADS], zpoff[S::ZLOADS > 0 ? S::ZLOADS : 1];
#pragma unroll
  for (int u = 0; u < S::LOADS; u++) {
    const int byte = (u * 256 + lane * 4) % (NT * S::BLOCK), blk = min(nb0 + first + byte / S::BLOCK, p.nt - 1);
    scoff[u] = (uint32_t)blk * (uint32_t)(p.chunks * S::BLOCK) + (uint32_t)(byte % S::BLOCK);
  }
#pragma unroll
  for (int u = 0; u < S::ZLOADS; u++) {
    const int byte = (u * 256 + lane * 4) % (NT * S::ZBLOCK), blk = min(nb0 + first + byte / S::ZBLOCK, p.nt - 1);
    zpoff[u] = (uint32_t)blk * (uint32_t)(p.chunks * S::ZBLOCK) + (uint32_t)(byte % S::ZBLOCK);
  }
  auto load_w = [&](int kt) {
    const uint32_t slot = (uint32_t)(kt & 1);
    kt = min(kt, p.kt - 1);
    const int chunk = GM == GM128 ? kt / p.chunk_div : kt;
#pragma unroll
    for (int u = 0; u < WL; u++) {
      const int blk = wave * WL + u;
      const uint8_t *base = p.tiles + ((size_t)min(nb0 + blk, p.nt - 1) * p.ktp + kt) * kTileBytes;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(w_off + slot * WG_WSLOT + (uint32_t)(blk * 1024)), "v"(woff), "s"(base) : "memory");
    }
    const uint8_t *sbase = reinterpret_cast<const uint8_t *>(p.tscales) + (size_t)chunk * S::BLOCK;
#pragma unroll
    for (int u = 0; u < S::LOADS; u++)
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(s_off + slot * S::BYTES + u * 256), "v"(scoff[u]), "s"(sbase) : "memory");
    if constexpr (HAS_ZP) {
      const uint8_t *zbase = p.tzps + (size_t)chunk * S::ZBLOCK;
#pragma unroll
      for (int u = 0; u < S::ZLOADS; u++)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(s_off + slot * S::BYTES + (S::LOADS + u) * 256), "v"(zpoff[u]), "s"(zbase) : "memory");
    }
  };

  // ---- LDS -> registers
  typedef uint32_t word_pair_t __attribute__((ext_vector_type(2)));
  word_pair_t wq[NT];  // of the two k-steps of a stage
  typedef _Float16 scale_t __attribute__((ext_vector_type(S::SPT == 1 ? 2 : S::SPT)));
  scale_t sv[NT];  // (f32 scales are rounded as the weights are)
  uint32_t zv[HAS_ZP ? NT : 1];
  auto read_w = [&](int kt, int half) {
    const uint8_t *src = w_lds + (kt & 1) * WG_WSLOT + first * 1024 + lane * 16 + half * 8;
#pragma unroll
    for (int j = 0; j < NT; j++) wq[j] = *reinterpret_cast<const word_pair_t *>(src + j * 1024);
    if (half == 1) return;
    const uint8_t *ss = s_lds + (kt & 1) * S::BYTES;
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const typename S::vec_t v = *reinterpret_cast<const typename S::vec_t *>(ss + j * S::BLOCK + r * (S::BLOCK / 16));
#pragma unroll
      for (int e = 0; e < S::SPT; e++) sv[j][e] = (_Float16)v[e];
      if constexpr (HAS_ZP) {
        const uint8_t *z = ss + S::LOADS * 256 + j * S::ZBLOCK + r * S::SPT;
        if constexpr (GM == GM32) zv[j] = *reinterpret_cast<const uint32_t *>(z);
        else if constexpr (GM == GM64) zv[j] = *reinterpret_cast<const uint16_t *>(z);
        else zv[j] = *z;
      }
    }
  };
  auto decode = [&](int j, int ks) {
    const int e = GM == GM32 ? ks : (GM == GM64 ? ks >> 1 : 0);
    // (opaque: the compiler would keep splats and constants of all blocks in registers from one k-step to the next)
    asm volatile("" : "+v"(sv[j]));
    const _Float16 s = sv[j][e];
    _Float16 c1v = (_Float16)(-1032.0f), c2v = (_Float16)(-72.0f);
    if constexpr (HAS_ZP) {
      asm volatile("" : "+v"(zv[j]));
      const _Float16 z = (_Float16)(float)((zv[j] >> (8 * e)) & 0xFFu);
      c1v = (_Float16)(-1024.0f) - z;
      c2v = (_Float16)(-64.0f) - z;
    }
    return decode8_exact(wq[j][ks & 1], nc, half2_t{c1v, c1v}, half2_t{c2v, c2v}) * half8_t{s, s, s, s, s, s, s, s};
  };
  const uint32_t g = 4u * (r >> 3) + ((r & 7) >> 1);
  const uint32_t rd0 = (uint32_t)(wm * MT * 2048) + (uint32_t)((r >> 3) * 1024) + (((r & 7) * 8 + (c ^ g)) * 16);  // k-step 1: ^ 64
  auto read_a = [&](int i, uint32_t slot, int h) { return *reinterpret_cast<const half8_t *>(wide_lds + slot + i * 2048 + (rd0 ^ (64u * h))); };

  float4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int AD = MT / 2;  // fragments of x in registers: the MFMAs of AD row tiles cover a read
  half8_t a[AD], b[2][NT];
  auto mfmas = [&](int i, const half8_t (&bb)[NT]) {
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bb[j], a[i % AD], acc[i][j], 0, 0, 0);
  };

  load_w(0);
  load_w(1);
  load_x(0, 0);
  load_x(1, WG_XSLOT);
  wide_barrier<XL>();
  load_x(2, 2 * WG_XSLOT);
  read_w(0, 0);
#pragma unroll
  for (int j = 0; j < NT; j++) b[0][j] = decode(j, 0);
#pragma unroll
  for (int i = 0; i < AD; i++) a[i] = read_a(i, 0, 0);

  uint32_t slot = 0;  // of the stage at hand
  auto next_slot = [&](uint32_t s) { return s + WG_XSLOT == WG_XSLOTS * WG_XSLOT ? 0u : s + WG_XSLOT; };
  // first k-step of a stage; the second one's weights are decoded between its MFMAs
  auto first_step = [&](auto H2) {
    constexpr int h2 = decltype(H2)::value;
#pragma unroll
    for (int i = 0; i < MT; i++) {
      mfmas(i, b[0]);
      a[i % AD] = i < MT - AD ? read_a(i + AD, slot, 0) : read_a(i + AD - MT, slot, 1);
      if ((i & 1) == 0 && i / 2 < NT) b[1][i / 2] = decode(i / 2, 2 * h2 + 1);
      __builtin_amdgcn_sched_barrier(0);  // (left alone the scheduler decodes far ahead and runs out of registers)
    }
  };
  // second k-step, and the step to the next stage behind its last fragment read
  auto second_step = [&](int kt, auto H2) {
    constexpr int h2 = decltype(H2)::value;
    read_w(kt + h2, h2 ^ 1);  // (the next tile's words have landed: their loads are older than this stage's activations)
#pragma unroll
    for (int i = 0; i < MT - AD; i++) {
      mfmas(i, b[1]);
      a[i % AD] = read_a(i + AD, slot, 1);
      if (i >= 2) b[0][i - 2] = decode(i - 2, h2 == 0 ? 2 : 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    const uint32_t ns = next_slot(slot);
    // the next stage: behind its activations in this wave's queue are those of the stage after it, and in front of an even
    // stage the weights requested with those
    if (h2 == 0) wide_barrier<XL>();
    else wide_barrier<XL + WL + SL>();
    // every wave is done with the stage at hand: its slot takes the third stage from here (and behind a tile's first stage,
    // which ends with the last words of the tile in registers, the weight slot takes the tile after next)
    if (h2 == 0) load_w(kt + 2);
    load_x(2 * kt + h2 + 3, slot);
#pragma unroll
    for (int i = MT - AD; i < MT; i++) {
      mfmas(i, b[1]);
      a[i % AD] = read_a(i + AD - MT, ns, 0);
      if (i - 2 < NT) b[0][i - 2] = decode(i - 2, h2 == 0 ? 2 : 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    slot = ns;
  };
  const std::integral_constant<int, 0> H0;
  const std::integral_constant<int, 1> H1;
  const int whole = p.stages >> 1;
  for (int kt = 0; kt < whole; kt++) {
    first_step(H0);
    second_step(kt, H0);
    first_step(H1);
    second_step(kt, H1);
  }
  if (p.stages & 1) {  // a K that ends in the middle of 128
    first_step(H0);
#pragma unroll
    for (int i = 0; i < MT; i++) {
      mfmas(i, b[1]);
      if (i < MT - AD) a[i % AD] = read_a(i + AD, slot, 1);
    }
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // nothing is in flight to the slots any more

  // ---- a wave's tile leaves in two halves of 64 rows through LDS of its own, as whole lines of 64 columns (a rolled loop: one
  // copy of the store code per half, not one per MFMA tile)
  float *red = reinterpret_cast<float *>(wide_lds) + wave * WG_ERED / 4;
  const bool vec = (p.ldy & 3) == 0;
  const int col = n0 + first * 16 + 4 * r;
#pragma unroll
  for (int i0 = 0; i0 < MT; i0 += MT / 2) {
#pragma unroll
    for (int i = 0; i < MT / 2; i++)
#pragma unroll
      for (int j = 0; j < NT; j++) *reinterpret_cast<float4_t *>(red + (16 * i + r) * WG_RS + 16 * j + 4 * c) = acc[i0 + i][j];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int row0 = m0 + (wm * MT + i0) * 16 + c;
#pragma unroll 4
    for (int q = 0; q < 2 * MT; q++) {
      const int row = row0 + 4 * q;
      if (row < p.m && col < p.n && r < 4 * NT) {
        float4_t v = *reinterpret_cast<const float4_t *>(red + (4 * q + c) * WG_RS + 4 * r);
        if (p.row_scale) v = v * p.row_scale[row];
        store_cols4(p.y, p.y_dtype, p.epi, p.ldy, p.n, row, col, vec, v);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// NB: column blocks of a tile, 16, 14 or 12.  Waves w and w + 4 share a SIMD: with 14 blocks the column quarters are 4, 4, 3 and
// 3 blocks wide and every SIMD has one wave of each kind.
template <int GM, bool SF16, bool HAS_ZP, int NB>
__global__ void __launch_bounds__(WG_THREADS, 2) int4_gemm_wide_kernel(WideArgs p, int tiles_m, int tiles_n) {
  // Tiles are numbered down bands of eight row tiles, column by column; an XCD (workgroup ids equal modulo 8) takes an eighth
  // of them in a row: 32 neighbours share row and column panels in its L2, and no XCD has more than its share (super-blocks of
  // 32 tiles gave four XCDs a second one at three row tiles x 85 columns: 700 x 24000 x 2048 140 us against 98)
  const int tiles = tiles_m * tiles_n, share = (tiles + 7) >> 3, t = (int)(blockIdx.x & 7) * share + (int)(blockIdx.x >> 3);
  if (t >= tiles) return;
  const int band = t / (8 * tiles_n), in_band = t - band * 8 * tiles_n, rows = min(8, tiles_m - 8 * band);
  const int tn = in_band / rows, tm = 8 * band + in_band % rows;
  const int m0 = tm * WG_BM, n0 = p.col0 + tn * 16 * NB;
  if constexpr (NB == 16) {
    wide_wave<GM, SF16, HAS_ZP, 4, 0>(p, m0, n0);
  } else if constexpr (NB == 12) {
    wide_wave<GM, SF16, HAS_ZP, 3, 0>(p, m0, n0);
  } else {
    static_assert(NB == 14, "column blocks of a tile");
    if (__builtin_amdgcn_readfirstlane(threadIdx.x) >= 256) wide_wave<GM, SF16, HAS_ZP, 3, 2>(p, m0, n0);
    else wide_wave<GM, SF16, HAS_ZP, 4, 0>(p, m0, n0);
  }
}

template <int GM, bool SF16, bool HAS_ZP, int NB>
int32_t wide_launch_one(const WideArgs &a, hipStream_t s) {
  constexpr int LOOP = WG_XSLOTS * WG_XSLOT + 2 * WG_WSLOT + 16 * WideScale<GM, SF16, HAS_ZP>::BYTES;
  constexpr int LDS = LOOP > 8 * WG_ERED ? LOOP : 8 * WG_ERED;
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kern = int4_gemm_wide_kernel<GM, SF16, HAS_ZP, NB>;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS); });
  if (attr_err != hipSuccess) return set_error(YSCV_HIP_ERR_DEVICE, "cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr_err));
  const int tiles_m = (a.m + WG_BM - 1) / WG_BM, tiles_n = (a.n - a.col0 + 16 * NB - 1) / (16 * NB);
  hipLaunchKernelGGL(kern, dim3((unsigned)((tiles_m * tiles_n + 7) / 8 * 8)), dim3(WG_THREADS), LDS, s, a, tiles_m, tiles_n);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

template <int GM, bool SF16, bool HAS_ZP>
int32_t wide_launch_nb(const WideArgs &a, int blocks, hipStream_t s) {
  // (with zero points and a scale per 32 k the 14-block form needs one register more than there are: 16 blocks then)
  if constexpr (!(GM == GM32 && HAS_ZP))
    if (blocks == 14) return wide_launch_one<GM, SF16, HAS_ZP, 14>(a, s);
  if (blocks == 12) return wide_launch_one<GM, SF16, HAS_ZP, 12>(a, s);
  return wide_launch_one<GM, SF16, HAS_ZP, 16>(a, s);
}
template <int GM, bool SF16>
int32_t wide_launch_zp(const WideArgs &a, int blocks, hipStream_t s) {
  return a.tzps ? wide_launch_nb<GM, SF16, true>(a, blocks, s) : wide_launch_nb<GM, SF16, false>(a, blocks, s);
}

}  // namespace

int32_t launch_int4_gemm_wide(const yscv_hip_int4_weight *w, const _Float16 *xh, const float *row_scale, size_t ldx, void *y, int y_dtype,
                              size_t m, size_t col0, size_t col1, int blocks, hipStream_t s, int epi) {
  WideArgs a;
  a.tiles = w->tiles;
  a.tscales = w->tscales;
  a.tzps = w->has_zp ? w->tzps : nullptr;
  a.xh = xh;
  a.row_scale = row_scale;
  a.y = y;
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
  a.y_dtype = y_dtype;
  a.epi = epi;
  const bool sf16 = w->scale_dtype == YSCV_HIP_F16;
  if (w->gm == GM32) return sf16 ? wide_launch_zp<GM32, true>(a, blocks, s) : wide_launch_zp<GM32, false>(a, blocks, s);
  if (w->gm == GM64) return sf16 ? wide_launch_zp<GM64, true>(a, blocks, s) : wide_launch_zp<GM64, false>(a, blocks, s);
  return sf16 ? wide_launch_zp<GM128, true>(a, blocks, s) : wide_launch_zp<GM128, false>(a, blocks, s);
}

}  // namespace yscv
