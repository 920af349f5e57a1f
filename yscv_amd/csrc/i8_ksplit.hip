// int8 x int8 -> int32 GEMM for shapes with few tiles: y[m][n] = sum_k a[m][k] * b[k][n], zero-point correction and
// requantising epilogue fused as in i8_gemm.hip.  Replaces int8_matmul_dispatch / int8_matmul_prepacked_dispatch
// (crates/yscv-kernels/src/ops/int8_matmul.rs:2407-2425) where i8_gemm_wide.hip's tiles are fewer than the CUs.
//
// Such a call is bound by latency, not by bytes or MFMAs, and large tiles make its chain long: few workgroups, each of
// which walks the whole K stage by stage with barriers between.  Here a workgroup owns a small
// tile of 16 MT rows x 16 NT columns, its waves split the K of the tile, and every wave feeds itself through slots of LDS
// of its own, filled by LDS-direct loads (A in whole 128-byte lines, B as it is packed): no barrier until the waves' tiles
// are added (integers, so in any order) and stored as whole rows.
// A pair is two k-steps of 64, 128 bytes of every row of the tile; a wave keeps NP pairs in flight, 96 .. 144 KB per CU.
// us, tiles of 64 x 128 whose waves walk all of K -> this one (m x n x k): 1 x 4096 x 4096 17.2 -> 5.7, 16 x 256 x 8192 20.5 -> 5.9, 64 x 4096 x 4096
// 18.5 -> 6.8, 128 x 4096 x 1024 9.2 -> 5.1, 197 x 768 x 3072 12.3 -> 5.1, 256 x 4096 x 4096 16.8 -> 12.3,
// 512 x 1024 x 1024 8.5 -> 5.0, 1024 x 768 x 768 8.4 -> 6.7.  What is left is launch, first loads and the last store (3 us)
// and, with the large tiles, the fill of a CU's LDS (64 x 64 tiles, K 4096: 512 KB per CU in 9 us).
#include <mutex>

#include "i8_common.hpp"

namespace yscv {

namespace {

template <int N>
__device__ __forceinline__ void iks_wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// one column of the result through the epilogue, as the four bytes that modes 0, 2, 3 and 4 store
__device__ __forceinline__ int32_t iks_word(const I8Args &p, int32_t v, int32_t corr, float comp, float lo, float hi) {
  if (p.mode() == 0) return v;
  if (p.mode() == 3) return __float_as_int((float)v);
  if (p.mode() == 2) return requant_dequant_bits(v, corr, comp, p.y_zp, p.round_mode(), lo, hi, p.dq_scale);
  return requant_f32_bits(v, corr, comp, p.y_zp, p.round_mode(), lo, hi);
}

constexpr int iks_row_ints(int nt) { return 16 * nt + 4; }  // 16 bytes of padding: rows fall into different banks
constexpr int iks_lds(int mt, int nt, int waves, int np) {
  const int slots = waves * np * (mt + nt) * 2048, red = waves * 16 * mt * iks_row_ints(nt) * 4;
  return slots > red ? slots : red;
}

// every XCD has a CU for each row tile of its column blocks (32 CUs)
__host__ __device__ __forceinline__ bool iks_whole_columns(int tiles_m, int tiles_n) { return ((tiles_n + 7) >> 3) * tiles_m <= 32; }

template <int MT, int NT, int WAVES, int NP>
__global__ void __launch_bounds__(64 * WAVES) i8_ksplit_kernel(I8Args p, int tiles_m, int tiles_n) {
  constexpr int PAIR = (MT + NT) * 2048, LOADS = 2 * (MT + NT);  // LDS bytes and load instructions of one pair
  static_assert(NP >= 2 && NP <= 4 && (NP - 1) * LOADS < 64, "vmcnt budget");
  extern __shared__ __attribute__((aligned(1024))) uint8_t iks_ring[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  // The row tiles of one column block run on one XCD (workgroup ids equal modulo 8), so its B reaches one L2, where a workgroup to each of its CUs
  // has room for them.  Where not (few column blocks, or a count just above a multiple of eight), tiles are numbered column block by column
  // block and an XCD takes an eighth of them in a row: no XCD has more than its share, and as many tiles as CUs do run at once.
  // us, whole column blocks and even shares: 22 x 64 x 64 2.6 and 3.0, 129 x 16 x 64 2.4 and 3.0 (an XCD that has nothing to do costs nothing),
  // 40 x 48 x 4096 4.0 and 4.4; 1912 x 160 x 1664 10.1 and 5.6, 3419 x 16 x 7616 40.4 and 6.2.
  int tn, tm;
  if (iks_whole_columns(tiles_m, tiles_n)) {
    const int at = (int)(blockIdx.x >> 3) / tiles_m;
    tn = (int)(blockIdx.x & 7) + 8 * at, tm = (int)(blockIdx.x >> 3) - at * tiles_m;
    if (tn >= tiles_n) return;
  } else {
    const int tiles = tiles_m * tiles_n, t = (int)(blockIdx.x & 7) * ((tiles + 7) >> 3) + (int)(blockIdx.x >> 3);
    if (t >= tiles) return;
    tn = t / tiles_m, tm = t - tn * tiles_m;
  }
  const int m0 = tm * 16 * MT, nb0 = tn * NT, nb_total = (p.n + 15) / 16;
  const int pairs = (p.ksteps + 1) >> 1;
  const int q_lo = pairs * wave / WAVES, q_hi = pairs * (wave + 1) / WAVES;

  // The per-column terms of the epilogue: a thread stores the same four columns of every row it stores, so they are requested
  // once and ahead of the loop (197 x 3072 x 768 requantised: 8.3 us with these loads behind it, 7.0 with them here).
  constexpr int CPR = 4 * NT;  // pieces of four columns in a row of the tile
  static_assert(64 * WAVES % CPR == 0, "a thread keeps its columns from row to row");
  const int col = nb0 * 16 + tid % CPR * 4;
  int32_t zc[4], corr[4];
  float comp[4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const int cc = min(col + e, p.n - 1);
    zc[e] = p.col_sum[cc];
    corr[e] = p.corr ? p.corr[cc] : 0;
    comp[e] = p.composite_v ? p.composite_v[cc] : p.composite;
  }

  int4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = int4_t{0, 0, 0, 0};

  if (q_lo < q_hi) {  // uniform in the wave
    // A: 16 rows of a pair as two pieces of eight whole 128-byte lines.  Lane i of piece h fetches 16-byte chunk (i & 7) ^ g
    // of row i / 8, g = 4 h + (i / 8) / 2, so that the sixteen rows of a fragment read fall into sixteen different slots.
    uint32_t aoff[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int row8 = lane >> 3, row = min(m0 + 16 * i + 8 * h + row8, p.m - 1);
        aoff[i][h] = (uint32_t)row * (uint32_t)p.lda + (uint32_t)(((lane & 7) ^ (4 * h + (row8 >> 1))) * 16);
      }
    const uint32_t boff = lane * 16;
    const uint8_t *brow[NT];  // uniform; column blocks past the end repeat the last one and are not stored
#pragma unroll
    for (int j = 0; j < NT; j++) brow[j] = reinterpret_cast<const uint8_t *>(p.frag) + (size_t)min(nb0 + j, nb_total - 1) * p.ksteps * 1024;
    // an odd count of k-steps: the second half of the last pair reads the first one's data again (and is not multiplied)
    const bool half_pair = p.ksteps & 1;
    uint8_t *slots = iks_ring + wave * NP * PAIR;
    const uint32_t slots_lds = (uint32_t)(size_t)slots;
    auto load_pair = [&](int q, uint32_t slot) {
      const char *abase = reinterpret_cast<const char *>(p.a) + (size_t)q * 128;
      const uint32_t back = half_pair && q == pairs - 1 ? 64u : 0u, back0 = (lane & 4) ? back : 0u, back1 = back - back0;
      const uint32_t dst = slots_lds + slot * PAIR;
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint32_t off = aoff[i][h] - (h ? back1 : back0);
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst + (2 * i + h) * 1024), "v"(off), "s"(abase) : "memory");
        }
#pragma unroll
      for (int j = 0; j < NT; j++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint8_t *bbase = brow[j] + (size_t)min(2 * q + h, p.ksteps - 1) * 1024;
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst + (2 * MT + 2 * j + h) * 1024), "v"(boff), "s"(bbase) : "memory");
        }
    };
    const int g = 4 * (r >> 3) + ((r & 7) >> 1);
    const int rd0 = (r >> 3) * 1024 + ((r & 7) * 8 + (c ^ g)) * 16;  // k-step 0 of a pair; k-step 1 sits at rd0 ^ 64
    const int4_t xr = {p.a_xor, p.a_xor, p.a_xor, p.a_xor};

#pragma unroll
    for (int u = 0; u < NP; u++)
      if (q_lo + u < q_hi) load_pair(q_lo + u, u);
    int slot = 0;
    for (int q = q_lo; q < q_hi; q++) {
      // pair q has landed when only the loads of the pairs behind it are in flight
      const int later = min(NP - 1, q_hi - 1 - q);  // uniform
      if (later == 0) iks_wait_vm<0>();
      else if (later == 1) iks_wait_vm<LOADS>();
      else if (later == 2) iks_wait_vm<(NP > 2 ? 2 : 0) * LOADS>();
      else iks_wait_vm<(NP > 3 ? 3 : 0) * LOADS>();
      const uint8_t *sl = slots + slot * PAIR;
      int4_t a[2][MT], b[2][NT];
#pragma unroll
      for (int h = 0; h < 2; h++) {
#pragma unroll
        for (int i = 0; i < MT; i++) a[h][i] = *reinterpret_cast<const int4_t *>(sl + i * 2048 + (rd0 ^ (64 * h)));
#pragma unroll
        for (int j = 0; j < NT; j++) b[h][j] = *reinterpret_cast<const int4_t *>(sl + (2 * MT + 2 * j + h) * 1024 + lane * 16);
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments are in registers: the slot may be filled again
      if (q + NP < q_hi) load_pair(q + NP, slot);
      slot = slot + 1 == NP ? 0 : slot + 1;
#pragma unroll
      for (int h = 0; h < 2; h++)
        if (2 * q + h < p.ksteps) {  // uniform
#pragma unroll
          for (int i = 0; i < MT; i++) {
            const int4_t av = a[h][i] ^ xr;
            // operands swapped: a lane holds four consecutive columns of one row
#pragma unroll
            for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(b[h][j], av, acc[i][j], 0, 0, 0);
          }
        }
    }
  }

  // ---- the waves' tiles meet in LDS and leave as whole rows ------------------------------------------------------------
  constexpr int RS = iks_row_ints(NT), ROWS = 16 * MT;
  __syncthreads();  // every wave has read its last slot
  int32_t *red = reinterpret_cast<int32_t *>(iks_ring);
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) *reinterpret_cast<int4_t *>(red + (wave * ROWS + 16 * i + r) * RS + 16 * j + 4 * c) = acc[i][j];
  __syncthreads();
  const float lo = (float)p.lo, hi = (float)p.hi;
  const int zp_mul = p.a_zp_dev ? 128 - (int)p.a_zp_dev[0] : p.zp_mul;
  const bool vec = (p.n & 3) == 0;
  for (int u = tid; u < ROWS * CPR; u += 64 * WAVES) {
    const int lrow = u / CPR, row = m0 + lrow;
    if (row >= p.m || col >= p.n) continue;
    const int32_t *src = red + lrow * RS + tid % CPR * 4;
    int4_t v = *reinterpret_cast<const int4_t *>(src);
#pragma unroll
    for (int w = 1; w < WAVES; w++) v += *reinterpret_cast<const int4_t *>(src + w * ROWS * RS);
#pragma unroll
    for (int e = 0; e < 4; e++) v[e] = (int32_t)((uint32_t)v[e] + (uint32_t)zp_mul * (uint32_t)zc[e]);
    const size_t o = (size_t)row * p.n + col;
    if (p.mode() == 1) {
      uint32_t packed = 0;
#pragma unroll
      for (int e = 0; e < 4; e++)
        packed |= (uint32_t)(uint8_t)requant_one(v[e], corr[e], comp[e], p.y_zp, p.round_mode(), lo, hi) << (8 * e);
      uint8_t *out = reinterpret_cast<uint8_t *>(p.out) + o;
      if (vec) {
        *reinterpret_cast<uint32_t *>(out) = packed;
      } else {
        for (int e = 0; e < 4; e++)
          if (col + e < p.n) out[e] = (uint8_t)(packed >> (8 * e));
      }
    } else {
      int4_t f;
#pragma unroll
      for (int e = 0; e < 4; e++) f[e] = iks_word(p, v[e], corr[e], comp[e], lo, hi);
      int32_t *out = reinterpret_cast<int32_t *>(p.out) + o;
      if (vec) {
        *reinterpret_cast<int4_t *>(out) = f;
      } else {
        for (int e = 0; e < 4; e++)
          if (col + e < p.n) out[e] = f[e];
      }
    }
  }
}

template <int MT, int NT, int WAVES, int NP>
int32_t iks_launch(const I8Args &p, hipStream_t s) {
  constexpr int LDS = iks_lds(MT, NT, WAVES, NP);
  static_assert(LDS <= 160 * 1024, "LDS of a CU");
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kern = i8_ksplit_kernel<MT, NT, WAVES, NP>;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS); });
  if (attr_err != hipSuccess) return set_error(YSCV_HIP_ERR_DEVICE, "cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr_err));
  const int tiles_m = (p.m + 16 * MT - 1) / (16 * MT), tiles_n = (p.n + 16 * NT - 1) / (16 * NT);
  const int each = iks_whole_columns(tiles_m, tiles_n) ? (tiles_n + 7) / 8 * tiles_m : (tiles_m * tiles_n + 7) / 8;  // workgroups of an XCD
  hipLaunchKernelGGL(kern, dim3(8 * (unsigned)each), dim3(64 * WAVES), LDS, s, p, tiles_m, tiles_n);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

// Tile shapes and what a workgroup of them takes: us to start, add its waves' tiles and end, and us per pair of a wave
// (fitted to 1 .. 2048 rows, N 256 .. 8192, K 256 .. 8192).
struct IksShape {
  int mt, nt, waves;
  double fixed, per_pair;
};
constexpr IksShape kIksShapes[] = {{1, 1, 8, 2.7, 0.42}, {1, 2, 8, 2.85, 0.44}, {1, 4, 4, 3.1, 0.54}, {2, 1, 8, 2.85, 0.45}, {2, 2, 8, 3.1, 0.50},
                                   {2, 4, 4, 3.8, 0.55}, {4, 2, 4, 3.75, 0.68}, {4, 4, 4, 4.5, 1.0}};
constexpr int kIksShapeCount = sizeof(kIksShapes) / sizeof(kIksShapes[0]);

// The shape with the shortest estimate among those whose workgroups all run at once, and that estimate.  (From two rounds over the
// CUs on the large tiles win, as they share operands among more MFMAs.)
int iks_pick(size_t m, size_t n, size_t ksteps, size_t cus, double &best_us) {
  int best = -1;
  best_us = 1e30;
  for (int i = 0; i < kIksShapeCount; i++) {
    const IksShape &sh = kIksShapes[i];
    const size_t tiles = ceil_div(m, (size_t)16 * sh.mt) * ceil_div(n, (size_t)16 * sh.nt);
    if (tiles > cus) continue;
    const double us = sh.fixed + sh.per_pair * ceil_div(ceil_div(ksteps, (size_t)2), (size_t)sh.waves);
    if (us < best_us) {
      best_us = us;
      best = i;
    }
  }
  return best;
}

int32_t iks_launch_shape(int shape, const I8Args &p, hipStream_t s) {
  switch (shape) {
    case 0: return iks_launch<1, 1, 8, 4>(p, s);
    case 1: return iks_launch<1, 2, 8, 3>(p, s);
    case 2: return iks_launch<1, 4, 4, 4>(p, s);
    case 3: return iks_launch<2, 1, 8, 3>(p, s);
    case 4: return iks_launch<2, 2, 8, 2>(p, s);
    case 5: return iks_launch<2, 4, 4, 3>(p, s);
    case 6: return iks_launch<4, 2, 4, 3>(p, s);
    default: return iks_launch<4, 4, 4, 2>(p, s);
  }
}

}  // namespace

double i8_ksplit_us(size_t m, size_t n, size_t ksteps, size_t cus) {
  double us;
  (void)iks_pick(m, n, ksteps, cus, us);
  return us;
}

int32_t launch_i8_ksplit(const I8Args &p, int num_cus, hipStream_t s) {
  double us;
  int shape = iks_pick((size_t)p.m, (size_t)p.n, (size_t)p.ksteps, num_cus > 0 ? (size_t)num_cus : 256, us);
  if (shape < 0) shape = kIksShapeCount - 1;  // (a K above 2^24 with more tiles than CUs)
  return iks_launch_shape(shape, p, s);
}

}  // namespace yscv
