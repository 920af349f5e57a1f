// Packed-int4 matmul for a few dozen to a few hundred activation rows (fp16-prepared activations):
// y[m][n] = sum_k x[m][k] * W[n][k].  Replaces packed_int4_gemm_dispatch
// (crates/yscv-kernels/src/ops/int4_matmul.rs:548-605) between the skinny kernel (one MFMA tile of rows) and the
// LDS-ring GEMM (tiles of 128 rows and more).
//
// At these sizes the time goes into latency, not into bytes or MFMAs: 64 rows against 4096 x 4096 are 9 MB of weights
// (2 us) and 2 GFLOP (1 us).  The LDS-ring kernel spends 0.45 us per 64-k stage on its chain weights -> decode -> LDS
// -> barrier -> fragments -> MFMA.  Here nothing is handed over inside the loop: a workgroup owns a tile of 16 MT rows x
// 16 NT columns of y, its eight waves split the K of the tile, each wave keeps the tile's accumulators and feeds itself:
// weights as they are stored straight into registers (one 128-bit load per lane is four k-steps), decoded once per MT
// MFMAs; activations through a slice of LDS of its own by LDS-direct loads, whole 128-byte lines in, fragments out.  No
// barrier until the eight partial tiles are added (fixed order) and stored as whole rows.
// (Fragments loaded straight into registers are sixteen rows x 64 bytes per load with neighbouring lanes in different
// rows: 30 GB/s per CU, a quarter of what whole lines get; 64 rows x 4096 x 4096 took 12.3 us that way.)
// us per call, nodes of one graph with a caller's workspace, the kernels before (LDS-ring; up to 32 rows int4_mid.hip) ->
// this one, fp16 rows, 32-groups, K 4096: 32 rows x 4096 10.9 -> 6.5, 64 x 4096 15.7 -> 7.9, 128 x 4096 17.0 -> 9.9, 256 x
// 4096 21.0 -> 15.1, 64 x 14336 21.1 -> 15.9; 128 x 1024 x 1024 9.8 -> 4.4.  (Called one by one, with the scratch the library
// then took per call: 21.7 -> 6.9, 25 -> 8.3, 25 -> 10.2, 25.4 -> 15.1, 25.5 -> 16.2, 9.5 -> 4.5.)
// The group scale is folded into fp16 weights as in the LDS-ring GEMM: fp16((q - zp) * s), rounded to 2^-11 per weight.  The MFMA is issued with the weights as the A operand: a lane holds four consecutive columns of a row.
#include <mutex>
#include <type_traits>

#include "int4_common.hpp"
#include "kernels.hpp"

namespace yscv {

namespace {

struct KsArgs {
  const uint8_t *tiles;
  const void *tscales;
  const uint8_t *tzps;  // null: zero point 8 everywhere
  const _Float16 *xh;
  const float *row_scale;  // null: 1
  void *y;
  float *partial;  // [parts][m][n] when K is also split over workgroups, else null
  int m, n, nt, ktp, chunks, chunk_div, ldx;
  int16_t y_dtype, epi;
  int kt, ksteps;  // 128-k tiles and 32-k steps that hold data
  int tiles_m, tiles_n, parts, kt_per;
};
static_assert(sizeof(KsArgs) <= kCheapArgs, "arguments of a launch");

template <int GM, bool SF16>
struct KsScale {
  static constexpr int SPT = GM == GM32 ? 4 : (GM == GM64 ? 2 : 1);
  static constexpr int BYTES = SPT * (SF16 ? 2 : 4);
  typedef typename std::conditional<SF16, _Float16, float>::type elem_t;
  typedef elem_t vec_t __attribute__((ext_vector_type(SPT)));
};

template <int NT, int GM, bool SF16, bool HAS_ZP>
struct KsTile {
  uint4_t w[NT];
  typename KsScale<GM, SF16>::vec_t s[NT];
  uint32_t z[HAS_ZP ? NT : 1];
};

template <int GM>
__device__ __forceinline__ uint32_t ks_load_zp(const uint8_t *p) {
  if constexpr (GM == GM32) return *reinterpret_cast<const uint32_t *>(p);
  if constexpr (GM == GM64) return *reinterpret_cast<const uint16_t *>(p);
  return *p;
}

// four consecutive columns of one row: a partial sum, or the result through the epilogue
__device__ __forceinline__ void ks_store(const KsArgs &p, int part, int row, int col, bool whole, float4_t v) {
  if (!p.partial) {
    store_cols4(p.y, p.y_dtype, p.epi, p.n, p.n, row, col, whole, v);
    return;
  }
  float *dst = p.partial + ((size_t)part * p.m + row) * p.n + col;
  if (whole) {
    *reinterpret_cast<float4_t *>(dst) = v;
  } else {
    for (int e = 0; e < 4; e++)
      if (col + e < p.n) dst[e] = v[e];
  }
}

// the MFMA B operands of a pair: k-step 0 at a0, k-step 1 at a1, 16-row groups 2 KiB apart; waits for them itself
template <int MT>
__device__ __forceinline__ void ks_read_pair(half8_t (&f)[2][MT], uint32_t a0, uint32_t a1) {
  if constexpr (MT == 2) {
    asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %4 offset:2048\n\tds_read_b128 %2, %5\n\tds_read_b128 %3, %5 offset:2048\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[1][0]), "=&v"(f[1][1]) : "v"(a0), "v"(a1) : "memory");
  } else {
    static_assert(MT == 4, "add a read for this tile height");
    asm volatile("ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:2048\n\tds_read_b128 %2, %8 offset:4096\n\tds_read_b128 %3, %8 offset:6144\n\t"
                 "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:2048\n\tds_read_b128 %6, %9 offset:4096\n\tds_read_b128 %7, %9 offset:6144\n\t"
                 "s_waitcnt lgkmcnt(0)"
                 : "=&v"(f[0][0]), "=&v"(f[0][1]), "=&v"(f[0][2]), "=&v"(f[0][3]), "=&v"(f[1][0]), "=&v"(f[1][1]), "=&v"(f[1][2]), "=&v"(f[1][3])
                 : "v"(a0), "v"(a1) : "memory");
  }
}

constexpr int KS_WAVES = 8;
// pairs of k-steps of x in flight per wave
constexpr int ks_np(int mt) { return mt <= 2 ? 4 : 2; }
// rows of the tile that are added at a time, and their LDS: eight waves' f32 rows, 16 bytes of padding per row (rows fall
// into different bank groups both when lanes write columns of sixteen rows and when threads read along a row)
constexpr int ks_pass_mt(int mt, int nt) { return mt * nt <= 16 ? mt : 16 / nt; }
constexpr int ks_red_bytes(int mt, int nt) { return KS_WAVES * 16 * ks_pass_mt(mt, nt) * (16 * nt + 4) * 4; }
constexpr int ks_x_bytes(int mt) { return KS_WAVES * ks_np(mt) * mt * 2048; }
constexpr int ks_lds(int mt, int nt) { return ks_red_bytes(mt, nt) > ks_x_bytes(mt) ? ks_red_bytes(mt, nt) : ks_x_bytes(mt); }

template <int MT, int NT, int GM, bool SF16, bool HAS_ZP>
__global__ void __launch_bounds__(64 * KS_WAVES) int4_ksplit_kernel(KsArgs p) {
  using S = KsScale<GM, SF16>;
  using Tile = KsTile<NT, GM, SF16, HAS_ZP>;
  // Loads return in order, so activations (L2) requested behind weights (HBM) wait for those: the weights of WD tiles are
  // requested up front, all of a wave's for K up to 4096 where the registers allow it
  constexpr int NP = ks_np(MT), WD = NT * (4 + (S::BYTES + 3) / 4 + (HAS_ZP ? 1 : 0)) <= 28 ? 4 : 2;
  extern __shared__ __attribute__((aligned(1024))) uint8_t ks_ring[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  // the row tiles of one column block run on one XCD (workgroup ids that are equal modulo 8), so its weights reach one L2
  const int q = (int)(blockIdx.x & 7) + 8 * ((int)(blockIdx.x >> 3) / p.tiles_m), tm = (int)(blockIdx.x >> 3) % p.tiles_m;
  if (q >= p.tiles_n * p.parts) return;
  const int part = q / p.tiles_n, tn = q % p.tiles_n;
  const int m0 = tm * 16 * MT, nt0 = tn * NT;
  const int kt_lo = part * p.kt_per, kt_n = min(p.kt - kt_lo, p.kt_per);
  const int t_lo = kt_lo + kt_n * wave / KS_WAVES, t_hi = kt_lo + kt_n * (wave + 1) / KS_WAVES;
  NibbleConsts nc;
  nc.init();

  float4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; i++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};

  if (t_lo < t_hi) {  // uniform in the wave
    // ---- weights: uniform base + 32-bit lane offset (opaque in each step, or the compiler turns base + offset into 64-bit
    // addresses per lane and load)
    uint32_t woff = lane * 16, soff = r * S::BYTES, zoff = r * S::SPT;
    size_t wrow[NT], srow[NT];  // uniform: first tile / first scale chunk of each 16-column block
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const size_t nt = (size_t)min(nt0 + j, p.nt - 1);  // blocks past the end repeat the last one and are not stored
      wrow[j] = nt * p.ktp;
      srow[j] = nt * p.chunks;
    }
    auto load_tile = [&](Tile &t, int kt) {
      const int chunk = GM == GM128 ? kt / p.chunk_div : kt;
      asm volatile("" : "+v"(woff), "+v"(soff), "+v"(zoff));
#pragma unroll
      for (int j = 0; j < NT; j++) {
        t.w[j] = *reinterpret_cast<const uint4_t *>(p.tiles + (wrow[j] + kt) * kTileBytes + woff);
        t.s[j] = *reinterpret_cast<const typename S::vec_t *>(reinterpret_cast<const uint8_t *>(p.tscales) + (srow[j] + chunk) * 16 * S::BYTES + soff);
        if constexpr (HAS_ZP) t.z[j] = ks_load_zp<GM>(p.tzps + (srow[j] + chunk) * 16 * S::SPT + zoff);
      }
    };
    // ---- activations: pair q = k-steps 2q and 2q + 1 of all rows, 16 rows as two pieces of eight whole 128-byte lines.  Lane i
    // of piece h fetches 16-byte chunk (i & 7) ^ g of row i / 8, g = 4 h + (i / 8) / 2, so that the sixteen rows a fragment
    // read touches fall into sixteen different 16-byte slots.
    uint32_t aoff[MT][2];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int row8 = lane >> 3, row = min(m0 + 16 * i + 8 * h + row8, p.m - 1);
        aoff[i][h] = (uint32_t)(((size_t)row * p.ldx + ((lane & 7) ^ (4 * h + (row8 >> 1))) * 8) * 2);
      }
    // K may end behind the first k-step of its last pair: the lanes of the second one read the first one's data again
    const int last_pair = (p.ksteps - 1) >> 1;
    const bool half_pair = p.ksteps & 1;
    const uint32_t slots = (uint32_t)(size_t)ks_ring + (uint32_t)(wave * NP * MT * 2048);
    auto load_x = [&](int q, uint32_t slot) {
      q = min(q, last_pair);
      const char *base = reinterpret_cast<const char *>(p.xh) + (size_t)q * 128;
      const uint32_t back = half_pair && q == last_pair ? 64u : 0u, back0 = (lane & 4) ? back : 0u, back1 = back - back0;
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint32_t dst = slots + slot * (MT * 2048) + (uint32_t)((2 * i + h) * 1024), off = aoff[i][h] - (h ? back1 : back0);
          asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory");
        }
    };
    const uint32_t g = 4u * (r >> 3) + ((r & 7) >> 1);
    const uint32_t rd0 = slots + (uint32_t)((r >> 3) * 1024) + (((r & 7) * 8 + (c ^ g)) * 16), rd1 = rd0 ^ 64u;  // k-steps 0 and 1

    Tile ring[WD];
#pragma unroll
    for (int u = 0; u < WD; u++) load_tile(ring[u], min(t_lo + u, t_hi - 1));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < NP; u++) load_x(2 * t_lo + u, u);
    uint32_t slot = 0;
    for (int kt0 = t_lo; kt0 < t_hi; kt0 += WD) {
#pragma unroll
      for (int u = 0; u < WD; u++) {
        const int kt = kt0 + u;
        if (kt < t_hi) {  // uniform
#pragma unroll
          for (int hf = 0; hf < 2; hf++) {
            const int q = 2 * kt + hf;
            half8_t a[2][MT];
            // The pair has landed when at most the loads of the NP - 1 pairs behind it are in flight (weight loads issued since
            // only make the wait longer); its fragments are read and waited for in one statement.
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NP - 1) * MT * 2) : "memory");
            ks_read_pair<MT>(a, rd0 + slot * (MT * 2048), rd1 + slot * (MT * 2048));
            load_x(q + NP, slot);
            slot = slot + 1 == NP ? 0 : slot + 1;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; h++) {
              const int ks = 2 * hf + h;
              if (2 * q + h < p.ksteps) {  // uniform; the steps past the end of K are the last wave's
                half8_t wf[NT];
#pragma unroll
                for (int j = 0; j < NT; j++) {
                  const int e = GM == GM32 ? ks : (GM == GM64 ? ks >> 1 : 0);
                  const uint32_t zq = HAS_ZP ? ((ring[u].z[HAS_ZP ? j : 0] >> (8 * e)) & 0xFFu) : 8u;
                  const _Float16 z = (_Float16)(float)zq;
                  const _Float16 c1v = (_Float16)(-1024.0f) - z, c2v = (_Float16)(-64.0f) - z;
                  const _Float16 s = (_Float16)ring[u].s[j][e];
                  wf[j] = decode8_exact(ring[u].w[j][ks], nc, half2_t{c1v, c1v}, half2_t{c2v, c2v}) * half8_t{s, s, s, s, s, s, s, s};
                }
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                  for (int j = 0; j < NT; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[j], a[h][i], acc[i][j], 0, 0, 0);
              }
            }
          }
          if (kt + WD < t_hi) load_tile(ring[u], kt + WD);
        }
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the pairs requested past the end have landed: the slots are free
  }

  // ---- the eight partial tiles meet in LDS, PM row tiles at a time, and leave as whole rows ---------------------------
  constexpr int PM = ks_pass_mt(MT, NT), RS = 16 * NT + 4, ROWS = 16 * PM;  // floats per row
  __syncthreads();  // every wave is done with its slots
  float *red = reinterpret_cast<float *>(ks_ring);
  const bool vec = (p.n & 3) == 0;
#pragma unroll
  for (int i0 = 0; i0 < MT; i0 += PM) {
    if (i0 > 0) __syncthreads();
#pragma unroll
    for (int i = 0; i < PM; i++)
#pragma unroll
      for (int j = 0; j < NT; j++)
        if (i0 + i < MT) *reinterpret_cast<float4_t *>(red + (wave * ROWS + 16 * i + r) * RS + 16 * j + 4 * c) = acc[(i0 + i) % MT][j];
    __syncthreads();
    constexpr int CPR = 4 * NT, UNITS = ROWS * CPR;
#pragma unroll
    for (int u0 = 0; u0 < UNITS; u0 += 64 * KS_WAVES) {
      const int u = u0 + tid, lrow = u / CPR, row = m0 + 16 * i0 + lrow, col = nt0 * 16 + u % CPR * 4;
      if ((UNITS % (64 * KS_WAVES) == 0 || u < UNITS) && 16 * i0 + lrow < 16 * MT && row < p.m && col < p.n) {
        const float *src = red + lrow * RS + u % CPR * 4;
        float4_t v = *reinterpret_cast<const float4_t *>(src);
#pragma unroll
        for (int w = 1; w < KS_WAVES; w++) v += *reinterpret_cast<const float4_t *>(src + w * ROWS * RS);
        if (p.row_scale) v = v * p.row_scale[row];
        ks_store(p, part, row, col, vec, v);
      }
    }
  }
}

template <int MT, int NT, int GM, bool SF16, bool HAS_ZP>
int32_t ks_launch_one(const KsArgs &a, hipStream_t s) {
  constexpr int LDS = ks_lds(MT, NT);
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  auto kern = int4_ksplit_kernel<MT, NT, GM, SF16, HAS_ZP>;
  std::call_once(once, [&] { attr_err = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, LDS); });
  if (attr_err != hipSuccess) return set_error(YSCV_HIP_ERR_DEVICE, "cannot reserve %d bytes of LDS: %s", LDS, hipGetErrorString(attr_err));
  const unsigned cols = (unsigned)(a.tiles_n * a.parts);
  hipLaunchKernelGGL(kern, dim3((cols + 7) / 8 * 8 * (unsigned)a.tiles_m), dim3(64 * KS_WAVES), LDS, s, a);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}

template <int MT, int NT, int GM, bool SF16>
int32_t ks_launch_zp(const KsArgs &a, hipStream_t s) {
  return a.tzps ? ks_launch_one<MT, NT, GM, SF16, true>(a, s) : ks_launch_one<MT, NT, GM, SF16, false>(a, s);
}
template <int MT, int NT>
int32_t ks_launch_gm(const KsArgs &a, int gm, bool sf16, hipStream_t s) {
  if (gm == GM32) return sf16 ? ks_launch_zp<MT, NT, GM32, true>(a, s) : ks_launch_zp<MT, NT, GM32, false>(a, s);
  if (gm == GM64) return sf16 ? ks_launch_zp<MT, NT, GM64, true>(a, s) : ks_launch_zp<MT, NT, GM64, false>(a, s);
  return sf16 ? ks_launch_zp<MT, NT, GM128, true>(a, s) : ks_launch_zp<MT, NT, GM128, false>(a, s);
}

// Tile shapes (16 MT rows x 16 NT columns) and what a workgroup of them takes: us to start, add its waves' tiles and
// end, and us per 128-k tile of K (fitted to 20 .. 256 rows, N 1024 .. 14336, K 1024 .. 14336).
struct KsShape {
  int mt, nt;
  double fixed, per_tile;
};
constexpr KsShape kShapes[] = {{2, 1, 3.3, 0.148}, {2, 2, 3.8, 0.158}, {2, 4, 4.8, 0.214}, {4, 1, 3.9, 0.197}, {4, 2, 4.3, 0.197}, {4, 4, 5.6, 0.290}};
constexpr int kShapeCount = sizeof(kShapes) / sizeof(kShapes[0]);

// x is read by every workgroup and should come from L2 (4 MB per XCD); up to twice that the kernel still won
constexpr size_t kKsplitXBytes = (size_t)8 << 20;

struct KsPlan {
  int shape;  // < 0: none fits
  int parts, kt_per;
};

// The shape and K split with the shortest estimated time among those whose workgroups all run at once: from two rounds
// over the CUs on, the LDS-ring GEMM, which shares operands across a larger tile, is as fast or faster (64 rows x 28672 x
// 4096: 35 us against 31).  A K split over workgroups costs its second kernel: 3.4 us and its traffic.
KsPlan ks_plan(size_t m, size_t n, size_t kt, int cus) {
  KsPlan best{-1, 1, (int)kt};
  double best_us = 1e30;
  for (int i = 0; i < kShapeCount; i++) {
    const size_t tiles = ceil_div(m, (size_t)16 * kShapes[i].mt) * ceil_div(n, (size_t)16 * kShapes[i].nt);
    for (size_t parts = 1; parts <= 4 && tiles * parts <= (size_t)cus; parts *= 2) {
      if (parts > 1 && (kt / parts < 8 || parts * m * n * sizeof(float) > kKsplitPartialCap)) break;
      const double us = kShapes[i].fixed + kShapes[i].per_tile * round_up(ceil_div(kt, parts), 8) +
                        (parts > 1 ? 3.4 + (double)(parts * m * n * 8) / 5e6 : 0.0);
      if (us < best_us) {
        best_us = us;
        best = KsPlan{i, (int)parts, (int)ceil_div(kt, parts)};
      }
    }
  }
  if (best.shape >= 0) best.parts = (int)ceil_div(kt, (size_t)best.kt_per);
  return best;
}

}  // namespace

bool int4_ksplit_takes(const yscv_hip_int4_weight *w, size_t m, int num_cus) {
  return w->tiled && m > 16 && m * w->k * sizeof(_Float16) <= kKsplitXBytes && ks_plan(m, w->n, w->kt, num_cus > 0 ? num_cus : 256).shape >= 0;
}

size_t int4_ksplit_partial_bytes(const yscv_hip_int4_weight *w, size_t m, int num_cus) {
  const KsPlan pl = ks_plan(m, w->n, w->kt, num_cus > 0 ? num_cus : 256);
  return pl.shape >= 0 && pl.parts > 1 ? (size_t)pl.parts * m * w->n * sizeof(float) : 0;
}

int32_t launch_int4_ksplit(const yscv_hip_int4_weight *w, const _Float16 *xh, const float *row_scale, size_t ldx, void *y, int y_dtype, size_t m,
                           hipStream_t s, int epi, float *partial, size_t partial_bytes) {
  if (epi == EPI_ADD_F32 && y_dtype != YSCV_HIP_F32) return set_error(YSCV_HIP_ERR_INVALID_ARG, "the add epilogue updates an f32 tensor");
  if (epi == EPI_SWIGLU && (w->n & 1)) return set_error(YSCV_HIP_ERR_INVALID_ARG, "SwiGLU epilogue needs an even row count");
  const Context *ctx = nullptr;
  YSCV_TRY(ensure_context(&ctx));
  KsPlan pl = ks_plan(m, w->n, w->kt, ctx->num_cus > 0 ? ctx->num_cus : 256);
  if (pl.shape < 0) return set_error(YSCV_HIP_ERR_INVALID_ARG, "%zu x %zu has too many tiles for the K-split kernel", m, w->n);
  if (pl.parts > 1 && (partial == nullptr || partial_bytes < (size_t)pl.parts * m * w->n * sizeof(float) || (reinterpret_cast<uintptr_t>(partial) & 15) != 0)) {
    pl.parts = 1;
    pl.kt_per = (int)w->kt;
  }
  KsArgs a;
  a.tiles = w->tiles;
  a.tscales = w->tscales;
  a.tzps = w->has_zp ? w->tzps : nullptr;
  a.xh = xh;
  a.row_scale = row_scale;
  a.y = y;
  a.partial = pl.parts > 1 ? partial : nullptr;
  a.m = (int)m;
  a.n = (int)w->n;
  a.nt = (int)w->nt;
  a.ktp = (int)w->ktp;
  a.chunks = (int)w->chunks;
  a.chunk_div = w->gm == GM128 ? (int)(w->g / 128) : 1;
  a.ldx = (int)ldx;
  a.y_dtype = y_dtype;
  a.epi = epi;
  a.kt = (int)w->kt;
  a.ksteps = (int)(w->k / 32);
  a.tiles_m = (int)ceil_div(m, (size_t)16 * kShapes[pl.shape].mt);
  a.tiles_n = (int)ceil_div(w->n, (size_t)16 * kShapes[pl.shape].nt);
  a.parts = pl.parts;
  a.kt_per = pl.kt_per;
  const bool sf16 = w->scale_dtype == YSCV_HIP_F16;
  int32_t st = YSCV_HIP_OK;
  switch (pl.shape) {
    case 0: st = ks_launch_gm<2, 1>(a, w->gm, sf16, s); break;
    case 1: st = ks_launch_gm<2, 2>(a, w->gm, sf16, s); break;
    case 2: st = ks_launch_gm<2, 4>(a, w->gm, sf16, s); break;
    case 3: st = ks_launch_gm<4, 1>(a, w->gm, sf16, s); break;
    case 4: st = ks_launch_gm<4, 2>(a, w->gm, sf16, s); break;
    default: st = ks_launch_gm<4, 4>(a, w->gm, sf16, s); break;
  }
  YSCV_TRY(st);
  if (a.partial) return launch_int4_partial_sum(a.partial, a.parts, a.m, a.n, y, y_dtype, epi, s);
  return YSCV_HIP_OK;
}

}  // namespace yscv
