// Packed-int4 matrix x one activation row, or up to four: packed_int4_gemv_dispatch (crates/yscv-kernels/src/ops/
// int4_matmul.rs:310) where the skinny kernel's workgroups, made for up to 16 rows and many blocks each, start slowly.
//
// A wave takes 16 weight rows x 512 k: every load it needs is requested at once (four 1 KiB tiles, one load of scales, one or two
// of activations) and nothing passes through LDS on the way to the matrix cores.  The 16 rows of the MFMA's activation
// operand carry the wave's 16 blocks of 32 k, so a lane's operand is eight consecutive activations, as they lie in memory, and
// it serves all sixteen MFMAs of the slice; of the result of block j = 4t + q only row j counts: register q of the lanes 16 t ..
// 16 t + 15, which also hold the scales of tile t.  f32 and bf16 activations are brought to 2^14 .. 2^15 by a power of two per
// slice, f32 split into fp16 hi + lo (22 bits), as in the skinny kernel; weights are exact (q - 8); a zero point enters as
// (8 - zp) * sum of the block's activations, one more MFMA against ones for all sixteen blocks.
// K above 4096 takes sixteen waves, so that few of them have a second or third slice behind the first (4096 x 14336 fp16 with
// eight waves 8.9 us, with sixteen 7.8).  Residual updates, SwiGLU and a folded norm (NormFold in kernels.hpp) are done by the threads
// that hold the sums, with their operands requested ahead of the weights.
// Bound: below a few MB of weights the launch and one round trip to memory each for arguments, loads and sums; above that the
// 4.5 - 5 TB/s that loads of this kind reach behind decode and MFMA.  One row, us a call in a graph of six, the skinny kernel (with its
// workspace) -> this one, weights from HBM | in a cache: 4096 x 4096 f32 10.7 -> 6.6 | 10.1 -> 5.6, fp16 7.0 -> 5.9 | 6.4 -> 5.0, bf16
// 8.7 -> 6.1 | 8.0 -> 5.2; 4096 x 14336 f32 17.1 -> 11.4 | 16.5 -> 9.5, fp16 14.1 -> 10.3 | 13.5 -> 7.5; 16384 x 1024 with zero points
// fp16 8.9 -> 5.9 | 8.5 -> 5.1.  LM heads: 151936 x 1024 fp16 27.7 -> 16.5, f32 42.0 -> 18.7; 128256 x 4096 fp16 54 -> 59, f32 68 -> 65.
// A graph step of the 7B-shape decoder at batch 1: 1619 -> 1376 us (q/k/v 7.3 -> 5.5, o 6.2 -> 4.7, gate/up 14.5 ->
// 13.6, down with its second pass 14.5 -> 8.6, traced), of the 24-layer one 692 -> 630.
// Relative error against 64 bits over those shapes and a dozen others: f32 0.99e-7 .. 1.29e-7 -> 0.80e-7 .. 0.90e-7; fp16 and bf16
// 5e-6 .. 1.3e-5 (0.5e-7 .. 0.9e-7 with zero points) -> 0.47e-7 .. 0.49e-7, as no 1024 stays in the weights here and the sums of
// more than 128 products are in 64 bits.  The low product is added behind the high one: the other order costs up to half as
// much again.
#include <type_traits>

#include "int4_common.hpp"
#include "int4_gemv_plan.hpp"
#include "kernels.hpp"

namespace yscv {

namespace {

__device__ __forceinline__ double sum_xor16_xor32(double v) {  // v + v[lane ^ 16], then the same over lane ^ 32
  float xl, yl, xh, yh;
  xor16_pair(__int_as_float(__double2loint(v)), xl, yl);
  xor16_pair(__int_as_float(__double2hiint(v)), xh, yh);
  v = __hiloint2double(__float_as_int(xh), __float_as_int(xl)) + __hiloint2double(__float_as_int(yh), __float_as_int(yl));
  xor32_pair(__int_as_float(__double2loint(v)), xl, yl);
  xor32_pair(__int_as_float(__double2hiint(v)), xh, yh);
  return __hiloint2double(__float_as_int(xh), __float_as_int(xl)) + __hiloint2double(__float_as_int(yh), __float_as_int(yl));
}

struct GemvPlainArgs {
  const uint8_t *tiles;
  const void *tscales;
  const uint8_t *tzps;
  const void *x;
  void *y;
  int m, n, k, nt, ktp, chunks, chunk_div;
  int groups, wgs;         // groups of rows, waves / split blocks of 16 each; workgroups that share them
  int slices, split_log2;  // 512-k slices of K; waves of a workgroup that share a block of 16 rows (1, 2, 4, 8 or 16)
  int y_dtype, epi;
};
static_assert(sizeof(GemvPlainArgs) <= kCheapArgs, "arguments of a launch");

struct GemvRowArgs : GemvPlainArgs {
  // a norm folded into this call (NormFold in kernels.hpp); null / 0 when unused
  const float *gamma_next, *pre;
  _Float16 *xg;
  float *ss_out;
  const float *ss_in, *pre_in;
  float *pre_next;
  int ss_in_count, ss_in_stride, ss_out_stride;
  float inv_d, eps;
};

// XD: type of the activations; f32 takes two MFMA operands, the others one.
// EPI: residual update, SwiGLU or a folded norm; a plain product leaves that code and its arguments out (one row, 4096 x 4096 fp16 4.0 instead of 4.2 us,
// 3000 x 704 f32 3.25 instead of 3.5: less to fetch at the start).
// KEEP: a wave has one slice of K (K <= 4096).  Its activations stay in registers while the workgroup goes through its groups of
// rows; without it a workgroup has one group and the waves go through their slices.
// waves that a SIMD has to hold
constexpr int gemv_per_simd(int m, int xd, bool zp, bool keep) { return m == 4 || (m == 2 && (!keep || (zp && xd == YSCV_HIP_F32))) ? 2 : 4; }

template <int M, int XD, int GM, bool SF16, bool HAS_ZP, bool KEEP, bool EPI>
__global__ void __launch_bounds__((64 * gemv_waves(M, KEEP)), (gemv_per_simd(M, XD, HAS_ZP, KEEP)))
int4_gemv_kernel(typename std::conditional<EPI, GemvRowArgs, GemvPlainArgs>::type args) {
  GemvRowArgs p;
  if constexpr (EPI) p = args;
  else static_cast<GemvPlainArgs &>(p) = args;
  constexpr int WAVES = gemv_waves(M, KEEP);
  if constexpr (!EPI) {
    p.epi = EPI_STORE;
    p.ss_in = nullptr;
    p.xg = nullptr;
  }
  constexpr int SPT = GM == GM32 ? 4 : (GM == GM64 ? 2 : 1);
  constexpr bool F32 = XD == YSCV_HIP_F32;
  typedef typename std::conditional<SF16, _Float16, float>::type elem_t;
  typedef elem_t scale_t __attribute__((ext_vector_type(SPT)));
  typedef uint8_t zp_t __attribute__((ext_vector_type(SPT)));
  __shared__ double part[2][WAVES][M][16];
  __shared__ float norm_factor[M];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, c = lane >> 4;
  const int split = 1 << p.split_log2, sub = wave >> p.split_log2, ks = wave & (split - 1);  // block of the group, first slice
  const int blocks = WAVES >> p.split_log2;
  NibbleConsts nc;
  nc.init();
  uint32_t magic_hi = 0x54005400u;
  asm volatile("" : "+v"(magic_hi));
  const half8_t off8 = {(_Float16)1032.0f, (_Float16)1032.0f, (_Float16)72.0f, (_Float16)72.0f,
                        (_Float16)1032.0f, (_Float16)1032.0f, (_Float16)72.0f, (_Float16)72.0f};
  const float4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};

  struct Weights {
    uint4_t w[4];
    scale_t s;
    zp_t z;
  };
  struct Acts {
    half8_t hi[M], lo[M];
    float4_t sum[M];  // zero points: the sums of the blocks of tile c
    float down[M];
  };
  struct Raw {
    float4_t x[M][2];  // f32: eight values; fp16 and bf16: the first four words
  };
  struct Sums {
    float v[M];
  };
  auto load = [&](int group, int sl) {
    Weights v;
    const int nt = min(group * blocks + sub, p.nt - 1);
    const uint8_t *t0 = p.tiles + ((size_t)nt * p.ktp + (size_t)sl * 4) * kTileBytes + lane * 16;
#pragma unroll
    for (int t = 0; t < 4; t++) v.w[t] = *reinterpret_cast<const uint4_t *>(t0 + t * kTileBytes);
    const int chunk = GM == GM128 ? min((sl * 4 + c) / p.chunk_div, p.chunks - 1) : sl * 4 + c;
    const size_t at = (((size_t)nt * p.chunks + chunk) * 16 + r) * SPT;
    v.s = *reinterpret_cast<const scale_t *>(reinterpret_cast<const elem_t *>(p.tscales) + at);
    if constexpr (HAS_ZP) v.z = *reinterpret_cast<const zp_t *>(p.tzps + at);
    return v;
  };
  auto load_x = [&](int sl) {
    Raw v;
    const int k0 = sl * 512 + 32 * r + 8 * c;  // K is a multiple of 32: a lane's eight values exist or do not
    const bool in = k0 < p.k;
    const int kk = in ? k0 : 0;
#pragma unroll
    for (int i = 0; i < M; i++) {
      const size_t at = (size_t)min(i, p.m - 1) * p.k + kk;  // rows past the last repeat it
      if constexpr (F32) {
        const float *src = static_cast<const float *>(p.x) + at;
        v.x[i][0] = *reinterpret_cast<const float4_t *>(src);
        v.x[i][1] = *reinterpret_cast<const float4_t *>(src + 4);
      } else {
        v.x[i][0] = *reinterpret_cast<const float4_t *>(static_cast<const _Float16 *>(p.x) + at);
      }
    }
#pragma unroll
    for (int i = 0; i < M; i++)
#pragma unroll
      for (int e = 0; e < 4; e++) {
        v.x[i][0][e] = in ? v.x[i][0][e] : 0.0f;
        if constexpr (F32) v.x[i][1][e] = in ? v.x[i][1][e] : 0.0f;
      }
    return v;
  };
  auto times = [&](half8_t hi, half8_t lo, half8_t b) {
    float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, b, zero, 0, 0, 0);
    if constexpr (F32) d = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo, b, d, 0, 0, 0);
    return d;
  };
  auto prepare = [&](const Raw &v) {
    Acts x;
#pragma unroll
    for (int i = 0; i < M; i++) {
      x.down[i] = 1.0f;
      if constexpr (XD == YSCV_HIP_F16) {
        union {
          float4_t f;
          half8_t h;
        } u;
        u.f = v.x[i][0];
        x.hi[i] = u.h;
      } else {
        float f[8], mx = 0.0f;
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const uint32_t two = __float_as_uint(v.x[i][0][e >> 1]);
          f[e] = F32 ? v.x[i][e >> 2][e & 3] : __uint_as_float((e & 1) ? two & 0xffff0000u : two << 16);
          mx = fmaxf(mx, fabsf(f[e]));
        }
        const uint32_t top = (__float_as_uint(wave_max(mx)) >> 23) & 255u, ex = min(268u - top, 253u);
        const float up = __uint_as_float(ex << 23);
        x.down[i] = __uint_as_float((254u - ex) << 23);
#pragma unroll
        for (int e = 0; e < 8; e++) {
          const float t = f[e] * up;
          x.hi[i][e] = (_Float16)t;
          if constexpr (F32) x.lo[i][e] = (_Float16)(t - (float)x.hi[i][e]);
        }
      }
      if constexpr (HAS_ZP) {
        const half8_t ones = {(_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f,
                              (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f, (_Float16)1.0f};
        x.sum[i] = times(x.hi[i], x.lo[i], ones);
      }
    }
    return x;
  };
  auto multiply = [&](const Weights &v, const Acts &x) {
    float sel[M][4];
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const half8_t b = extract8(v.w[t][q], nc, magic_hi) - off8;
#pragma unroll
        for (int i = 0; i < M; i++) {
          const float4_t d = times(x.hi[i], x.lo[i], b);
          sel[i][q] = t == 0 ? d[q] : (c == t ? d[q] : sel[i][q]);
        }
        if constexpr (M > 1) __builtin_amdgcn_sched_barrier(0);  // results of many blocks at once do not fit the registers
      }
    Sums o;
#pragma unroll
    for (int i = 0; i < M; i++) {
      float acc = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int e = GM == GM32 ? q : (GM == GM64 ? q >> 1 : 0);
        if constexpr (HAS_ZP) sel[i][q] = fmaf(8.0f - (float)v.z[e], x.sum[i][q], sel[i][q]);
        acc = fmaf((float)v.s[e], sel[i][q], acc);
      }
      o.v[i] = acc * x.down[i];
    }
    return o;
  };
  // the thread's row of the weight block and of the activations in the closing sums
  const int own_b = (tid >> 4) & (blocks - 1), own_m = (tid >> 4) >> (31 - __builtin_clz(WAVES) - p.split_log2);
  // What the folded norm needs, requested ahead of everything else: the partial sums of squares (row i is added up by the i-th
  // wave from the end), and the residuals of the first group in the threads that will update them
  float ss[4] = {0.0f, 0.0f, 0.0f, 0.0f}, ss_pre = 1.0f, h_old = 0.0f, h_mul = 0.0f;
  const int ss_row = WAVES - 1 - wave;
  const bool sums_norm = p.ss_in && ss_row < min(M, p.m);  // uniform in the wave
  if (sums_norm) {
#pragma unroll
    for (int i = 0; i < 4; i++) ss[i] = p.ss_in[(size_t)ss_row * p.ss_in_stride + min(lane * 4 + i, p.ss_in_count - 1)];
    ss_pre = p.pre_in[ss_row];
  }
  if (p.epi == EPI_ADD_F32 && own_m < M) {
    const int row = min(((int)blockIdx.x * blocks + own_b) * 16 + (tid & 15), p.n - 1), i = min(own_m, p.m - 1);
    h_old = static_cast<const float *>(p.y)[(size_t)i * p.n + row];
    if (p.xg) h_mul = p.gamma_next[row] * p.pre[i];
  }
  auto norm_sum = [&] {  // before the barrier of the first group
    if (sums_norm) {
#pragma unroll
      for (int i = 0; i < 4; i++) ss[i] = lane * 4 + i < p.ss_in_count ? ss[i] : 0.0f;
      const float inv_rms = 1.0f / sqrtf(wave_sum((ss[0] + ss[1]) + (ss[2] + ss[3])) * p.inv_d + p.eps);
      if (lane == 0) {
        norm_factor[ss_row] = inv_rms / ss_pre;
        if (p.pre_next && blockIdx.x == 0) p.pre_next[ss_row] = norm_fold_prescale(inv_rms);
      }
    }
  };
  auto store_row = [&](int group, int row, float v) {
    if (p.ss_in) v *= norm_factor[min(own_m, p.m - 1)];
    const bool live = row < p.n && own_m < p.m;
    const size_t at = (size_t)own_m * p.n + row;
    if (p.epi == EPI_ADD_F32) {
      float *h = static_cast<float *>(p.y) + at;
      const bool first = group == (int)blockIdx.x;
      const float hn = live ? (first ? h_old : *h) + v : 0.0f;
      if (live) *h = hn;
      if (p.xg) {  // the sixteen lanes of a block leave one sum of squares
        const float mul = first ? h_mul : (live ? p.gamma_next[row] * p.pre[own_m] : 0.0f);
        if (live) p.xg[at] = (_Float16)fminf(fmaxf(hn * mul, -65504.0f), 65504.0f);
        const float sq = row_sum16(hn * hn);
        if ((tid & 15) == 0 && live) p.ss_out[(size_t)own_m * p.ss_out_stride + group * blocks + own_b] = sq;
      }
    } else if (p.epi == EPI_SWIGLU) {  // rows 2i and 2i + 1 of the weight are gate i and up i
      const float up = dpp_move<DPP_XOR1>(v);
      if (live && !(row & 1)) store_out(p.y, (size_t)own_m * (p.n >> 1) + (row >> 1), silu(v) * up, p.y_dtype);
    } else if (live) {
      store_out(p.y, at, v, p.y_dtype);
    }
  };
  // from the 128 k of a lane on the sums are in 64 bits; the waves' meet in LDS; only LDS is waited for, the loads ahead stay
  // in flight
  struct Totals {
    double v[M];
  };
  auto finish = [&](int group, int buf, const Totals &total) {
#pragma unroll
    for (int i = 0; i < M; i++) {
      const double t = sum_xor16_xor32(total.v[i]);
      if (lane < 16) part[buf][wave][i][lane] = t;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (own_m < M) {
      double v = 0.0;
      for (int w = 0; w < split; w++) v += part[buf][own_b * split + w][own_m][tid & 15];
      store_row(group, (group * blocks + own_b) * 16 + (tid & 15), (float)v);
    }
  };
  auto widen = [](const Sums &a) {
    Totals t;
#pragma unroll
    for (int i = 0; i < M; i++) t.v[i] = (double)a.v[i];
    return t;
  };
  Totals nothing;
#pragma unroll
  for (int i = 0; i < M; i++) nothing.v[i] = 0.0;

  if constexpr (KEEP) {  // two buffers: a wave past the barrier of group i + 1 has read the sums of group i
    const int sl = min(ks, p.slices - 1), step = p.wgs;
    const bool in = ks < p.slices;
    int group = (int)blockIdx.x, buf = 0;
    const Raw xr = load_x(sl);
    Weights v = load(group, sl);
    const Acts x = prepare(xr);
    norm_sum();
    for (; group + step < p.groups; group += step, buf ^= 1) {
      const Weights nx = load(group + step, sl);
      finish(group, buf, in ? widen(multiply(v, x)) : nothing);
      v = nx;
    }
    finish(group, buf, in ? widen(multiply(v, x)) : nothing);
  } else {
    int sl = ks;
    Totals total = nothing;
    auto add = [&](const Sums &a) {
#pragma unroll
      for (int i = 0; i < M; i++) total.v[i] += (double)a.v[i];
    };
    if (sl < p.slices) {  // uniform in the wave
      Raw xr = load_x(sl);
      Weights v = load((int)blockIdx.x, sl);
      for (; sl + split < p.slices; sl += split) {
        const Raw xn = load_x(sl + split);
        const Weights nx = load((int)blockIdx.x, sl + split);
        add(multiply(v, prepare(xr)));
        xr = xn;
        v = nx;
      }
      add(multiply(v, prepare(xr)));
    }
    norm_sum();
    finish((int)blockIdx.x, 0, total);
  }
}

template <int M, int XD, int GM, bool SF16, bool EPI>
int32_t gemv_go(const GemvRowArgs &all, unsigned grid, hipStream_t s) {
  const typename std::conditional<EPI, GemvRowArgs, GemvPlainArgs>::type &a = all;
  const bool keep = a.slices <= 8;
  const dim3 threads(64 * gemv_waves(M, keep));
  if (keep && a.tzps) hipLaunchKernelGGL((int4_gemv_kernel<M, XD, GM, SF16, true, true, EPI>), dim3(grid), threads, 0, s, a);
  else if (keep) hipLaunchKernelGGL((int4_gemv_kernel<M, XD, GM, SF16, false, true, EPI>), dim3(grid), threads, 0, s, a);
  else if (a.tzps) hipLaunchKernelGGL((int4_gemv_kernel<M, XD, GM, SF16, true, false, EPI>), dim3(grid), threads, 0, s, a);
  else hipLaunchKernelGGL((int4_gemv_kernel<M, XD, GM, SF16, false, false, EPI>), dim3(grid), threads, 0, s, a);
  YSCV_HIP_TRY(hipGetLastError());
  return YSCV_HIP_OK;
}
template <int M, int XD, int GM, bool SF16>
int32_t gemv_epi(const GemvRowArgs &a, unsigned grid, hipStream_t s) {
  if (a.epi == EPI_STORE && !a.ss_in) return gemv_go<M, XD, GM, SF16, false>(a, grid, s);
  return gemv_go<M, XD, GM, SF16, true>(a, grid, s);
}
template <int M, int XD>
int32_t gemv_gm(const GemvRowArgs &a, unsigned grid, int gm, bool sf16, hipStream_t s) {
  if (gm == GM32) return sf16 ? gemv_epi<M, XD, GM32, true>(a, grid, s) : gemv_epi<M, XD, GM32, false>(a, grid, s);
  if (gm == GM64) return sf16 ? gemv_epi<M, XD, GM64, true>(a, grid, s) : gemv_epi<M, XD, GM64, false>(a, grid, s);
  return sf16 ? gemv_epi<M, XD, GM128, true>(a, grid, s) : gemv_epi<M, XD, GM128, false>(a, grid, s);
}
template <int M>
int32_t gemv_xd(const GemvRowArgs &a, unsigned grid, int x_dtype, int gm, bool sf16, hipStream_t s) {
  if (x_dtype == YSCV_HIP_F32) return gemv_gm<M, YSCV_HIP_F32>(a, grid, gm, sf16, s);
  if (x_dtype == YSCV_HIP_BF16) return gemv_gm<M, YSCV_HIP_BF16>(a, grid, gm, sf16, s);
  return gemv_gm<M, YSCV_HIP_F16>(a, grid, gm, sf16, s);
}

}  // namespace

bool int4_gemv_takes(const yscv_hip_int4_weight *w, const void *x, int x_dtype, size_t m, int num_cus) {
  if (!w->tiled || m < 1 || m > 4 || (reinterpret_cast<uintptr_t>(x) & 15) != 0 || w->k % 32 != 0) return false;
  if (w->n >= ((size_t)1 << 31) || w->k >= ((size_t)1 << 30)) return false;
  const GemvRows rows = x_dtype == YSCV_HIP_F32 ? GEMV_F32 : (x_dtype == YSCV_HIP_BF16 ? GEMV_BF16 : GEMV_F16);
  return gemv_pays(m, rows, w->has_zp, gemv_shape(w->ktp, w->nt, m), num_cus);
}

int32_t launch_int4_gemv(const yscv_hip_int4_weight *w, const void *x, int x_dtype, void *y, int y_dtype, size_t m, int epi,
                         const NormFold *nf, int num_cus, hipStream_t s) {
  if (epi == EPI_ADD_F32 && y_dtype != YSCV_HIP_F32)
    return set_error(YSCV_HIP_ERR_INVALID_ARG, "residual accumulation needs an f32 output");
  if (epi == EPI_SWIGLU && (w->n & 1)) return set_error(YSCV_HIP_ERR_INVALID_ARG, "SwiGLU epilogue needs an even row count");
  GemvRowArgs a = {};
  a.tiles = w->tiles;
  a.tscales = w->tscales;
  a.tzps = w->has_zp ? w->tzps : nullptr;
  a.x = x;
  a.y = y;
  a.m = (int)m;
  a.n = (int)w->n;
  a.k = (int)w->k;
  a.nt = (int)w->nt;
  a.ktp = (int)w->ktp;
  a.chunks = (int)w->chunks;
  a.chunk_div = w->gm == GM128 ? (int)(w->g / 128) : 1;
  const GemvShape g = gemv_shape(w->ktp, w->nt, m);
  a.slices = g.slices;
  a.split_log2 = g.split_log2;
  a.groups = g.groups;
  a.y_dtype = y_dtype;
  a.epi = epi;
  if (nf && nf->ss_in) {
    if (nf->ss_in_count < 1 || nf->ss_in_count > 256 || !nf->pre_in)
      return set_error(YSCV_HIP_ERR_INVALID_ARG, "folded norm: %d partial sums of the row", nf->ss_in_count);
    a.ss_in = nf->ss_in;
    a.pre_in = nf->pre_in;
    a.pre_next = nf->pre_next;
    a.ss_in_count = nf->ss_in_count;
    a.ss_in_stride = nf->ss_in_stride;
    a.inv_d = nf->inv_d;
    a.eps = nf->eps;
  }
  if (nf && nf->xg) {
    if (epi != EPI_ADD_F32 || !nf->gamma_next || !nf->ss_out || !nf->ss_out_count || !nf->pre || nf->ss_out_stride < (int)w->nt)
      return set_error(YSCV_HIP_ERR_INVALID_ARG, "folded norm: the producing call is a residual update with gamma and a place for the sums");
    a.gamma_next = nf->gamma_next;
    a.pre = nf->pre;
    a.xg = nf->xg;
    a.ss_out = nf->ss_out;
    a.ss_out_stride = nf->ss_out_stride;
    *nf->ss_out_count = (int)w->nt;
  }
  unsigned grid = (unsigned)a.groups;
  if (a.slices <= 8) {
    // Groups of a workgroup, where it may have several.  From 16 per CU, as many as keep all workgroups on the chip together:
    // 128256 x 4096 58.6 us with f32 activations and 51.6 with fp16, one group each 67.9 and 54.4.  Below that the 16-bit types are
    // best with one (28672 x 4096 14.0 against 14.8 us, 151936 x 1024 15.8 against 17.1), and f32, which splits its activations anew in
    // each workgroup, with two (16.2 against 16.9, 18.5 against 20.0) once there are more than four per CU.
    const int rounds = a.groups >= 16 * num_cus ? (a.groups + 2 * num_cus - 1) / (2 * num_cus)
                                                : (x_dtype == YSCV_HIP_F32 && a.groups > 4 * num_cus ? 2 : 1);
    grid = (unsigned)((a.groups + rounds - 1) / rounds);
  }
  a.wgs = (int)grid;
  const bool sf16 = w->scale_dtype == YSCV_HIP_F16;
  if (m == 1) return gemv_xd<1>(a, grid, x_dtype, w->gm, sf16, s);
  if (m == 2) return gemv_xd<2>(a, grid, x_dtype, w->gm, sf16, s);
  return gemv_xd<4>(a, grid, x_dtype, w->gm, sf16, s);
}

}  // namespace yscv
