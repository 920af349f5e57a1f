// Which tiles the int4 GEMMs of more than 16 rows take (int4_gemm_ring.hip, int4_gemm_wide.hip).  Host code only, without the
// HIP headers.
#pragma once

#include <cstddef>

namespace yscv {

constexpr size_t plan_ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }

// Tiles, rows x columns: of int4_gemm_ring.hip, and from kWide on of int4_gemm_wide.hip
enum : int { RING_128x128 = 0, RING_32x128, RING_64x128, kWide = 16 };
enum : int { WIDE_256x256 = 0, WIDE_256x192, WIDE_128x256, WIDE_128x192, WIDE_TILES };

struct GemmPlan {
  int one;           // tile of the launch, or of the first of two launches
  int second;        // < 0: one launch; else the tile of the launch that takes the columns from split_col on
  size_t split_col;
  int splits, kt_per;  // K split of a single launch (splits == 1: none): parts of kt_per 128-k tiles
};

// f32 partial products of a K split travel in the caller's workspace: at most 16 MB of them, and 31 MB together with a prepared fp16 copy
// of the activations (yscv_hip_int4_matmul_static has 32 MB for both).
inline size_t plan_partial_cap(size_t m, size_t kt) {
  const size_t x_bytes = m * kt * 128 * 2, all = (size_t)31 << 20, most = (size_t)16 << 20;
  const size_t room = x_bytes >= all ? 0 : all - x_bytes;
  return room < most ? room : most;
}

// Up to 64 rows.  The tile height follows m: the MFMA work of a workgroup, and with it the time a weight tile stays in LDS, is
// proportional to the tile's rows whether they exist or not, so a short m streams the weights faster on a 32- or 64-row tile.
// Tiles that cover at most half the CUs are cut along K, each part with at least four 128-k tiles (eight stages): the number of parts
// with the shortest estimated time, rounds over the CUs x (a part's k-tiles at 0.9 us each + 5 us to start and end a workgroup), + 5 us for
// the kernel that adds the parts.
inline GemmPlan short_plan(size_t m, size_t n, size_t kt, size_t cus) {
  GemmPlan pl{m <= 32 ? RING_32x128 : RING_64x128, -1, 0, 1, (int)kt};
  const size_t tiles = plan_ceil_div(n, (size_t)128);
  if (tiles * 2 > cus || kt < 8) return pl;
  size_t best_ks = 1, best_t = kt * 18 + 100;  // units of 0.05 us
  for (size_t ks = 2; ks <= 16 && ks <= kt / 4 && ks * m * n * sizeof(float) <= plan_partial_cap(m, kt); ks++) {
    const size_t t = plan_ceil_div(tiles * ks, cus) * (plan_ceil_div(kt, ks) * 18 + 100) + 100;
    if (t < best_t) {
      best_t = t;
      best_ks = ks;
    }
  }
  if (best_ks >= 2) {
    pl.kt_per = (int)plan_ceil_div(kt, best_ks);
    pl.splits = (int)plan_ceil_div(kt, (size_t)pl.kt_per);
  }
  return pl;
}

// us that rounds of one kind of tile take over the CUs, `kt` 128-k tiles deep: whole rounds at the clock that all CUs busy leave, a
// last round that fills a part of them at a higher one (the card holds its power, not its clock: 64 stages of a 256 x 256 tile take
// 91 us on 256 CUs, 68 on 32), but never below what one tile takes.
struct TileTime {
  int tile;
  size_t bm, bn;
  double full_fixed, full_kt, fast_fixed, fast_kt;
};
inline double tile_rounds_us(const TileTime &t, size_t tiles, size_t kt, size_t cus) {
  const double full = t.full_fixed + t.full_kt * (double)kt, fast = t.fast_fixed + t.fast_kt * (double)kt;
  const size_t rest = tiles % cus;
  const double last = rest == 0 ? 0.0 : (full * (double)rest / (double)cus > fast ? full * (double)rest / (double)cus : fast);
  return (double)(tiles / cus) * full + last;
}
// Fitted to the times of every tile, with K whole and cut, and of every pair of them, at 790 shapes: 65 .. 2048 rows, N 256 .. 125 000, K
// 512 .. 14 000, fp16 rows.  The plan is 1.2 % slower than the fastest candidate on average there, 20 % at most (with the costs of the ring
// tiles larger than 128 x 128 in front, as it was: 3.7 %, 44 %).
constexpr TileTime kTileTime[] = {{kWide + WIDE_256x256, 256, 256, 8.7, 2.73, 10.6, 2.59}, {kWide + WIDE_256x192, 256, 192, 5.8, 2.27, 10.1, 1.98},
                                  {kWide + WIDE_128x256, 128, 256, 3.8, 1.59, 8.1, 1.38},  {kWide + WIDE_128x192, 128, 192, 2.6, 1.21, 7.5, 1.13},
                                  {RING_128x128, 128, 128, 4.9, 0.96, 7.5, 0.90},          {RING_64x128, 64, 128, 3.5, 0.66, 5.8, 0.67}};

// The plan of a launch.  Above 64 rows the shortest estimated time of every tile there is, in one launch, with K cut over workgroups, or
// (the wide tiles) with the columns of whole rounds in one launch and the rest in the tiles that suit it.  us of the op, the LDS-ring GEMM
// with tiles of up to 256 x 128 -> this, fp16 rows, groups of 32: 2048 x 4096 x 4096 71 -> 58, 2048 x 8192 x 4096 108 -> 100, 512 x
// 14336 x 4096 66 -> 53, 150 x 28672 x 4096 64 -> 53, 700 x 5632 x 4096 56 -> 42; 128 x 28672 x 4096 43 -> 39.
inline GemmPlan int4_plan(size_t m, size_t n, size_t kt, size_t cus) {
  if (m <= 64) return short_plan(m, n, kt, cus);
  constexpr double kSumLaunch = 3.2;  // us (a second launch costs nothing that shows)
  auto tiles_of = [&](const TileTime &t, size_t cols) { return plan_ceil_div(m, t.bm) * plan_ceil_div(cols, t.bn); };
  auto sum_us = [&](size_t parts) { return kSumLaunch + (double)(parts * m * n * 8) / 5e6; };  // partial products out and in
  double best = 1e30;
  GemmPlan pl{};
  auto take = [&](double us, const GemmPlan &p) {
    if (us < best) {
      best = us;
      pl = p;
    }
  };
  const size_t cap = plan_partial_cap(m, kt);
  for (const TileTime &t : kTileTime) {
    const size_t tiles = tiles_of(t, n);
    take(tile_rounds_us(t, tiles, kt, cus), GemmPlan{t.tile, -1, 0, 1, (int)kt});
    // K cut over workgroups: under a round of tiles, parts of at least four 128-k tiles
    for (size_t parts = 2; tiles < cus && parts <= 16 && parts <= kt / 4 && parts * m * n * sizeof(float) <= cap; parts++) {
      const size_t per = plan_ceil_div(kt, parts), used = plan_ceil_div(kt, per);
      if (used == parts) take(tile_rounds_us(t, tiles * parts, per, cus) + sum_us(parts), GemmPlan{t.tile, -1, 0, (int)parts, (int)per});
    }
    // the columns of whole rounds, and the rest in the tiles that suit it
    const size_t tm = plan_ceil_div(m, t.bm), cols = tiles / cus * cus / tm;
    if (t.tile < kWide || cols == 0 || cols * t.bn >= n) continue;
    const double whole = tile_rounds_us(t, tm * cols, kt, cus);
    for (const TileTime &u : kTileTime)
      if (u.tile >= kWide) take(whole + tile_rounds_us(u, tiles_of(u, n - cols * t.bn), kt, cus), GemmPlan{t.tile, u.tile, cols * t.bn, 1, (int)kt});
  }
  return pl;
}

}  // namespace yscv
