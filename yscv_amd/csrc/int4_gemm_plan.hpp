// Which tiles the int4 GEMMs of more than 16 rows take (int4_gemm_ring.hip, int4_gemm_wide.hip).  Host code only, without the
// HIP headers.
#pragma once

#include <cstddef>

namespace yscv {

constexpr size_t plan_ceil_div(size_t a, size_t b) { return (a + b - 1) / b; }

// Tiles of int4_gemm_wide.hip, rows x columns; a plan names them kWide + tile
enum : int { WIDE_256x256 = 0, WIDE_256x192, WIDE_128x256, WIDE_128x192, WIDE_TILES };
constexpr int kWide = 16;

// Column blocks of 16 of the 256-row tile shapes 5, 6, 7 below, and for which kinds of weight ring_plan counts with them.
constexpr int wide_tile_blocks(int shape) { return 16 - 2 * (shape - 5); }
constexpr bool wide_tile_built(int gm, bool has_zp, int blocks) {
  return blocks == 16 || blocks == 12 || (blocks == 14 && !(gm == 0 && has_zp));
}

// Tile shapes: 0 = 128 x 128, 1 = 128 x 256, 2 = 256 x 128 (m > 128), 3 = 32 x 128 (m <= 32), 4 = 64 x 128 (m <= 64),
// 5, 6, 7 = 256 x 256, 256 x 224, 256 x 192 (m > 256).  The ring kernel has 0, 3 and 4; where the others are the cheapest, int4_plan names
// tiles of int4_gemm_wide.hip
struct RingPlan {
  int one;           // shape of the launch, or of the first of two launches
  int second;        // < 0: one launch; else the shape of the launch that takes the columns from split_col on
  size_t split_col;
  int splits, kt_per;  // K split of a single launch (splits == 1: none)
};

// gm: the weight's scales_per_chunk class (GM32 = 0 ...); has_zp: it has zero points
inline RingPlan ring_plan(size_t m, size_t n, size_t kt, size_t cus, int gm, bool has_zp) {
  RingPlan pl{0, -1, 0, 1, (int)kt};
  size_t tiles;
  if (m <= 32) {
    // The tile height follows m: the MFMA work of a workgroup, and with it the time a weight tile stays in LDS, is
    // proportional to the tile's rows whether they exist or not, so a short m streams the weights faster on a
    // 32- or 64-row tile.
    pl.one = 3;
    tiles = plan_ceil_div(n, (size_t)128);
  } else if (m <= 64) {
    pl.one = 4;
    tiles = plan_ceil_div(n, (size_t)128);
  } else {
    // Larger tiles: 128 x 256 (a third fewer fragment reads per MFMA) and 256 x 128 (the same, and every decoded
    // weight feeds twice as many MFMAs).  A workgroup needs about 1.72 / 1.63 times as long for them as for a
    // 128 x 128 tile; they pay when the tiles come in rounds over the CUs and the larger ones need sufficiently fewer
    // rounds.  When the last round of the best shape would leave most CUs idle, the columns of its whole rounds go to
    // one launch and the rest to a second one with the shape that suits the rest (2048 rows x 14336 columns in 256 x 128
    // tiles: three rounds, then one round of 128 x 128 tiles, instead of three and a half).
    struct Shape {
      size_t bm, bn, cost;
      int code;
    };
    // cost: time of one tile in hundredths of a 128 x 128 tile's (measured on K 4096: 40 us; the 64-row tile 30 us).
    // The 64-row tile decodes every weight twice as often per MFMA; it pays where it fills CUs that the taller tiles
    // would leave idle (512 rows against N 4096: 256 tiles instead of 128).
    // The 256 x 256 tile of int4_gemm_wide.hip takes 110 us where two rounds of 256 x 128 tiles take 138 (weights without
    // zero points; with them its gain depends on the clock, see its header).
    const Shape shapes[7] = {{128, 128, 100, 0}, {128, 256, 172, 1}, {256, 128, 163, 2}, {256, 256, 280, 5}, {256, 224, 250, 6}, {256, 192, 225, 7},
                             {64, 128, 75, 4}};
    auto allowed = [&](const Shape &sh) {
      return sh.code == 2 ? m > 128 : (sh.code >= 5 ? m > 256 && wide_tile_built(gm, has_zp, wide_tile_blocks(sh.code)) : true);
    };
    // Where the rows of the output come in no whole float4 the epilogue of the 256-row tiles stores element by element, in as many
    // instructions for 12 or 14 column blocks as for 16: some 4 us of a 192-column tile that its table entry does not hold, counted at
    // this K (1024 x 8874 x 768: 34.0 us in 128-row tiles, 36.6 in 192 columns; K 4096 94.6 and 91.9; 585 x 14891 x 544 35.1 and 39.6).
    const size_t scalar = n % 4 != 0 ? 352 / (kt > 0 ? kt : 1) : 0;
    auto cost_of = [&](const Shape &sh) { return sh.cost + (sh.code == 7 ? scalar : (sh.code == 6 ? scalar / 2 : 0)); };
    // best single shape for columns [c0, n): cost of its rounds over the CUs
    auto best_single = [&](size_t c0, int *which, size_t *tiles_out) {
      size_t best = (size_t)-1;
      for (const Shape &sh : shapes) {
        if (!allowed(sh)) continue;
        const size_t t = plan_ceil_div(m, sh.bm) * plan_ceil_div(n - c0, sh.bn);
        const size_t cost = plan_ceil_div(t, cus) * cost_of(sh);
        if (cost < best) {
          best = cost;
          *which = sh.code;
          *tiles_out = t;
        }
      }
      return best;
    };
    size_t best = best_single(0, &pl.one, &tiles);
    const size_t launch_cost = 10;  // a second launch: about a tenth of a tile time
    for (int i = 0; i < 6; i++) {
      if (!allowed(shapes[i])) continue;
      const size_t tm = plan_ceil_div(m, shapes[i].bm), tn = plan_ceil_div(n, shapes[i].bn);
      const size_t rounds = tm * tn / cus;    // whole rounds
      const size_t cols = rounds * cus / tm;  // whole tile columns inside them
      if (rounds == 0 || cols == 0 || cols >= tn) continue;
      int rest = 0;
      size_t rest_tiles = 0;
      const size_t cost =
          plan_ceil_div(tm * cols, cus) * cost_of(shapes[i]) + best_single(cols * shapes[i].bn, &rest, &rest_tiles) + launch_cost;
      if (cost < best) {
        best = cost;
        pl.one = shapes[i].code;
        pl.second = rest;
        pl.split_col = cols * shapes[i].bn;
      }
    }
    if (pl.second >= 0) return pl;
  }
  // K split: a shape whose tiles cover at most half the CUs is cut along k, each part with at least four 128-k tiles
  // (eight stages), as long as the f32 partial sums stay within 16 MB and, together with a prepared fp16 copy of the
  // activations, within 31 MB (they travel in the caller's workspace; yscv_hip_int4_matmul_static has 32 MB for
  // both).  The number of splits is the one with the shortest estimated time, rounds over the CUs x (a part's k-tiles at
  // 0.9 us each + 5 us to start and end a workgroup), + 5 us for the kernel that adds the parts.
  if (tiles * 2 <= cus && kt >= 8) {
    size_t best_ks = 1, best_t = kt * 18 + 100;  // units of 0.05 us
    const size_t x_bytes = m * kt * 128 * 2;
    const size_t room = x_bytes >= ((size_t)31 << 20) ? 0 : ((size_t)31 << 20) - x_bytes;
    const size_t cap = room < ((size_t)16 << 20) ? room : ((size_t)16 << 20);
    for (size_t ks = 2; ks <= 16 && ks <= kt / 4; ks++) {
      if (ks * m * n * sizeof(float) > cap) break;
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
  }
  return pl;
}

// us that rounds of one kind of tile take over the CUs, `kt` 128-k tiles deep: whole rounds at the clock that all CUs busy leave, a
// last round that fills a part of them at a higher one (the card holds its power, not its clock: 64 stages of a 256 x 256 tile take
// 91 us on 256 CUs, 68 on 32), but never below what one tile takes.
struct TileTime {
  size_t bm, bn;
  double full_fixed, full_kt, fast_fixed, fast_kt;
};
inline double tile_rounds_us(const TileTime &t, size_t tiles, size_t kt, size_t cus) {
  const double full = t.full_fixed + t.full_kt * (double)kt, fast = t.fast_fixed + t.fast_kt * (double)kt;
  const size_t rest = tiles % cus;
  const double last = rest == 0 ? 0.0 : (full * (double)rest / (double)cus > fast ? full * (double)rest / (double)cus : fast);
  return (double)(tiles / cus) * full + last;
}
// fitted to 128 .. 2048 rows, N 2049 .. 28672, K 1024 and 4096, fp16 rows, groups of 32; the ring kernel's tiles of 128 and 64 rows for
// comparison
constexpr TileTime kWideTime[WIDE_TILES] = {
    {256, 256, 8.0, 2.90, 5.5, 2.12}, {256, 192, 5.5, 2.34, 4.5, 1.74}, {128, 256, 5.5, 1.56, 4.5, 1.25}, {128, 192, 4.8, 1.52, 4.2, 1.06}};
constexpr TileTime kRingTime[2] = {{128, 128, 1.5, 1.06, 1.5, 1.06}, {64, 128, 1.5, 0.76, 1.5, 0.76}};

// The plan of a launch: ring_plan's, or tiles of int4_gemm_wide.hip where their estimated time is shorter.  From 65 rows on (a
// 128-row tile decodes a weight once for all of them; the 64-row ring tile is half of one).  us of the op, ring plan -> this one, fp16
// rows, groups of 32: 2048 x 4096 x 4096 71 -> 58, 2048 x 8192 x 4096 108 -> 100, 512 x 14336 x 4096 66 -> 53, 150 x 28672 x 4096 64 ->
// 53, 700 x 5632 x 4096 56 -> 42; 128 x 28672 x 4096 43 -> 39.
inline RingPlan int4_plan(size_t m, size_t n, size_t kt, size_t cus, int gm, bool has_zp) {
  RingPlan ring = ring_plan(m, n, kt, cus, gm, has_zp);
  if (m <= 64) return ring;
  constexpr double kSecondLaunch = 1.0, kSumLaunch = 5.5;  // us
  auto tiles_of = [&](const TileTime &t, size_t cols) { return plan_ceil_div(m, t.bm) * plan_ceil_div(cols, t.bn); };
  auto sum_us = [&](size_t parts) { return kSumLaunch + (double)(parts * m * n * 8) / 4e6; };  // partial products out and in
  double best = 1e30;
  // (its larger tiles and its second launches never beat these)
  if ((ring.one == 0 || ring.one == 4) && ring.second < 0) {
    const TileTime &t = ring.one == 0 ? kRingTime[0] : kRingTime[1];
    best = tile_rounds_us(t, tiles_of(t, n) * (size_t)ring.splits, (size_t)ring.kt_per, cus) + (ring.splits > 1 ? sum_us((size_t)ring.splits) : 0.0);
  }
  RingPlan pl = ring;
  const size_t x_bytes = m * kt * 128 * 2, cap = x_bytes >= ((size_t)31 << 20) ? 0 : (((size_t)31 << 20) - x_bytes < ((size_t)16 << 20) ? ((size_t)31 << 20) - x_bytes : (size_t)16 << 20);
  for (int i = 0; i < WIDE_TILES; i++) {
    const TileTime &t = kWideTime[i];
    const size_t tiles = tiles_of(t, n);
    auto take = [&](double us, const RingPlan &p) {
      if (us < best) {
        best = us;
        pl = p;
      }
    };
    take(tile_rounds_us(t, tiles, kt, cus), RingPlan{kWide + i, -1, 0, 1, (int)kt});
    // K cut over workgroups: under a round of tiles, parts of at least four 128-k tiles, the same bounds on scratch as the ring plan's
    for (size_t parts = 2; tiles < cus && parts <= 16 && parts <= kt / 4 && parts * m * n * sizeof(float) <= cap; parts++) {
      const size_t per = plan_ceil_div(kt, parts), used = plan_ceil_div(kt, per);
      if (used == parts) take(tile_rounds_us(t, tiles * parts, per, cus) + sum_us(parts), RingPlan{kWide + i, -1, 0, (int)parts, (int)per});
    }
    // the columns of whole rounds, and the rest in the tiles that suit it
    const size_t tm = plan_ceil_div(m, t.bm), cols = tiles / cus * cus / tm;
    if (cols == 0 || cols * t.bn >= n) continue;
    const double whole = tile_rounds_us(t, tm * cols, kt, cus) + kSecondLaunch;
    for (int j = 0; j < WIDE_TILES; j++)
      take(whole + tile_rounds_us(kWideTime[j], tiles_of(kWideTime[j], n - cols * t.bn), kt, cus), RingPlan{kWide + i, kWide + j, cols * t.bn, 1, (int)kt});
  }
  return pl;
}

}  // namespace yscv
