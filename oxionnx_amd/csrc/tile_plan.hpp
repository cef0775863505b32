// The block tile and the K slices of a contraction on the MFMA engine, by
// estimated time.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace ohip {

// Tile ids that name one unsplit block tile (launch.hpp); 10 and 11 force
// split-K on the 64x64 / 128x128 (eight-wave) tile.
inline bool plain_tile_id(int t) { return (t >= 1 && t <= 9) || (t >= 12 && t <= 14) || t == 16 || t == 18; }
// OHIP_SPLITS=n (2..16) forces that many split-K slices wherever a split
// plan is made (a measurement switch)
inline int forced_splits() {
  static const int v = [] {
    const char* e = std::getenv("OHIP_SPLITS");
    const int n = e ? std::atoi(e) : 0;
    return n >= 2 && n <= 16 ? n : 0;
  }();
  return v;
}

// A block tile and the K slices it runs with (splits > 1: tile 10 or 11);
// us: its estimated time without the launch (0: a forced plan, not estimated).
struct TilePlan {
  int splits, tile;
  float us = 0.0f;
};

// What a block of a tile costs, in us: a stage of 128 bytes of K when its CU
// is not short of bandwidth or MFMA rate (lat), a stage's share of the CU
// when it is (bw: n resident blocks take max(lat, n * bw) a stage), and
// everything outside the K loop (fix).  res: blocks a CU holds (LDS).
struct TileCost {
  int id, bp, bq, res;
  float lat, bw, fix;
};
// The reduction of `s` slices of `mb` MB of partial sums in all.
struct ReduceCost {
  float fix, per_mb, per_slice;
};
enum class PlanKind { Dense, DenseF32, Conv };   // f16 / bf16 / int8 rows; f32 of any loader; im2col rows

// The tile and the split of a contraction P x Q (x batch) over kc 16-byte
// chunks, by the cost of every candidate.  The tiles' constants are a
// least-squares fit to 178 shapes (M 12-4096, K 64-16384, N 64-11008; 1x1-5x5
// convolutions of 7-112 pixels; f16, f32, int8) timed on every tile, graph
// replay, and so are the slices of the 16-bit and int8 convolutions (their
// reduction's launch also costs the host about 1.5 us, which is in its fixed
// term whether or not a host waits: a capture has to plan as the eager call
// before it did, for the same scratch and the same bits).  The slices of the
// other kinds are fitted to 244 products of 33-1500 rows timed on 2-16 slices,
// eager and by replay (their mean), by the loss of the choice: 0.3 % in the
// mean for f32 (4 % at most), 0.9 % for f16 (10 %) and 1.7 % for int8 (9 %).
// Every count up to ten is a candidate there: 48 blocks of f32 200x2048x768
// fill a round with five slices (16.7 us; four 18.3, six 19.5).  Against rules
// on the number of blocks: f16 1024x1024x768 13.7 -> 9.0 us (split, now
// unsplit), 1500x1024x2048 18.0 -> 12.7, 838x2688x2880 37 -> 24.
// Grids of a round of 256x256 tiles and a long K take tile 16 outright: its
// advantage there is the clock and the cache, which the stages' cost does
// not show (4096x4096x11008 f16 291 us against 324 on tiles 3, 4 and 18).
// A convolution's tile 1 is charged 0.5 us a round above its fit: the fit's
// replays find every operand in the cache, a forward's convolution does not,
// and two LDS stages hide less of that than tile 9's four.  (Seen on 512 blocks
// of one generator's 3x3 stride-2 f16 convolution: 11.7 us on tile 1, 10.4 on
// 9.  24 other unsplit convolutions by replay: f16 0-6 % faster on tile 9, int8
// 3-5 % faster on tile 1, which the charge costs them.)
// The split is symmetric in P and Q (a convolution splits alike in NCHW and
// NHWC output), so it is chosen without the one tile that is not square or
// paired, 18 (whose 4-byte outputs do not fit its stage buffers: wide_out).
inline TilePlan plan_tiles(PlanKind kind, int P, int Q, int kc, int override_tile, int batch = 1,
                           bool wide_out = false, bool may_split = true) {
  static constexpr TileCost kDense[] = {{1, 64, 64, 4, .342f, .215f, .50f},   {9, 64, 64, 2, .287f, .178f, .78f},
                                        {8, 128, 128, 2, .519f, .340f, 1.10f}, {12, 128, 128, 1, .373f, .373f, 1.93f},
                                        {2, 128, 128, 1, .349f, .349f, 2.50f}, {3, 256, 128, 1, .475f, .475f, 2.80f},
                                        {4, 128, 256, 1, .475f, .475f, 2.80f}, {16, 256, 256, 1, .902f, .887f, 4.36f},
                                        {18, 192, 256, 1, .787f, .733f, 3.27f}};
  static constexpr TileCost kF32[] = {{1, 64, 64, 4, .664f, .571f, .53f},     {9, 64, 64, 2, .654f, .565f, .98f},
                                      {8, 128, 128, 2, 1.80f, 1.92f, 1.65f},  {12, 128, 128, 1, 2.04f, 2.04f, 1.68f},
                                      {3, 256, 128, 1, 3.47f, 3.47f, 2.25f},  {4, 128, 256, 1, 3.47f, 3.47f, 2.25f},
                                      {16, 256, 256, 1, 7.09f, 7.09f, 7.69f}};
  static constexpr TileCost kConv[] = {{1, 64, 64, 4, .522f, .234f, 1.17f},   {9, 64, 64, 2, .386f, .254f, 1.17f},
                                       {8, 128, 128, 2, .633f, .403f, 1.56f}, {12, 128, 128, 1, .510f, .510f, 2.15f},
                                       {3, 256, 128, 1, .708f, .708f, 4.0f},  {4, 128, 256, 1, .708f, .708f, 4.0f}};
  const ReduceCost red = kind == PlanKind::Dense      ? ReduceCost{1.5f, .50f, .14f}
                         : kind == PlanKind::DenseF32 ? ReduceCost{2.0f, .40f, .14f}
                                                      : ReduceCost{1.21f + 1.5f, .321f, .121f};
  const TileCost* tab = kind == PlanKind::Dense ? kDense : kind == PlanKind::DenseF32 ? kF32 : kConv;
  const int ntab = kind == PlanKind::Dense      ? (int)(sizeof(kDense) / sizeof(TileCost))
                   : kind == PlanKind::DenseF32 ? (int)(sizeof(kF32) / sizeof(TileCost))
                                                : (int)(sizeof(kConv) / sizeof(TileCost));
  const int64_t nk = std::max<int64_t>(1, ((int64_t)kc + 7) / 8);
  // How many of `s` slices have stages: the kernels give each ceil(nk / s), so
  // the last of 6 slices of 10 stages would only write zeros for the reduction
  // to read.  As many slices as that are as short.
  auto filled = [&](int s) {
    const uint32_t per = ((uint32_t)nk + s - 1) / s;
    return (int)(((uint32_t)nk + per - 1) / per);
  };
  if (plain_tile_id(override_tile)) return {1, override_tile};
  if (override_tile != 0 && override_tile != 10 && override_tile != 11) {   // a forced path that does not apply here
    override_tile = 0;
    may_split = false;
  }
  if (forced_splits()) return {may_split ? forced_splits() : 1, override_tile ? override_tile : may_split ? 10 : 9};
  if (override_tile != 0)
    return {may_split ? std::max(2, filled((int)std::min<int64_t>(16, nk / 2 > 0 ? nk / 2 : 1))) : 1,
            may_split ? override_tile : override_tile == 11 ? 8 : 9};
  auto blocks = [&](int bp, int bq) {
    return (int64_t)(((uint32_t)P + (uint32_t)bp - 1) / (uint32_t)bp) * (((uint32_t)Q + (uint32_t)bq - 1) / (uint32_t)bq) *
           batch;
  };
  auto time = [&](const TileCost& t, int64_t nb, int64_t stages) {
    const uint32_t ncu = (uint32_t)std::min<int64_t>((nb + 255) >> 8, 1 << 24), res = (uint32_t)t.res;
    const uint32_t q = ncu >> (res >> 1), rem = ncu & (res - 1);   // (res is 1, 2 or 4)
    return t.fix * (float)(q + (rem ? 1 : 0)) +
           (float)stages * ((float)q * std::max(t.lat, (float)t.res * t.bw) + (rem ? std::max(t.lat, (float)rem * t.bw) : 0.0f));
  };
  if (nk > 16 && blocks(256, 256) >= 256)   // (the convolutions' table has no tile 16: the dense cost)
    return {1, 16, time(kind == PlanKind::DenseF32 ? kF32[6] : kDense[7], blocks(256, 256), nk)};
  TilePlan best{1, 1};
  float cost = INFINITY;
  for (int i = 0; i < ntab; ++i) {
    const TileCost& t = tab[i];
    if (t.id == 18) continue;
    if (wide_out && kind == PlanKind::Dense && t.bp * t.bq > 128 * 128) continue;   // unstaged 4-byte outputs
    const int64_t nb = blocks(t.bp, t.bq);
    const float c = time(t, nb, nk);
    if (c < cost) { cost = c; best = {1, t.id}; }
  }
  // Few stages: a reduction's launch costs a waiting host more than the slices
  // gain (f16 165x768x128 eager 7.2 us, 8.4 in four slices; of a batch, which a
  // transposing launch precedes, f32 5 x 16x238x180 14.6 and 16.1; staged f16
  // convolutions 2x32x8x8 -> 144 5x5 12.6 and 14.1)
  const bool split = may_split && cost >= (kind == PlanKind::Conv ? 6.3f : 4.6f);
  const float launch = kind != PlanKind::Conv && batch > 1 ? 1.0f : 0.0f;
  for (int i = 0; split && i < ntab; ++i) {
    const TileCost& t = tab[i];
    if (t.id != 9 && t.id != 8) continue;
    const int64_t nb = blocks(t.bp, t.bq);
    const float mb = (float)P * (float)Q * (float)batch * 4e-6f;
    // (each count a constant: small eager calls wait for this)
    auto slices = [&](auto count) {
      constexpr uint32_t most = decltype(count)::value;
      const uint32_t per = ((uint32_t)nk + most - 1) / most;
      if (per < 2) return false;
      const int s = per * (most - 1) < (uint32_t)nk ? (int)most : filled(most);
      const float cs = time(t, nb * s, per) + red.fix + launch + red.per_slice * (float)s + red.per_mb * mb * (float)s;
      if (cs < cost) { cost = cs; best = {s, t.id == 9 ? 10 : 11}; }
      return true;
    };
    auto all = [&](auto... count) { (void)(slices(count) && ...); };
    using std::integral_constant;
    if (kind == PlanKind::Conv)
      all(integral_constant<int, 2>{}, integral_constant<int, 3>{}, integral_constant<int, 4>{}, integral_constant<int, 6>{},
          integral_constant<int, 8>{}, integral_constant<int, 12>{}, integral_constant<int, 16>{});
    else
      all(integral_constant<int, 2>{}, integral_constant<int, 3>{}, integral_constant<int, 4>{}, integral_constant<int, 5>{},
          integral_constant<int, 6>{}, integral_constant<int, 7>{}, integral_constant<int, 8>{}, integral_constant<int, 9>{},
          integral_constant<int, 10>{}, integral_constant<int, 12>{}, integral_constant<int, 14>{},
          integral_constant<int, 16>{});
  }
  if (best.splits == 1 && kind == PlanKind::Dense && !wide_out) {
    const TileCost& t = kDense[ntab - 1];
    const float c = time(t, blocks(t.bp, t.bq), nk);
    if (c < cost) { cost = c; best.tile = t.id; }
  }
  best.us = cost;
  return best;
}

// Rows up to which Gemm may run GEMV, and the skinny kernel (skinny.hip).
constexpr int kMaxGemvM = 8;
constexpr int kMaxSkinnyM = 32;
// Whether a few rows of a product with n weight rows of kc chunks run the
// skinny kernel instead of GEMV (up to kMaxGemvM) or the engine (its plan),
// by estimated times in us past the launch.  The skinny kernel's waves walk K
// in steps of 256 chunks a block, at the memory's rate if that is slower; the
// blocks of 16 weight rows each read the activations again, and a second
// activation tile (over 16 rows) costs every weight byte more.  GEMV reads the
// activations again for every weight row or two.  Rows that GEMV or the engine
// would pack first cost them a launch (2.5), and 16-bit rows at odd addresses
// (not whole dwords) cost the skinny kernel's loads (8x3787x512 f16 10.6 us, 7.4
// at K = 3788; 23x3787x1658 20.3 against 13.0 packed); the engine's unsplit plans are
// 2 us slower at so few rows than at those its fit saw.  Fitted to 21 weights
// of 256-70001 rows and 512-25088 columns at 2-32 rows, f16 and f32 (graph
// replay), where both sides were timed: the choice is within 0.4 % of the
// faster one in the mean, 1.2x at most (3.3 % and 1.57x without the activations'
// terms: f16 32x4096x11008 36 us against 23 on the engine, 24x2048x8192 13.3
// against 11.7).  5x768x3072 f16 6.6 -> 4.2 us, 8x4096x4096 36 -> 9.6, 9x4096x11008
// 25.8 -> 21.5, f32 16x4096x4096 26 -> 21; 5x25088x512 f16 stays GEMV (11.3
// against 34: 32 blocks).
inline bool skinny_wins(bool f32, int64_t m, int64_t n, int64_t kc, bool pack, bool odd, const TilePlan& engine) {
  const float steps = (float)((kc + 31) / 32), mb = (float)n * (float)kc * 16e-6f, rows = (float)m;
  const float acts = (float)((n + 15) / 16) * (float)kc * rows * 16e-6f;   // MB
  const float step = f32 ? .29f + .0125f * rows : .25f + .0115f * rows;
  const float rate = f32 ? (steps >= 8.0f ? 5.4f : 4.2f) : steps >= 16.0f ? 6.5f : steps >= 8.0f ? 5.4f : 4.6f;   // MB a us
  const float skinny =
      std::max(step * steps, mb / rate) + acts * (f32 ? .01f : m > kMaxGemvM ? .05f : 0.0f) + (m > 16 ? mb * (f32 ? .2f : .12f) : 0.0f) +
      (odd ? .028f * steps * rows : 0.0f);
  const float other = m <= kMaxGemvM ? mb / 7.0f + rows * (.33f + (f32 ? .02f : m <= 2 ? .018f : .04f) * mb)
                                     : engine.us + (engine.splits == 1 ? 2.2f : 1.5f);
  return skinny < other + (pack ? 2.5f : 0.0f);
}

}  // namespace ohip
