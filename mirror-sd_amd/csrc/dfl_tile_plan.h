// Host-side planning of the tile GEMM (dfl_tile.hip): the workgroup tile shape of an
// M x N x K product and its LDS size.  Pure host code, so a host test can check plans
// without a GPU.
#pragma once

#include <algorithm>
#include <cstddef>

#include "dfl_kernels.h"

namespace dfl {

constexpr int TG_LDS_BUDGET = 160 * 1024;  // one workgroup per CU

// The tile shapes the library instantiates: wm wave rows of mtw m-tiles (32 rows) each and wn
// wave columns of rbw weight row-blocks (32 columns) each, kc k per LDS stage.
// cyc: cycles of 2.4 GHz per k-block (32 k) of a workgroup while every CU runs one, measured
// over one to twenty rounds of 96 to 4096 rows (spread about 10 %): what the copies (9 to 32
// KiB a k-block), the fragment reads, the dequantisation and the MFMAs (64 mtw rbw cycles a
// wave) come to together.
// int8: every wave dequantises the weight blocks it multiplies, so two wave rows (each block
// dequantised twice per workgroup, not four times) take 128 x 128 in 458 us at 4096 x 10240 x
// 5120 against 494 with four rows of 1 x 4, and 128 x 64 in 560 against 593; the 256 x 128
// wave hides it under its MFMAs (375 us).  256 x 256 was slower in every arrangement (416-440).
// fp16, 777 x 4096 x 20480: 128 x 128 166 us, 256 x 64 225.
struct TileShape {
  int wt, wm, mtw, rbw, wn, kc, cyc;
};
constexpr TileShape kTileShapes[] = {
    {WT_INT8, 4, 1, 1, 1, 64, 410},    // 128 x 32
    {WT_INT8, 2, 2, 1, 2, 64, 450},    // 128 x 64
    {WT_INT8, 2, 2, 2, 2, 64, 690},    // 128 x 128
    {WT_INT8, 4, 2, 4, 1, 64, 1100},   // 256 x 128
    {WT_F16, 4, 2, 2, 1, 64, 860},     // 256 x 64
    {WT_F16, 4, 1, 4, 1, 64, 680},     // 128 x 128
    {WT_F16, 4, 2, 4, 1, 32, 1200},    // 256 x 128
    {WT_F16, 4, 2, 4, 2, 32, 2200},    // 256 x 256
};
// Independent MFMA accumulation chains of an output block: with two (int8 tiles of up to 128 x
// 128, whose few MFMAs a k-block would wait for each other) the halves of the k-blocks
// alternate between them and the chains are added at the end.
constexpr int tile_chains(int wt, int mtw, int rbw) { return wt == WT_INT8 && mtw * rbw < 8 ? 2 : 1; }
// Fewest k of a plane of the ingest's fc, whose planes the norm sums without a launch of its
// own (the plan counts one): twice what a workgroup's stage buffers hold, as shorter ranges spend
// their time filling them.  One-layer ingests with planes of at least 1024 / at least 64 k: hidden
// 2048 (K 10240), 65 rows 50 / 61 us, 128 rows 51 / 63; hidden 1024, 200 rows 40 / 47; hidden 512
// and 256 (33 / 31, as unsplit) give it up, and keep the sums of the whole product.
constexpr int FC_PLANE_K = 1024;
constexpr int kNumTileShapes = (int)(sizeof(kTileShapes) / sizeof(kTileShapes[0]));

// The 4-wave shapes add four loader waves that issue every global -> LDS copy (the compute
// waves never stall on a full memory queue, and four issuing waves copy 20-28 % faster than
// one: the copy rate is bounded by how fast copies are issued); the 8-wave shapes have no room
// for more waves' registers, so their compute waves issue the copies themselves.
constexpr int tile_loaders(int wm, int wn) { return wm * wn == 4 ? 4 : 0; }
// Bytes of one stage: the X records of the workgroup's m-tiles (2 KiB per tile and k-block
// of 32) and its weight blocks (1 KiB per row-block and 32 (int8) or 16 (fp16) k).
constexpr int tile_stage_bytes(int wt, int wm, int mtw, int rbw, int wn, int kc) {
  return wm * mtw * (kc / 32) * 2048 + rbw * wn * (kc / (wt == WT_INT8 ? 32 : 16)) * 1024;
}
// Stage buffers: as many as fit the LDS budget, at most 8, at most 3 more than a wave's
// vmcnt field (6 bits) counts in stages of its share of the copies, at least 3.  All but
// three of them are in flight while the compute waves read one and multiply another.
constexpr int tile_stages(int wt, int wm, int mtw, int rbw, int wn, int kc) {
  const int sb = tile_stage_bytes(wt, wm, mtw, rbw, wn, kc);
  const int loaders = tile_loaders(wm, wn);
  const int issuers = loaders ? loaders : wm * wn;
  const int per_wave = (sb / 1024 + issuers - 1) / issuers;
  const int by_lds = TG_LDS_BUDGET / sb;
  const int by_cnt = 3 + 63 / (per_wave > 0 ? per_wave : 1);
  const int s = by_lds < by_cnt ? by_lds : by_cnt;
  return s < 3 ? 3 : (s > 8 ? 8 : s);
}

// The instantiated shape (and split-K factor) with the least estimated time, in cycles of
// 2.4 GHz: rounds of one workgroup per CU x k-blocks x cycles per k-block, where a last
// partial round after full ones counts 0.75-1 of a round (its few workgroups copy faster:
// 0.75 measured at 16 of 256).  A split-K (allowed with split) runs fewer k-blocks per
// workgroup on larger tiles, so less X per flop, but each workgroup writes its fp32 tile
// (about 21 B per cycle) and a reduction launch reads every plane (about 1.4 KB per cycle
// over the chip, plus 12000 cycles of launch and tail).  Fitted to the measured times of
// the 8B- and 27B-class stacked products, the prompt-sized K|V ingest and the fp16
// lm_head (each picks its measured-fastest plan).
// Re-tiling (allowed with retile, no split-K): a plan of more tiles than CUs whose last
// round is partial may run that round's tiles on a smaller shape whose tiles divide them,
// several workgroups per tile over the whole K (the same sums), so that the last round
// finishes sooner; it costs one more launch (about 12000 cycles).
// Only the sub-shapes with the parent's accumulation chains qualify, so a tile's sums do
// not depend on which round it ran in.
// chains (optional): only shapes with that many accumulation chains, so that a product's sums
// are those of another plan (unsplit sums depend on the chains alone).
// pairs: each wave must hold gate|up row-block pairs (SWIGLU), i.e. an even rbw.
// plane_k: the fewest k of a split-K plane.
inline TilePlan tile_plan(int M, int N, int K, int wt, int n_cu, bool pairs = false,
                          bool split = false, bool retile = false, int chains = 0,
                          int plane_k = 64) {
  TilePlan best{};
  double best_t = 1e300;
  for (const TileShape& s : kTileShapes) {
    if (s.wt != wt || K % s.kc || (pairs && s.rbw % 2) ||
        (chains && tile_chains(wt, s.mtw, s.rbw) != chains))
      continue;
    const int bm = 32 * s.wm * s.mtw, bn = 32 * s.rbw * s.wn;
    if (N % bn) continue;
    const long long tiles = (long long)((M + bm - 1) / bm) * (N / bn);
    for (int sp = 1; sp <= (split ? 16 : 1) && sp * plane_k <= std::max(K, plane_k); sp *= 2) {
      if (sp > 1 && tiles * sp > n_cu) break;
      const long long full = tiles * sp / n_cu, part = tiles * sp % n_cu;
      const double rounds =
          (double)full + (part == 0 ? 0.0 : full > 0 ? 0.75 + 0.25 * part / n_cu : 1.0);
      double t = rounds * ((double)K / 32 / sp) * s.cyc;
      if (sp > 1)
        t += (double)bm * bn * 4 / 21.0 + (double)(sp + 1) * M * N * 4 / 1400.0 + 12000.0;
      if (t < best_t * 0.999) {
        best_t = t;
        best.wm = s.wm;
        best.mtw = s.mtw;
        best.rbw = s.rbw;
        best.wn = s.wn;
        best.kc = s.kc;
        best.tiles_m = (M + bm - 1) / bm;
        best.tiles_n = N / bn;
        best.splits = sp;
        best.head_tiles = 0;
        best.tail_shape = -1;
      }
    }
    const long long full = tiles / n_cu, part = tiles % n_cu;
    if (!retile || full < 1 || part == 0) continue;
    for (int i = 0; i < kNumTileShapes; ++i) {
      const TileShape& u = kTileShapes[i];
      const int um = 32 * u.wm * u.mtw, un = 32 * u.rbw * u.wn;
      if (u.wt != wt || K % u.kc || (pairs && u.rbw % 2) || bm % um || bn % un ||
          (um == bm && un == bn) || tile_chains(wt, u.mtw, u.rbw) != tile_chains(wt, s.mtw, s.rbw))
        continue;
      const long long sub = (long long)(bm / um) * (bn / un);
      const long long ur = (part * sub + n_cu - 1) / n_cu;   // rounds of the sub-tiles
      const double t = ((double)full * s.cyc + (double)ur * u.cyc) *
                           ((double)K / 32) + 12000.0;
      if (t < best_t * 0.999) {
        best_t = t;
        best.wm = s.wm;
        best.mtw = s.mtw;
        best.rbw = s.rbw;
        best.wn = s.wn;
        best.kc = s.kc;
        best.tiles_m = (M + bm - 1) / bm;
        best.tiles_n = N / bn;
        best.splits = 1;
        best.head_tiles = (int)(full * n_cu);
        best.tail_shape = i;
      }
    }
  }
  return best;
}

// Floats of the split-K planes that a product of 1 .. rows rows may be planned with (an F32 or
// RESID product with re-tiled last rounds): the most over every row count, as neither the factor
// nor the planes grow evenly with the rows.  A workspace of this size holds every plan, so that
// a product's split, and with it the order of its sums, is a rule on the product alone.
inline size_t tile_plane_floats(int rows, int N, int K, int wt, int n_cu, int plane_k = 64) {
  size_t most = 0;
  for (int M = 1; M <= rows; ++M) {
    const TilePlan p = tile_plan(M, N, K, wt, n_cu, false, true, true, 0, plane_k);
    if (p.splits > 1) most = std::max(most, (size_t)p.splits * M * N);
  }
  return most;
}

inline size_t tile_lds_bytes(int wt, const TilePlan& p) {
  return (size_t)tile_stages(wt, p.wm, p.mtw, p.rbw, p.wn, p.kc) *
         tile_stage_bytes(wt, p.wm, p.mtw, p.rbw, p.wn, p.kc);
}

}  // namespace dfl
