// Tile choice of the 16x16x32-MFMA GEMMs (bfa_gemm.h), shared by the linear
// layers (linear_gemm.hip) and the QKV projection (qkv_prefill.hip).
#pragma once

#include <stdint.h>

#include <type_traits>

#include "bfa_host.h"

namespace bfa {

// The tiles, and a stage's time on a full chip (BM x BN x 64, 256 workgroups,
// measured at 6000 tokens with K = 4096 and 14336): the planner compares tiles
// by rounds x stages x this.  The wide tiles do more per LDS byte (0.95 us for
// 128 x 256 against 1.55 for twice the work), the small ones fill a short grid.
// 64 x 256, 320 x 128 and 4-wave 160 x 128 and 64 x 128 tiles were never ahead
// of the best of these by more than 0.4 us (three models' MLPs, 80 to 6000 tokens).
template <int MA_, int RW_, int CW_, int NS_>
struct GemmTileShape {
  static constexpr int MA = MA_, RW = RW_, CW = CW_, NS = NS_;
};
struct GemmTileInfo {
  int ma, rw, cw;
  double stage_us;
};
constexpr GemmTileInfo kGemmTiles[] = {
    {8, 2, 4, 1.55},  // 0: 256 x 256, 2 stages
    {6, 2, 4, 1.30},  // 1: 192 x 256, 2
    {5, 2, 4, 1.12},  // 2: 160 x 256, 3
    {4, 2, 4, 0.95},  // 3: 128 x 256, 3
    {4, 4, 2, 0.96},  // 4: 256 x 128, 3
    {3, 4, 2, 0.75},  // 5: 192 x 128, 4
    {2, 4, 2, 0.58},  // 6: 128 x 128, 5
    {1, 4, 2, 0.38},  // 7:  64 x 128, 6
};
constexpr int kNumGemmTiles = static_cast<int>(sizeof(kGemmTiles) / sizeof(kGemmTiles[0]));

// f(GemmTileShape) of a tile id
template <class F>
void gemm_tile_dispatch(int tile, F f) {
  switch (tile) {
    case 0: f(GemmTileShape<8, 2, 4, 2>{}); break;
    case 1: f(GemmTileShape<6, 2, 4, 2>{}); break;
    case 2: f(GemmTileShape<5, 2, 4, 3>{}); break;
    case 3: f(GemmTileShape<4, 2, 4, 3>{}); break;
    case 4: f(GemmTileShape<4, 4, 2, 3>{}); break;
    case 5: f(GemmTileShape<3, 4, 2, 4>{}); break;
    case 6: f(GemmTileShape<2, 4, 2, 5>{}); break;
    default: f(GemmTileShape<1, 4, 2, 6>{}); break;
  }
}

struct GemmPlan {
  int tile;
  int tiles_m, tiles_n;
  int full;    // tiles taken whole; the others are split over K
  int splits;
  int64_t part_bytes;
};

// Each tile is weighed with every tile whole and, where the last round is not
// full, with that round's tiles split over K as often as the CUs allow: rounds
// times (stages x stage_us + fixed_us for fill and epilogue), and for split
// tiles the second launch (split_us) and the partials' round trip (3 TB/s), which
// may take up to part_limit bytes.  Overrides: BFA_TUNE_GEMM_TILE,
// BFA_TUNE_GEMM_SPLITS.
inline GemmPlan gemm_plan(int64_t m, int64_t wrows, int64_t k, double fixed_us, double split_us,
                          int64_t part_limit) {
  const int ot = tuning(BFA_TUNE_GEMM_TILE), os = tuning(BFA_TUNE_GEMM_SPLITS);
  const int64_t kt = k / 64;
  GemmPlan best{};
  double cost = 0;
  for (int id = 0; id < kNumGemmTiles; ++id) {
    if (ot >= 0 && ot < kNumGemmTiles && id != ot) continue;
    const GemmTileInfo& t = kGemmTiles[id];
    GemmPlan p{};
    p.tile = id;
    const int64_t tm = cdiv(m, 16 * t.ma * t.rw), tn = cdiv(wrows, 64 * t.cw);
    const int64_t tiles = tm * tn, rounds = tiles / 256, rest = tiles % 256;
    p.tiles_m = static_cast<int>(tm);
    p.tiles_n = static_cast<int>(tn);
    p.full = static_cast<int>(tiles);
    p.splits = 1;
    double c = static_cast<double>(rounds + (rest > 0)) * (kt * t.stage_us + fixed_us);
    int64_t s = rest > 0 ? 256 / rest : 1;
    if (os >= 1) s = os;
    s = std::min<int64_t>(std::min<int64_t>(s, kt), 32);
    const int64_t bytes = rest * s * t.rw * t.cw * t.ma * 4 * 64 * 16;
    if (rest > 0 && s > 1 && bytes <= part_limit) {
      const double cs = static_cast<double>(rounds) * (kt * t.stage_us + fixed_us) +
                        static_cast<double>(cdiv(rest * s, 256)) * (cdiv(kt, s) * t.stage_us + fixed_us) + split_us +
                        static_cast<double>(bytes) / 3.0e6;
      if (cs < c || os > 1) {
        c = cs;
        p.full = static_cast<int>(rounds * 256);
        p.splits = static_cast<int>(s);
        p.part_bytes = bytes;
      }
    }
    if (best.splits == 0 || c < cost) {
      best = p;
      cost = c;
    }
  }
  return best;
}

}  // namespace bfa
