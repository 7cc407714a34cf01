// How a prefill launch is cut into workgroups: host code only, nothing of HIP in it.
#pragma once

#include <stdint.h>

#include <algorithm>

#include "sqattn.h"

namespace sq {

constexpr int kPlanTile = 64;            // keys per tile
constexpr int kMaxSplitWork = 512;       // workgroups per (batch, q head) of a launch with split key ranges
constexpr int kPlanCUs = 256, kPlanMaxRounds = 4;

// One workgroup of a split launch: part `part` of `parts` of query block `qb`; `slot` is the first of the block's `parts`
// places in the partial results (parts > 1)
struct SplitWork {
  uint16_t qb, slot;
  uint8_t part, parts;
};

struct LaunchPlan {
  int waves = 8;                 // per workgroup, where the launch is not split (a split one has 8)
  int n_work = 0, n_slots = 0;   // n_work == 0: not to be split
  int share = 0;                 // tiles of the longest part
  SplitWork work[kMaxSplitWork];
};

// Tiles the workgroup of query rows [r0, r1) walks: everything up to its diagonal, or sink and windows (of the widest head)
inline int tiles_of_block(const sq_prefill_params* p, int64_t r0, int64_t r1, int w_max) {
  const int64_t hi = (p->q_offset + r1 + kPlanTile - 1) / kPlanTile;
  if (p->window_mode == SQ_WINDOW_NONE) return (int)hi;
  const int64_t lo = std::max<int64_t>(0, (p->q_offset + r0) / p->block_m * p->block_m + p->block_m - w_max) / kPlanTile;
  return (int)std::min(hi, hi - std::min(lo, hi) + p->sink / kPlanTile);
}

// A launch whose query blocks do not fill the chip is as long as its longest chain of tiles: 64 workgroups of up to 64 tiles
// (4096 tokens, 4 heads) left three quarters of the CUs idle.  Two remedies, chosen by an estimate of the launch's
// length; all constants are measured times.
//  * Split key ranges: several workgroups per query block, each with a contiguous share of the block's steps, and a second
//    kernel that merges their accumulators.  The e4m3 modes with a static or absmax grid (1 .. 4), whose P depends on the
//    row's running maximum, first run a pass that only forms the parts' row maxima (MODE 7), so that every part starts from
//    the reference point it would have had.  4096 tokens, 4 / 1 heads: mode 0 88 -> 42 us, mode 1 132 -> 66, mode 2 141 ->
//    62; a chunk of 512 rows behind 16384 tokens at 28 / 4 heads 325 -> 132 us in mode 0.  Mode 5 stays whole: where its reference
//    point stands depends on every tile sum before (a jump of 2^100 puts it on that tile's maximum), not on a maximum.
//  * Workgroups of 128 rows (4 waves): one wave per SIMD walks a tile in 0.7 to 0.82 of the time two take for theirs.  Short
//    prompts, where a merge costs more than it saves: 777 tokens, 28 / 4 heads, mode 0 30.5 -> 24.1 us (split: 34), mode 1
//    38.2 -> 28.4, mode 5 38.0 -> 30.2; 2048 tokens (448 workgroups) 57 -> 52, at 3000 the 8-wave launch is ahead (82
//    against 95).  Up to 128 rows four waves of the 8-wave workgroup have no rows, so the others have a SIMD each there too
//    and all eight copy the tiles: 0.07 to 0.1 us less per tile, against a smaller launch's 0.1 (mode 0) to 1.5 us.  The
//    sides meet at kFewRowsTiles: 64 rows, 28 / 4 heads, mode 5: 1 tile 21.1 us with 4 waves, 22.4 with 8; 17 tiles 33.2 / 33.4; 65
//    tiles 69.8 / 65.8 (2049 tiles 1560 / 1376); int8 Q.K^T: 1 tile 13.3 / 15.0, 17 tiles 33.8 / 33.7, 65 tiles 95.6 / 90.7.
// A tile of an 8-wave workgroup takes kStepUs on an otherwise idle chip and about 30 % more on a full one, which lowers its
// clock: 8192 rows behind 24576 tokens, 3.5 workgroups per CU, take 2685 us split evenly or not.
// Mode 2 (26 sizes, every form forced): the plan within 8 % of the best form everywhere, 1.5 % in the mean.
inline void plan_launch(const sq_prefill_params* p, bool own4, int64_t B, int64_t Hq, int64_t Nq, LaunchPlan& plan, bool int8qk = false) {
  const int mode = int8qk ? 6 : p->p_quant;
  constexpr int kCUs = kPlanCUs, kMaxRounds = kPlanMaxRounds, kMinTiles = 4;
  static const float kStepUs[7] = {1.35f, 1.75f, 2.05f, 1.4f, 1.15f, 1.15f, 1.35f};   // by P mode; 6: int8 Q.K^T
  constexpr float kFixUs = 8.f;      // a workgroup's launch, first loads and epilogue
  static const float kFourWaves[7] = {0.76f, 0.7f, 0.73f, 1.f, 1.f, 0.76f, 0.76f};
  static const int kFewRowsTiles[7] = {2, 2, 5, 0, 0, 16, 11};
  constexpr float kFullChip = 0.3f;
  constexpr float kMergeUs = 6.f, kPartUs = 0.07f;   // the merge; a part's 130 KB written and read again
  constexpr float kRefUs = 8.f, kRefTileUs = 0.6f;   // MODE 7: launch and fixed part, per tile
  plan.waves = 8;
  plan.n_work = plan.n_slots = 0;
  if (own4 && p->window_mode == SQ_WINDOW_SIZES && p->block_m == 64) {
    plan.waves = 2;   // separate 4-bit operands with 64-row blocks: a workgroup of one block (with 128-row blocks: DUAL)
    return;
  }
  const int64_t nQB = (Nq + 255) / 256, mult = B * Hq;
  if (mult * nQB > kMaxRounds * kCUs) return;
  const float step = kStepUs[mode];
  // Mode 4's step is the shortest beside the same row-maximum pass, so a split in two that fills the chip loses: chains of like
  // length on up to half the CUs run at the idle chip's rate (1.00 us a tile, 1.02 on 128 CUs), the pass slows down on a full
  // chip.  8192 rows behind 57344 keys, 4 / 1 heads (128 chains): 1057 us whole, 1163 split; 4096 behind 32768: 637 whole, 393
  // split; without a context, where the chains are unlike, 3000 rows of 8 / 8 heads 80 whole, 70 split.
  const bool fp8_pv = p->p_quant == SQ_P_E4M3_FP8_PV;
  int w_max = 0;
  if (p->window_mode == SQ_WINDOW_SIZES)
    for (int h = 0; h < Hq; ++h) w_max = std::max(w_max, std::max(p->w8[h], p->w4[h]));
  // one workgroup per block of `rows` rows: the blocks of a head, longest first, on kCUs / mult CUs (each of them stands
  // for the same block of every head)
  int len[kMaxRounds * kCUs], longest = 0;
  bool even_fp8 = false;
  auto unsplit_us = [&](int rows, float tile_us) {
    const int n = (int)((Nq + rows - 1) / rows), cus = (int)std::max<int64_t>(1, kCUs / mult), rounds = (int)((mult + kCUs - 1) / kCUs);
    struct Cu { float load, tiles; } cu[kCUs] = {};
    const auto later = [](const Cu& x, const Cu& y) { return x.load > y.load; };   // a heap with the least loaded CU in front
    float total = 0, last = 0, last_tiles = 0;
    for (int qb = n - 1; qb >= 0; --qb) {
      const int t = tiles_of_block(p, (int64_t)qb * rows, std::min<int64_t>(Nq, (int64_t)(qb + 1) * rows), w_max);
      if (rows == 256) {
        len[qb] = t;
        longest = std::max(longest, t);
      }
      std::pop_heap(cu, cu + cus, later);
      Cu& c = cu[cus - 1];
      c.load += (t * tile_us + kFixUs) * rounds;
      c.tiles += (float)t * rounds;
      total += (float)t * mult;
      if (c.load > last) {
        last = c.load;
        last_tiles = c.tiles;
      }
      std::push_heap(cu, cu + cus, later);
    }
    if (rows == 256) even_fp8 = fp8_pv && n * mult <= kCUs / 2 && total > 0.75f * n * mult * longest;
    return last + (even_fp8 ? 0.f : kFullChip) * std::min(1.f, total / (kCUs * last_tiles)) * last_tiles * tile_us;
  };
  float best = unsplit_us(256, step);
  const bool four_waves = !own4 && (p->p_quant <= SQ_P_E4M3_BLOCK || p->p_quant == SQ_P_E4M3_MX_FP8_PV);
  if (four_waves && (Nq > 128 || longest <= kFewRowsTiles[mode]) && mult * ((Nq + 127) / 128) <= 2 * kCUs) {
    const float us = unsplit_us(128, step * kFourWaves[mode]);
    if (us < best) {
      best = us;
      plan.waves = 4;
    }
  }
  if (longest <= kMinTiles || (own4 && p->p_quant != SQ_P_NONE) || p->p_quant == SQ_P_E4M3_MX_FP8_PV) return;
  const bool ref_pass = p->p_quant >= SQ_P_E4M3_STATIC && p->p_quant <= SQ_P_E4M3_FP8_PV;
  // the parts of modes 0 and 6 start from the row's scores of tile 0, which windows without a sink do not reach
  if (!ref_pass && p->window_mode == SQ_WINDOW_SIZES && p->sink < kPlanTile) return;
  auto workgroups = [&](int cap) {
    int64_t n = 0;
    for (int qb = 0; qb < nQB; ++qb) n += (len[qb] + cap - 1) / cap;
    return n;
  };
  float total = 0;
  for (int qb = 0; qb < nQB; ++qb) total += (float)len[qb] * mult;
  int cap = 0;
  for (int m = 1; m <= kMaxRounds; ++m) {
    int lo = kMinTiles, hi = longest;   // the smallest share that keeps to m workgroups per CU
    while (lo < hi) {
      const int c = (lo + hi) / 2;
      if (workgroups(c) * mult <= m * kCUs) hi = c;
      else lo = c + 1;
    }
    if (lo >= longest || workgroups(lo) > kMaxSplitWork) continue;
    float us = m * (lo * step * (1.f + kFullChip * std::min(1.f, total / (kCUs * m * lo))) + kFixUs) + kMergeUs + kPartUs * mult * workgroups(lo);
    if (ref_pass) us += m * lo * kRefTileUs * (even_fp8 ? 1.f + kFullChip * std::min(1.f, total / (kCUs * m * lo)) : 1.f) + kRefUs;
    if (us < 0.97f * best) {
      best = us;
      cap = lo;
    }
  }
  if (cap == 0) return;
  plan.share = cap;
  for (int64_t qb = nQB - 1; qb >= 0; --qb) {
    const int parts = std::min((len[qb] + cap - 1) / cap, 255);
    for (int i = 0; i < parts; ++i) plan.work[plan.n_work++] = SplitWork{(uint16_t)qb, (uint16_t)plan.n_slots, (uint8_t)i, (uint8_t)parts};
    if (parts > 1) plan.n_slots += parts;
  }
  // longest shares first
  std::stable_sort(plan.work, plan.work + plan.n_work, [&](const SplitWork& x, const SplitWork& y) { return (int64_t)len[x.qb] * y.parts > (int64_t)len[y.qb] * x.parts; });
}

// Whether the row-maximum pass of a split launch also forms the V^T tiles, two at a time in each of its workgroups that have no
// part to look at (one per query block): where they are done with it before the parts are, at 1.3 us a round against
// 0.6 us a tile.  4096 tokens, 4 / 1 heads, mode 2 (1 round, shares of 10) 64.4 -> 59.3 us; 512 rows behind 16384 tokens, 28 / 4
// heads, mode 1 (10 rounds, shares of 65) 224 -> 214.  Beyond it the pass would wait for them: 64 rows behind 16384 tokens (19 rounds, shares of
// 29) keep the launch of their own.
inline bool prep_beside_pass(int share, int64_t v_tiles, int64_t idle) { return 1.3f * (float)((v_tiles + 2 * idle - 1) / (2 * idle)) <= 0.6f * share + 1.f; }

}  // namespace sq
