// Host entry of the prompt-sized append (append_bulk.hip).
#pragma once
#include "append_row.h"

namespace kvq {

constexpr int kBulkMaxWaves = 8;      // waves per work-group at most
constexpr int kBulkWaveSlots = 8192;  // most waves per side: 8 a SIMD on 256 CUs
// Fewest new tokens per (b, head).  A wave takes 8 tokens at least, so below that lanes idle and
// one row a wave is as good.
constexpr int kBulkMinTokens = 8;
// 32-token tiles per side from which a wave takes 32 (16) tokens, else 8: a longer tile has more
// loads in flight, a shorter one gives more waves.  Measured in us for 8 / 16 / 32 tokens a wave:
// 256 tiles (INT8, 2 x 4096 tokens) 5.4 / 5.8 / 7.9, 1024 (KIVI INT4, 4 x 8191) 21.2 / 12.5 / 12.5,
// 1504 (INT4, 8 x 6001) 14.6 / 13.2 / 14.3.
constexpr int kBulkTiles32 = 2048, kBulkTiles16 = 512;
// Tiles for which a work-group has 8 waves instead of 4 where a side counts clipped values (a static
// table and a status word).  A work-group that clipped adds to the side's one status word and such
// atomics queue (about 10 ns each), so half as many help where about every tile clips; a count that
// stays 0 only pays for the coarser grid.  us for 4 / 8 waves, INT8 tables that clip half of the values,
// and tables that clip none: 1056 tiles 9.6 / 8.9 and 7.8 / 8.7, 1504 10.9 / 9.9 and 8.2 / 8.9, 1952
// 13.2 / 11.4 and 9.5 / 9.2, 3000 18.3 / 14.3 and 12.2 / 12.1, 8128 60.6 / 44.9 and 44.2 / 44.7.  Above
// kBulkWaveSlots a wave takes several tiles; clipping sides still gain there for a while (12000 73.0 /
// 64.6), those that clip nothing lose (8 bits of KIVI, 10016 tiles 60.7 / 63.5, 14016 71.5 / 78.8).
// Sides that count nothing keep 4: INT8 with the 99.9 percentile 2112 tiles 20.6 / 23.2, 4096 30.9 /
// 31.9, 8128 51.2 / 53.2; the mixed cache 2112 22.6 / 26.2.
constexpr int kBulkWideFrom = 1728, kBulkWideTo = kBulkWaveSlots;

// Order statistics of a percentile (ranks and weight, as torch.quantile computes them) and
// whether a static table has a per-token policy.
struct BulkSide {
  int top2, policy;
  int local;             // the rescue threshold is found by the append's work-groups
  int lo, hi, blo, bhi;  // ranks near the top; KIVI V: near the bottom
  float w, bw;
};

// A launch of the tile kernel
struct BulkPlan {
  BulkSide ks, vs;
  int ck, cv;       // the sides' formats, TILE32 apart from rows
  int tok;          // tokens a wave takes at a time
  int waves;        // a work-group
  unsigned groups;  // work-groups a side
};

// Whether the tile kernel takes the append of k and v, and how.  It takes what the engines hand over:
// both sides INT8_SYM or both INT4_SYM, any two KIVI formats, INT8_SYM with INT4_KIVI, INT4_ASYM or
// INT8_SYM K with TILE32 V, and any of the former's sides alone, from kBulkMinTokens tokens on, with
// 16-byte aligned rows, code rows aligned to a lane's store and percentiles within the two largest
// (smallest) values of a group.  Every other append is the row kernel's at any length: INT4_ASYM in
// token rows on both sides or either INT4_ASYM side alone, and FP16 rows beside a quantized side (the
// engines copy those with torch and append the other side alone).  The caller has validated both
// sides (fill_dev); a side's group rescue has its threshold selected in its scratch, or with `local`
// (at most kRescueMax scales) every work-group finds it.
bool bulk_plan(const AppendDev& k, const AppendDev& v, bool local, BulkPlan& p);
void append_bulk(const AppendDev& k, const AppendDev& v, const BulkPlan& p, hipStream_t st);

}  // namespace kvq
