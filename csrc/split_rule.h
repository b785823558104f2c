// How many workgroups share a row's keys in the attention of a prompt step (both extensions' bindings).
#pragma once

#include <algorithm>
#include <cstdint>

// Times in us of the two forms: one kernel over all keys (its start, a tile of 32 keys of a workgroup by itself, workgroups per compute unit
// up to which that holds), and split keys with a merge (the same, and the bytes of partial results of one split).
struct SplitTimes {
  double one_start, one_tile, one_resident;
  double split_start, split_tile, split_resident;
};

// The number of splits, `most` halved or 1, that is estimated to take least. Splits fill the chip where row tiles are few, but write and
// read fp32 results of every row; chosen only to have 2048 workgroups in flight they took 1.5 - 5 times as long as no split
// (attention over 8 x 500 rows, 16 heads of 128 + 128: 80 us in 8 splits, 22 in one kernel; 16 x 250 of 32 heads: 112 / 23). They stay for few
// rows behind many keys (16 rows behind 8000: 29 / 220) and are halved in between (1000 behind 2000: 16 splits 87, 4 63, none 78). Over 2502
// random steps of attention and latent attention the choice is 0.6 % from the best of 1 - 16 splits in the mean; 13 of them are more than 3 % slower than
// in all splits, 14 % at most, and the mean is 1.67 times as fast.
// `one_keys`: the keys that a row tile of the kernel without splits walks, fewer than `keys` where a window follows the rows (1500 rows with a
// window of 1024, capped scores: 89 us in the two splits that the whole portion's keys would call for, 51 in one kernel).
inline int64_t best_splits(const SplitTimes& t, int64_t most, int64_t keys, int64_t one_keys, int64_t one_wgs, int64_t split_wgs, int64_t cus,
                           int64_t split_bytes) {
  const double tiles = (double)keys / 32.0, c = (double)cus;
  double least = t.one_start + t.one_tile * (double)one_keys / 32.0 * std::max(1.0, (double)one_wgs / (t.one_resident * c));
  int64_t best = 1;
  for (int64_t n = most; n > 1; n /= 2) {
    const double turns = std::max(1.0, (double)(split_wgs * n) / (t.split_resident * c));
    const double us = t.split_start + t.split_tile * tiles / (double)n * turns + 2.0 * (double)n * (double)split_bytes / 3.5e6;
    if (us < least) least = us, best = n;
  }
  return best;
}
