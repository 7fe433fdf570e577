// launch_split.hpp -- how much work one launch may carry (host arithmetic only).
#pragma once

#include <stdint.h>

namespace gbsk {

// HIP refuses launches of 2^32 work-items (grid x block) and more, that is of 2^26
// waves. Kernels of four waves a workgroup round up to a multiple of four, so
// four less: every launch below counts its waves against this.
constexpr int64_t LAUNCH_WAVES = ((int64_t)1 << 26) - 4;

// most rows (matrices, groups of them) of `waves` waves each in one launch, a
// multiple of `step`
constexpr int64_t launch_rows(int64_t waves, int64_t step = 1) { return LAUNCH_WAVES / waves / step * step; }

// Workgroups of a permanent launch (one wave each): `groups` of matrices, W chunks
// each; with W > 1 padded to a multiple of the 8 XCDs the chunks are dealt to
// (of the groups, if fewer).
constexpr int64_t perm_grid(int64_t groups, int W) {
  const int64_t g8 = groups < 8 ? groups : 8;
  return W == 1 ? groups : (groups + g8 - 1) / g8 * g8 * W;
}

// Several buckets in one launch, in order.
struct LaunchRoom {
  int64_t used = 0;
  // the number of a bucket's next rows (`waves` waves each) that still fit, taken
  // off the room; 0: the launch is full
  int64_t take(int64_t rows, int64_t waves) {
    const int64_t fit = (LAUNCH_WAVES - used) / waves;
    const int64_t n = rows < fit ? rows : fit;
    used += n * waves;
    return n;
  }
};

}  // namespace gbsk
