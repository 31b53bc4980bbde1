// launch.h -- sizes of one-dimensional launches, included by tslb.hip inside its
// anonymous namespace.
//
// A launch holds its work-items, blocks times threads, in 32 bits: HIP refuses
// exactly 2^32 of them and starts only the remainder of more than that, without
// an error.  A state buffer has more words than that from 390 million nodes in
// FP32, so a fill strides over it with a bounded grid.
#pragma once

constexpr long long kMaxFillBlocks = 1 << 18;  // of 256 threads: 1024 per CU

inline unsigned fill_blocks(long long n) {
  const long long b = (n + 255) / 256;
  return (unsigned)(b < 1 ? 1 : (b < kMaxFillBlocks ? b : kMaxFillBlocks));
}
