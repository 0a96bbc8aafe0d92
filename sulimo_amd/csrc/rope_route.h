// rope_route.h - which RoPE calls rope_f16_vec_kernel takes, and its grid. Host arithmetic
// only, so that a CPU test can compile it.
#pragma once

#include <limits.h>
#include <stdint.h>

namespace sulimo {

constexpr int kRopeHeads = 4;      // heads of a thread
constexpr int kRopeThreads = 256;  // threads of a workgroup

struct RopeVecGrid {
  unsigned x, y;  // workgroups: (token, four pairs) by 256, groups of heads; x = 0: not its call
};

// Whole quads of pairs, in rows and halves of 16- and 8-byte alignment; thread numbers
// (up to the end of the last workgroup) that an int holds, and at most 65535 groups of
// heads. Other calls take rope_f16_kernel, whose numbers are 64-bit.
inline RopeVecGrid rope_vec_grid(int head_count, int head_dim, int rope_dim, int n) {
  if (head_count < 1 || n < 1 || rope_dim < 8 || rope_dim % 8 || head_dim % 8) return {0, 0};
  const int64_t x = ((int64_t)n * (rope_dim / 8) + kRopeThreads - 1) / kRopeThreads;
  const int64_t y = ((int64_t)head_count + kRopeHeads - 1) / kRopeHeads;
  if (x * kRopeThreads > INT_MAX || y > 65535) return {0, 0};
  return {(unsigned)x, (unsigned)y};
}

}  // namespace sulimo
