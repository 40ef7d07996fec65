// The rows of one token's choices in the order that combine adds them, for kernels that fold it in.
#pragma once

#include "common.h"

namespace combine_core {

constexpr int AT_ONCE = 8;   // choices whose rows are asked for together

// Up to AT_ONCE choices of a token: their rows of y in ascending expert id (slot where ids repeat), and the
// router weight of each (1 where y is already scaled). The same in every lane.
struct Choices {
  int row[AT_ONCE];
  float weight[AT_ONCE];
};

// Every wavefront ranks for itself: lane j holds choice j, a rank is a count over lane reads, and the j-th row
// is read from the lane whose rank is j. No LDS, no barrier, and the rows' addresses are scalars, so a
// token's k rows are k loads in flight behind one wait for its ids.
__device__ __forceinline__ Choices ranked(const int* __restrict__ idx, const int* __restrict__ pos_of,
                                          const half_t* __restrict__ w, size_t at, int k) {
  const int lane = threadIdx.x & 63;
  const int mine = lane < k ? idx[at + lane] : 0x7fffffff;
  const int src = lane < k ? pos_of[at + lane] : 0;
  const float wt = lane < k && w ? (float)w[at + lane] : 1.f;
  int rank = 0;
#pragma unroll
  for (int j = 0; j < AT_ONCE; ++j) {
    const int other = read_lane(mine, j);
    if (j < k) rank += (other < mine) || (other == mine && j < lane);
  }
  Choices c;
#pragma unroll
  for (int j = 0; j < AT_ONCE; ++j) {
    const uint64_t who = __ballot(lane < k && rank == j);
    const int from = who ? __builtin_ctzll(who) : 0;   // past the last choice: a row that exists
    c.row[j] = read_lane(src, from);
    c.weight[j] = read_lane(wt, from);
  }
  return c;
}

}  // namespace combine_core
