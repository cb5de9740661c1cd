// spic_wave.hpp -- counting of keyed particles by waves.  Internal to
// libspic.so; device code only.
#pragma once

#include <hip/hip_runtime.h>

namespace spic {

// Counters of a workgroup in LDS at most (24 KB), where kernels count
// particles per tile.
constexpr int kLdsTiles = 6144;

// Adds this lane's particle to the counter of its key and returns its rank
// there.  Lanes of one wave that share a key take one atomic together
// (particles of a run are near each other in most orders); after four
// distinct keys the remaining lanes take one each.
__device__ __forceinline__ unsigned int key_rank(unsigned int *cnt, unsigned int key,
                                                 bool active) {
  const int lane = threadIdx.x & 63;
  unsigned long long todo = __ballot(active);
  int leader = lane;
  unsigned int off = 0, group = 1;
  for (int round = 0; round < 4 && todo; ++round) {
    const int first = __ffsll((long long)todo) - 1;
    const unsigned int k0 = (unsigned int)__builtin_amdgcn_readlane((int)key, first);
    const bool mine = ((todo >> lane) & 1ull) && key == k0;
    const unsigned long long same = __ballot(mine);
    if (mine) {
      leader = first;
      off = (unsigned int)__popcll(same & ((1ull << lane) - 1ull));
      group = (unsigned int)__popcll(same);
    }
    todo &= ~same;
  }
  unsigned int r = 0;
  if (active && lane == leader) r = atomicAdd(cnt + key, group);
  return (unsigned int)__shfl((int)r, leader) + off;
}

}  // namespace spic
