// fof_pairwalk.h -- the particle pairs of two runs, shared out over lanes.
#pragma once

#include <stdint.h>

#ifdef __HIPCC__
#define FOF_HD __host__ __device__ __forceinline__
#else
#define FOF_HD inline
#endif

namespace fof {

// Pairs (i, j), i < m1, j < m2, in row-major order: the lane that starts at
// pair `first` visits every kPairLanes-th from there, until i >= m1.  The
// pair's number is never formed: m1 m2 passes 2^32 from 65536 particles a run
// (sizes below 2^31).
constexpr uint32_t kPairLanes = 16;

struct PairWalk {
  uint32_t i, j, di, dj, m2;
  FOF_HD PairWalk(uint32_t first, uint32_t m2_)
      : i(first / m2_), j(first % m2_), di(kPairLanes / m2_), dj(kPairLanes % m2_), m2(m2_) {}
  FOF_HD void step() {
    i += di;
    j += dj;
    if (j >= m2) j -= m2, i++;
  }
};

}  // namespace fof
