// Whole small levels of an index build in one launch (small_levels.hip).
#pragma once

#include "assign.h"
#include "cluster.h"

namespace hira {

constexpr int kSmallItems = 1024;      // what its LDS has room for
constexpr int kSmallCentroids = 32;
constexpr int small_pairs(int D) { return D <= 128 ? 32768 : 8192; }  // items times centroids

struct SmallLevels {
    const void* x;                     // (T, K[first - 1], D) bf16 items of level `first`
    const int32_t* n_live;             // (T) how many of them a tree holds, the first ones (then first = 1, last = 2); or NULL
    int32_t first, last;               // levels first .. last - 1
    int32_t K[HIRA_MAX_LEVELS];        // K[l - 1] items are clustered into K[l] blocks
    int32_t* slots[HIRA_MAX_LEVELS];   // (T, K[l], bf)
    void* cent_t[HIRA_MAX_LEVELS];     // (T, K[l], D) block centres in bf16
    float* cent;                       // (T, K[l], D)
    uint64_t seed;
    int32_t niter, pack_rounds, bf;
};
int launch_small_levels(const SmallLevels& p, int D, int num_trees, hipStream_t s);

}  // namespace hira
