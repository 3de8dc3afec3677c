// rd_choose.hpp -- launchers for the greedy choose kernels (rd_choose.hip).
#pragma once

#include "rd_common.hpp"

namespace rdhip {

template <typename T>
struct ChooseArgs {
    const T* P;
    int64_t pStride;
    const int* pIndex;        // optional position -> point map
    T* S;
    int64_t sStride;
    const SegDesc* segs;
    int numSegs;
    int* segK;
    const T* segRSqr;
    int* chosenIdx;           // per chosen slot: segment-relative index of the chosen sample
    int* overflow;
    // large segments (rounds of resolve and filter); small ones run in one block each
    const int* segLarge;      // per segment: 1 = large
    int numLarge;
    const int* largeSeg;      // [numLarge] their indices
    const int* largeBlock;    // [numLarge + 1] first filter block of each (kChooseBlock samples a block)
    uint64_t* open;           // one bit per own sample, 4 words per filter block; set: not decided yet
    int* base;                // [numLarge] chosen points the open samples have been tested against
    int* cursor;              // [numLarge] first word of the segment that may hold an open sample
    int* doneCount;           // large segments without an open sample
};

constexpr int kChooseBlock = 256;    // samples per filter block: one word of `open` per wave
constexpr int kChooseBatch = 1024;   // candidates one resolve step decides

// Chunk schedule of the fixed-launch form (rdhip_choose_noalloc): chunk c covers samples
// [choose_chunk_start(c), choose_chunk_start(c+1)).
__host__ __device__ inline int choose_chunk_start(int c) {
    if (c <= 0) return 0;
    if (c == 1) return 2048;
    if (c == 2) return 8192;
    if (c == 3) return 32768;
    long long v = 32768LL + (long long)(c - 3) * 65536LL;
    return v > 0x7fffffffLL ? 0x7fffffff : (int)v;
}

// every small segment, one block each
template <typename T>
hipError_t launch_choose_small(const ChooseArgs<T>& a, int dim, hipStream_t st);
// all samples of the large segments open, nothing chosen
template <typename T>
hipError_t launch_choose_open(const ChooseArgs<T>& a, int numBlocks, hipStream_t st);
// tests the open samples of filter blocks [block0, block0 + numBlocks) against the chosen points
// added since the last test (fresh: every sample of the blocks against all chosen points)
template <typename T>
hipError_t launch_choose_filter(const ChooseArgs<T>& a, int dim, int block0, int numBlocks, bool fresh,
                                hipStream_t st);
// decides the first open samples of every large segment: up to maxBatches batches of
// kChooseBatch (0: all of them), of the samples below endSample only (< 0: all)
template <typename T>
hipError_t launch_choose_resolve(const ChooseArgs<T>& a, int dim, int endSample, int maxBatches, hipStream_t st);

}  // namespace rdhip
