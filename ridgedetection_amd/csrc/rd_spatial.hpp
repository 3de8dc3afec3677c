// rd_spatial.hpp -- incremental evolve scan: samples in a spatial order, cut into blocks with
// bounding boxes, so that a block looks only at the chosen points that can be nearest to one of
// its samples, and only when one of those may have changed.  Kernels in rd_spatial.hip.
#pragma once

#include "rd_evolve.hpp"

namespace rdhip {

constexpr int kBoxThreads = 256;
constexpr int kBoxSamples = 512;   // samples of a block

// Where a segment's samples lie: bits of the spatial key, the coordinate each bit halves (4 bits
// each, first split lowest) and the affine map of every coordinate onto its share of the bits.
template <typename T>
struct SpatialMap {
    T lo[kMaxDim];
    T scale[kMaxDim];
    unsigned long long split;
    int bits[kMaxDim];
};

constexpr int kSpatialBitsMax = 16;
constexpr int kBoundsItem = 4096;   // samples of a partial bounds block

// Spatial order of the positions of every segment (built once per points and segments).
template <typename T>
struct SpatialBuild {
    const T* P;
    int64_t pStride;
    const int* pIndex;
    const SegDesc* segs;
    int numSegs;
    const WorkItem* items;      // bounds items: kBoundsItem positions each
    int numItems;
    const int* segFirstItem;    // numSegs + 1
    T* partial;                 // [numItems][2 dim]
    SpatialMap<T>* maps;        // [numSegs]
    int keyBits;                // spatial bits below the segment number
    int* keys;                  // per position
};

// keys of all positions: segment number, then the spatial key
template <typename T>
hipError_t launch_spatial_keys(const SpatialBuild<T>& b, int dim, hipStream_t st);
// Q[d][i] = coordinate d of position perm[i]
template <typename T>
hipError_t launch_spatial_gather(const T* P, int64_t pStride, const int* pIndex, const int* perm, int64_t n, int dim,
                                 T* Q, int64_t qStride, hipStream_t st);
// box[b][0, dim) / [dim, 2 dim): lower and upper corner of box item b's samples
template <typename T>
hipError_t launch_spatial_boxes(const T* Q, int64_t qStride, const WorkItem* items, const SegDesc* segs, int numItems,
                                int dim, T* box, hipStream_t st);

template <typename T>
struct BoxScanArgs {
    const T* Q;                 // samples in spatial order
    int64_t qStride;
    const int* perm;            // spatial position -> position
    const WorkItem* items;      // segment, [start, end) of its spatial positions, pad: box
    const int* numItemsDev;     // optional: the items in use
    const T* box;
    T* bound;                   // per box: its samples' labels depend on the chosen points within
    const T* S;
    const T* Sold;              // chosen points before their last move
    int64_t sStride;
    const SegDesc* segs;
    const int* segK;
    const int* segDone;
    const T* segRSqr;
    const int* allDone;
    int* labS;                  // label per spatial position
    int* labels;                // label per position
    const int* moved;           // per slot: 1 if the last iteration moved it
    int* touched;               // per slot: set to 1 when its members change
    int* hist;                  // per segment [key][block] counts of rd_chain.hpp
    const int64_t* histSegOff;
    int itemSize;
};

// first: every box is evaluated and no count is kept (label_hist follows); otherwise the counts
// and touched flags follow the labels that change.
template <typename T>
hipError_t launch_box_scan(const BoxScanArgs<T>& a, int dim, int numItems, bool first, hipStream_t st);

// The [key][block] counts of rd_chain.hpp from the labels, one block per item.
hipError_t launch_label_hist(const WorkItem* items, const int* numItemsDev, int numItems, const SegDesc* segs,
                             const int* segK, const int* segDone, const int* labels, int* hist,
                             const int64_t* histSegOff, int itemSize, const int* allDone, hipStream_t st);

}  // namespace rdhip
