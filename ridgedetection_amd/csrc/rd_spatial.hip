// rd_spatial.hip -- the incremental evolve scan (nearest chosen point of every sample,
// rd/cpu/brute_force/evolve.hpp:32-77).
//
// The samples of a segment are put once into a spatial order (a key of midpoint splits of the
// widest side of the bounding box, radix sorted) and cut into blocks of kBoxSamples with bounding
// boxes.  Per iteration a block
//   1. is skipped when no chosen point that moved in the last iteration lies, before or after the
//      move, within the distance `bound` that decided its labels;
//   2. otherwise bounds every sample's nearest distance from above by the smallest farthest
//      distance U of a chosen point to the box, and looks only at the chosen points whose nearest
//      distance to the box is at most min(U, r^2), with the reference's distance, in ascending
//      order with strict <, which gives the reference's label;
//   3. passes on only the labels that changed: the label in position order, the member counts of
//      rd_chain.hip's blocks, and a flag on the two chosen points whose members changed, which are
//      the only ones the ordering and the sums look at afterwards.
// The box distances round exactly as the reference's distance does, term by term and in the same
// order, and rounding is monotone, so for every sample p of the box and chosen point s
//   nearest(box, s) <= D_ref(p, s) <= farthest(box, s)
// holds for the computed values.  A chosen point with nearest > min(U, r^2) is therefore farther
// than the nearest one, or outside r: it cannot be the label.  The same holds in step 1: the chosen
// points within `bound` are where they were, so the label is too.
//
// Bounds: with every block evaluated, ~2 passes over the segment's K chosen points per 512 samples
// (~40 operations per 64 x 1 pairs of chosen points and boxes) and ~10 exact distances a sample,
// instead of K screened ones; once few points move, one load of their flags per block.
#include "rd_spatial.hpp"
#include "rd_chain.hpp"

namespace rdhip {

namespace {

template <typename T>
__device__ __forceinline__ T wave_min(T v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o));
    return v;
}
template <typename T>
__device__ __forceinline__ T wave_max(T v) {
#pragma unroll
    for (int o = kWave / 2; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o));
    return v;
}

// lower and upper corner of a block's samples: each thread's lo / hi reduced over the block
template <typename T, int DIM, int W>
__device__ __forceinline__ void block_corners(T (&lo)[DIM], T (&hi)[DIM], T* out, T (&sh)[W][2 * DIM]) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = wave_min(lo[d]);
        hi[d] = wave_max(hi[d]);
        if (lane == 0) {
            sh[wave][d] = lo[d];
            sh[wave][DIM + d] = hi[d];
        }
    }
    __syncthreads();
    if ((int)threadIdx.x < DIM) {
        T l = sh[0][threadIdx.x], h = sh[0][DIM + threadIdx.x];
        for (int w = 1; w < W; ++w) {
            l = fmin(l, sh[w][threadIdx.x]);
            h = fmax(h, sh[w][DIM + threadIdx.x]);
        }
        out[threadIdx.x] = l;
        out[DIM + threadIdx.x] = h;
    }
}

template <typename T, int DIM>
__global__ __launch_bounds__(256) void spatial_bounds_kernel(SpatialBuild<T> b) {
    __shared__ T sh[4][2 * DIM];
    const WorkItem it = b.items[blockIdx.x];
    const SegDesc sd = b.segs[it.seg];
    T lo[DIM], hi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = FpTraits<T>::big;
        hi[d] = -FpTraits<T>::big;
    }
    for (int i = it.start + (int)threadIdx.x; i < it.end; i += 256) {
        const int64_t n = point_of(b.pIndex, sd.pOff + i);
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            // infinities stay out: they would leave every finite sample in one cell
            const T x = b.P[d * b.pStride + n];
            if (!(fabs(x) < FpTraits<T>::big)) continue;
            lo[d] = fmin(lo[d], x);
            hi[d] = fmax(hi[d], x);
        }
    }
    block_corners<T, DIM, 4>(lo, hi, b.partial + (int64_t)blockIdx.x * 2 * DIM, sh);
}

// One wave per segment: its corners, then the sides to halve, always the longest one.
template <typename T, int DIM>
__global__ __launch_bounds__(kWave) void spatial_map_kernel(SpatialBuild<T> b) {
    const int s = blockIdx.x, lane = lane_id();
    T lo[DIM], hi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = FpTraits<T>::big;
        hi[d] = -FpTraits<T>::big;
    }
    for (int i = b.segFirstItem[s] + lane; i < b.segFirstItem[s + 1]; i += kWave)
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            lo[d] = fmin(lo[d], b.partial[(int64_t)i * 2 * DIM + d]);
            hi[d] = fmax(hi[d], b.partial[(int64_t)i * 2 * DIM + DIM + d]);
        }
    T side[DIM];
    int bits[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = wave_min(lo[d]);
        hi[d] = wave_max(hi[d]);
        side[d] = T(0.5) * hi[d] - T(0.5) * lo[d];   // half: finite
        bits[d] = 0;
    }
    unsigned long long split = 0;
    for (int q = 0; q < b.keyBits; ++q) {
        int best = 0;
        T w = side[0];
#pragma unroll
        for (int d = 1; d < DIM; ++d)
            if (side[d] > w) {
                w = side[d];
                best = d;
            }
        split |= (unsigned long long)best << (4 * q);
#pragma unroll
        for (int d = 0; d < DIM; ++d)
            if (d == best) {
                side[d] = side[d] * T(0.5);
                ++bits[d];
            }
    }
    if (lane != 0) return;
    SpatialMap<T>& m = b.maps[s];
    m.split = split;
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const T half = T(0.5) * hi[d] - T(0.5) * lo[d];
        const T cells = (T)(1 << bits[d]);
        m.lo[d] = lo[d];
        m.scale[d] = half > T(0) ? T(0.5) * cells / half : T(0);
        m.bits[d] = bits[d];
    }
}

template <typename T, int DIM>
__global__ __launch_bounds__(256) void spatial_key_kernel(SpatialBuild<T> b) {
    const WorkItem it = b.items[blockIdx.x];
    const SegDesc sd = b.segs[it.seg];
    const SpatialMap<T>& m = b.maps[it.seg];
    for (int i = it.start + (int)threadIdx.x; i < it.end; i += 256) {
        const int64_t n = point_of(b.pIndex, sd.pOff + i);
        int cell[DIM], left[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const T f = (b.P[d * b.pStride + n] - m.lo[d]) * m.scale[d];
            const int top = (1 << m.bits[d]) - 1;
            cell[d] = f >= (T)top ? top : f > T(0) ? (int)f : 0;   // NaN: 0
            left[d] = m.bits[d];
        }
        int key = 0;
        for (int q = 0; q < b.keyBits; ++q) {
            const int sd2 = (int)(m.split >> (4 * q)) & 15;
#pragma unroll
            for (int d = 0; d < DIM; ++d)
                if (d == sd2) {
                    --left[d];
                    key = (key << 1) | ((cell[d] >> left[d]) & 1);
                }
        }
        b.keys[sd.pOff + i] = (int)((unsigned)it.seg << b.keyBits) | key;
    }
}

template <typename T, int DIM>
__global__ __launch_bounds__(256) void spatial_gather_kernel(const T* __restrict__ P, int64_t pStride,
                                                             const int* __restrict__ pIndex,
                                                             const int* __restrict__ perm, int64_t n,
                                                             T* __restrict__ Q, int64_t qStride) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int64_t src = point_of(pIndex, perm[i]);
#pragma unroll
        for (int d = 0; d < DIM; ++d) Q[d * qStride + i] = P[d * pStride + src];
    }
}

template <typename T, int DIM>
__global__ __launch_bounds__(kBoxThreads) void spatial_box_kernel(const T* __restrict__ Q, int64_t qStride,
                                                                  const WorkItem* __restrict__ items,
                                                                  const SegDesc* __restrict__ segs,
                                                                  T* __restrict__ box) {
    __shared__ T sh[kBoxThreads / kWave][2 * DIM];
    const WorkItem it = items[blockIdx.x];
    const int64_t p0 = segs[it.seg].pOff;
    T lo[DIM], hi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = FpTraits<T>::big;
        hi[d] = -FpTraits<T>::big;
    }
    for (int i = it.start + (int)threadIdx.x; i < it.end; i += kBoxThreads)
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
            const T x = Q[d * qStride + p0 + i];   // a NaN coordinate's sample has no label
            lo[d] = fmin(lo[d], x);
            hi[d] = fmax(hi[d], x);
        }
    block_corners<T, DIM, kBoxThreads / kWave>(lo, hi, box + (int64_t)it.pad * 2 * DIM, sh);
}

// smallest and largest computed distance of the box's samples to s (see above)
template <typename T, int DIM>
__device__ __forceinline__ T box_nearest(const T (&lo)[DIM], const T (&hi)[DIM], const T (&s)[DIM]) {
    T acc = T(0);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const T t = fmax(fmax(lo[d] - s[d], s[d] - hi[d]), T(0));
        const T sq = t * t;
        acc = acc + sq;
    }
    return acc;
}
template <typename T, int DIM>
__device__ __forceinline__ T box_farthest(const T (&lo)[DIM], const T (&hi)[DIM], const T (&s)[DIM]) {
    T acc = T(0);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        const T t = fmax(fabs(lo[d] - s[d]), fabs(hi[d] - s[d]));
        const T sq = t * t;
        acc = acc + sq;
    }
    return acc;
}

template <typename T, int DIM, bool kFirst>
__global__ __launch_bounds__(kBoxThreads) void box_scan_kernel(BoxScanArgs<T> a) {
    constexpr int kW = kBoxThreads / kWave, kPer = kBoxSamples / kBoxThreads;
    __shared__ T cs[DIM][kBoxThreads];
    __shared__ int ck[kBoxThreads];
    __shared__ int wcnt[kW];
    __shared__ T wmin[kW];
    if (*a.allDone) return;
    const int nItems = a.numItemsDev ? *a.numItemsDev : (int)gridDim.x;
    if ((int)blockIdx.x >= nItems) return;
    const WorkItem it = a.items[xcd_item(blockIdx.x, nItems)];
    if (a.segDone[it.seg]) return;
    const SegDesc sd = a.segs[it.seg];
    const int K = a.segK[it.seg];
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const int64_t ss = a.sStride;
    const T* __restrict__ Sb = a.S + sd.sOff;
    T lo[DIM], hi[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
        lo[d] = a.box[(int64_t)it.pad * 2 * DIM + d];
        hi[d] = a.box[(int64_t)it.pad * 2 * DIM + DIM + d];
    }
    if constexpr (!kFirst) {
        const T bound = a.bound[it.pad];
        const T* __restrict__ So = a.Sold + sd.sOff;
        bool hit = false;
        for (int k = tid; k < K; k += kBoxThreads) {
            if (!a.moved[sd.sOff + k]) continue;
            T s[DIM], o[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) {
                s[d] = Sb[d * ss + k];
                o[d] = So[d * ss + k];
            }
            hit = hit || !(box_nearest<T, DIM>(lo, hi, s) > bound) || !(box_nearest<T, DIM>(lo, hi, o) > bound);
        }
        if (!__syncthreads_or(hit)) return;
    }
    T p[kPer][DIM];
    int64_t pos[kPer];
    bool valid[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = it.start + j * kBoxThreads + tid;
        valid[j] = i < it.end;
        pos[j] = sd.pOff + (valid[j] ? i : it.start);
#pragma unroll
        for (int d = 0; d < DIM; ++d) p[j][d] = a.Q[d * a.qStride + pos[j]];
    }
    const T rSqr = a.segRSqr[it.seg];
    T far = FpTraits<T>::big;
    for (int k = tid; k < K; k += kBoxThreads) {
        T s[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) s[d] = Sb[d * ss + k];
        far = fmin(far, box_farthest<T, DIM>(lo, hi, s));
    }
    far = wave_min(far);
    if (lane == 0) wmin[wave] = far;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < kW; ++w) far = fmin(far, wmin[w]);
    const T bound = fmin(far, rSqr);
    if (tid == 0) a.bound[it.pad] = bound;

    T best[kPer];
    int at[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        best[j] = FpTraits<T>::big;
        at[j] = -1;
    }
    for (int c0 = 0; c0 < K; c0 += kBoxThreads) {
        const int k = c0 + tid;
        T s[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) s[d] = Sb[d * ss + min(k, K - 1)];
        const bool cand = k < K && !(box_nearest<T, DIM>(lo, hi, s) > bound);
        const uint64_t m = __ballot(cand);
        if (lane == 0) wcnt[wave] = __popcll(m);
        __syncthreads();
        int o = __popcll(m & lanes_below()), n = 0;
#pragma unroll
        for (int w = 0; w < kW; ++w) {
            o += w < wave ? wcnt[w] : 0;
            n += wcnt[w];
        }
        if (cand) {
            ck[o] = k;
#pragma unroll
            for (int d = 0; d < DIM; ++d) cs[d][o] = s[d];
        }
        __syncthreads();
        for (int c = 0; c < n; ++c) {
            const int kc = ck[c];
            T sc[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) sc[d] = cs[d][c];
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const T e = exact_sqdist<T, DIM>(p[j], sc);
                const bool closer = e < best[j];
                best[j] = closer ? e : best[j];
                at[j] = closer ? kc : at[j];
            }
        }
        __syncthreads();   // cs, ck and wcnt are rewritten
    }
    const int nb = (sd.nP + a.itemSize - 1) / a.itemSize;
    int* __restrict__ hist = a.hist + a.histSegOff[it.seg];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (!valid[j]) continue;
        const int l = at[j] >= 0 && best[j] <= rSqr ? (int)(sd.sOff + at[j]) : -1;
        if constexpr (kFirst) {
            a.labS[pos[j]] = l;
            a.labels[a.perm[pos[j]]] = l;
        } else {
            const int was = a.labS[pos[j]];
            if (l == was) continue;
            a.labS[pos[j]] = l;
            const int at0 = a.perm[pos[j]];
            a.labels[at0] = l;
            const int col = (int)(at0 - sd.pOff) / a.itemSize;
            if (was >= 0) {
                atomicAdd(&hist[(int64_t)(was - sd.sOff) * nb + col], -1);
                a.touched[was] = 1;
            }
            if (l >= 0) {
                atomicAdd(&hist[(int64_t)(l - sd.sOff) * nb + col], 1);
                a.touched[l] = 1;
            }
        }
    }
}

__global__ __launch_bounds__(256) void label_hist_kernel(const WorkItem* __restrict__ items,
                                                         const int* __restrict__ numItemsDev,
                                                         const SegDesc* __restrict__ segs,
                                                         const int* __restrict__ segK,
                                                         const int* __restrict__ segDone,
                                                         const int* __restrict__ labels, int* __restrict__ hist,
                                                         const int64_t* __restrict__ histSegOff, int itemSize,
                                                         const int* __restrict__ allDone) {
    __shared__ int lh[kChainMaxKeys];
    if (*allDone) return;
    const int n = numItemsDev ? *numItemsDev : (int)gridDim.x;
    if ((int)blockIdx.x >= n) return;
    const WorkItem it = items[xcd_item(blockIdx.x, n)];
    if (segDone[it.seg]) return;
    const SegDesc sd = segs[it.seg];
    const int K = min(segK[it.seg], kChainMaxKeys);
    for (int k = threadIdx.x; k < K; k += 256) lh[k] = 0;
    __syncthreads();
    for (int i = it.start + (int)threadIdx.x; i < it.end; i += 256) {
        const int k = labels[sd.pOff + i] - (int)sd.sOff;
        if (k >= 0 && k < K) atomicAdd(&lh[k], 1);
    }
    __syncthreads();
    const int nb = (sd.nP + itemSize - 1) / itemSize;
    int* __restrict__ col = hist + histSegOff[it.seg] + it.start / itemSize;
    for (int k = threadIdx.x; k < K; k += 256) col[(int64_t)k * nb] = lh[k];
}

}  // namespace

template <typename T>
hipError_t launch_spatial_keys(const SpatialBuild<T>& b, int dim, hipStream_t st) {
    if (b.numItems <= 0) return hipSuccess;
    bool ok = false;
    RD_DISPATCH_DIM(dim, {
        hipLaunchKernelGGL((spatial_bounds_kernel<T, DIM>), dim3(b.numItems), dim3(256), 0, st, b);
        hipLaunchKernelGGL((spatial_map_kernel<T, DIM>), dim3(b.numSegs), dim3(kWave), 0, st, b);
        hipLaunchKernelGGL((spatial_key_kernel<T, DIM>), dim3(b.numItems), dim3(256), 0, st, b);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_spatial_gather(const T* P, int64_t pStride, const int* pIndex, const int* perm, int64_t n, int dim,
                                 T* Q, int64_t qStride, hipStream_t st) {
    const unsigned blocks = (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + 255) / 256, 65536));
    bool ok = false;
    RD_DISPATCH_DIM(dim, {
        hipLaunchKernelGGL((spatial_gather_kernel<T, DIM>), dim3(blocks), dim3(256), 0, st, P, pStride, pIndex, perm,
                           n, Q, qStride);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_spatial_boxes(const T* Q, int64_t qStride, const WorkItem* items, const SegDesc* segs, int numItems,
                                int dim, T* box, hipStream_t st) {
    if (numItems <= 0) return hipSuccess;
    bool ok = false;
    RD_DISPATCH_DIM(dim, {
        hipLaunchKernelGGL((spatial_box_kernel<T, DIM>), dim3(numItems), dim3(kBoxThreads), 0, st, Q, qStride, items,
                           segs, box);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_box_scan(const BoxScanArgs<T>& a, int dim, int numItems, bool first, hipStream_t st) {
    if (numItems <= 0) return hipSuccess;
    bool ok = false;
    RD_DISPATCH_DIM(dim, {
        if (first)
            hipLaunchKernelGGL((box_scan_kernel<T, DIM, true>), dim3(numItems), dim3(kBoxThreads), 0, st, a);
        else
            hipLaunchKernelGGL((box_scan_kernel<T, DIM, false>), dim3(numItems), dim3(kBoxThreads), 0, st, a);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

hipError_t launch_label_hist(const WorkItem* items, const int* numItemsDev, int numItems, const SegDesc* segs,
                             const int* segK, const int* segDone, const int* labels, int* hist,
                             const int64_t* histSegOff, int itemSize, const int* allDone, hipStream_t st) {
    if (numItems <= 0) return hipSuccess;
    hipLaunchKernelGGL(label_hist_kernel, dim3(numItems), dim3(256), 0, st, items, numItemsDev, segs, segK, segDone,
                       labels, hist, histSegOff, itemSize, allDone);
    return hipGetLastError();
}

#define RD_SPATIAL_INSTANCES(T)                                                                                   \
    template hipError_t launch_spatial_keys<T>(const SpatialBuild<T>&, int, hipStream_t);                          \
    template hipError_t launch_spatial_gather<T>(const T*, int64_t, const int*, const int*, int64_t, int, T*,      \
                                                 int64_t, hipStream_t);                                            \
    template hipError_t launch_spatial_boxes<T>(const T*, int64_t, const WorkItem*, const SegDesc*, int, int, T*,  \
                                                hipStream_t);                                                      \
    template hipError_t launch_box_scan<T>(const BoxScanArgs<T>&, int, int, bool, hipStream_t);
RD_SPATIAL_INSTANCES(float)
RD_SPATIAL_INSTANCES(double)
#undef RD_SPATIAL_INSTANCES

}  // namespace rdhip
