// rd_choose.hip -- greedy choose (rd/cpu/brute_force/choose.hpp:36-70) for a batch of segments.
//
// Semantics: sample 0 is chosen; sample i is chosen iff no already chosen sample lies at
// squared distance <= r*r (exact reference distance).  The decision depends on every
// earlier decision, so candidates are decided in sample order, a batch of one candidate per
// thread of a block at a time (resolve_batch):
//   * every wave builds the 64 x 64 conflict bits of its own candidates in parallel (a
//     candidate's coordinates reach the other lanes by v_readlane);
//   * the waves then take turns: the wave whose turn it is walks its surviving candidates in
//     order with scalar bit operations only (the first survivor is chosen and its conflict
//     word clears the candidates it covers), publishes the points it chose in LDS, and the
//     later waves drop the candidates they cover.
// Segments of at most a few thousand own samples run all batches in one block.  Large segments
// keep one "open" bit per sample and alternate two launches: resolve (one block takes the first
// 1024 open samples in order and decides them) and filter (the whole GPU tests the samples still
// open against the points just chosen).  Every open sample has been tested against all chosen
// points but those of the last resolve, so the bits are exactly the samples the serial walk
// would still have to look at.  Output per segment: K, the chosen coordinates in the segment's
// slots and the chosen samples' indices (segment-relative, ascending).
//
// Bounds: the filter is VALU work, one pass over the samples per chosen point and no more in
// total than one evolve scan; resolve is a dependence chain of ~40 cycles per chosen point.  The
// form this replaces decided one survivor per block-wide barrier (~200 us per 256 samples that are
// mostly chosen) and walked every 256 samples of a large cloud with one block (~0.7 us each, also
// when all were covered).  Choose phase before -> after: 200k 6-D points with ~11,000 chosen
// 173 -> 3.1 ms (13 resolves of 0.12 ms, 12 filters of 0.118 ms); 1M helix 6.2 -> 0.27 ms (filters
// of 21 us); 20k spiral 1.49 -> 0.14 ms (5 resolves of 12 us); 2k spiral, one block, 241 -> 53 us.
#include "rd_choose.hpp"

namespace rdhip {

namespace {

// LDS of resolve_batch: the points the current wave chose, double buffered so that one barrier
// separates a turn from the next.
template <typename T, int DIM>
struct TurnLds {
    T s[2][DIM][kWave];
    int n[2];
};

// Drops candidates covered by the chosen points [k0, k1) of the segment (in global memory, written
// by this block before a barrier or by an earlier launch): 64 points per coalesced load.
template <typename T, int DIM>
__device__ __forceinline__ bool drop_covered(const T (&p)[DIM], bool live, const T* Sb, int64_t ss, int k0, int k1,
                                             T rSqr) {
    const int lane = lane_id();
    for (int k = k0; k < k1; k += kWave) {
        if (!__ballot(live)) break;
        T q[DIM];
        const int kk = min(k + lane, k1 - 1);
#pragma unroll
        for (int d = 0; d < DIM; ++d) q[d] = Sb[d * ss + kk];
        const int m = min(kWave, k1 - k);
        for (int j = 0; j < m; ++j) {
            T s[DIM];
#pragma unroll
            for (int d = 0; d < DIM; ++d) s[d] = read_lane(q[d], j);
            if (exact_sqdist<T, DIM>(p, s) <= rSqr) live = false;
        }
    }
    return live;
}

// Decides one batch: thread t holds candidate t (coordinates p, sample index i; live: a candidate
// no chosen point covers so far), in sample order over the threads.  Appends the chosen ones to the
// segment's slots from K on and returns the new K.  Every thread of the block takes part; n waves
// (the first ones) hold candidates.
template <typename T, int DIM>
__device__ __forceinline__ int resolve_batch(const T (&p)[DIM], int i, bool live, int waves, T rSqr, T* Sb,
                                             int64_t ss, int* cidx, int K, int cap, TurnLds<T, DIM>& sh) {
    const int lane = lane_id(), wave = threadIdx.x / kWave;
    const uint64_t below = lanes_below();
    // bit j: lane j's candidate conflicts with this lane's
    uint64_t row = 0;
    {
        const uint64_t alive = __ballot(live);
        if (alive & (alive - 1))
            for (uint64_t m = alive; m; m &= m - 1) {
                const int j = __builtin_ctzll(m);
                T s[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) s[d] = read_lane(p[d], j);
                row |= exact_sqdist<T, DIM>(p, s) <= rSqr ? (uint64_t(1) << j) : 0;
            }
    }
    for (int g = 0; g < waves; ++g) {
        const int buf = g & 1;
        if (wave == g) {
            uint64_t al = __ballot(live), ch = 0;
            while (al) {
                const int j = __builtin_ctzll(al);
                const uint64_t bit = uint64_t(1) << j;
                ch |= bit;
                al &= ~(read_lane(row, j) | bit);
            }
            if ((ch >> lane) & 1) {
                const int r = __popcll(ch & below);
#pragma unroll
                for (int d = 0; d < DIM; ++d) sh.s[buf][d][r] = p[d];
                if (K + r < cap) {
#pragma unroll
                    for (int d = 0; d < DIM; ++d) Sb[d * ss + K + r] = p[d];
                    cidx[K + r] = i;
                }
            }
            if (lane == 0) sh.n[buf] = __popcll(ch);
        }
        __syncthreads();
        const int n = sh.n[buf];
        K += n;
        if (wave > g && __ballot(live))
            for (int c = 0; c < n; ++c) {
                T s[DIM];
#pragma unroll
                for (int d = 0; d < DIM; ++d) s[d] = sh.s[buf][d][c];
                if (exact_sqdist<T, DIM>(p, s) <= rSqr) live = false;
            }
    }
    __syncthreads();   // the last turn's points are read before the next batch's first turn
    return K;
}

}  // namespace

// One block per small segment.
template <typename T, int DIM, int TH>
__global__ __launch_bounds__(TH) void choose_small_kernel(ChooseArgs<T> a) {
    __shared__ TurnLds<T, DIM> sh;
    const int seg = blockIdx.x;
    if (seg >= a.numSegs || (a.segLarge && a.segLarge[seg])) return;
    const SegDesc sd = a.segs[seg];
    const int n = sd.nOwn;
    const T rSqr = a.segRSqr[seg];
    T* Sb = a.S + sd.sOff;
    int* cidx = a.chosenIdx + sd.sOff;
    int K = 0;
    for (int c0 = 0; c0 < n; c0 += TH) {
        const int i = c0 + (int)threadIdx.x;
        bool live = i < n;
        const int64_t src = point_of(a.pIndex, sd.pOff + (live ? i : c0));
        T p[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) p[d] = a.P[d * a.pStride + src];
        live = drop_covered<T, DIM>(p, live, Sb, a.sStride, 0, K, rSqr);
        const int waves = (min(TH, n - c0) + kWave - 1) / kWave;
        K = resolve_batch<T, DIM>(p, i, live, waves, rSqr, Sb, a.sStride, cidx, K, sd.sCap, sh);
        if (K > sd.sCap) {
            if (threadIdx.x == 0) atomicOr(a.overflow, 1);
            K = sd.sCap;
            break;
        }
    }
    if (threadIdx.x == 0) a.segK[seg] = K;
}

namespace {
// the large segment of a filter block
__device__ __forceinline__ int block_segment(const int* __restrict__ first, int n, int block) {
    int lo = 0, hi = n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (first[mid] <= block) lo = mid; else hi = mid - 1;
    }
    return lo;
}
}  // namespace

template <typename T>
__global__ __launch_bounds__(256) void choose_open_kernel(ChooseArgs<T> a, int numBlocks) {
    const int b = blockIdx.x * 64 + threadIdx.x / 4;   // filter block; thread: one of its 4 words
    if (b < numBlocks) {
        const int l = block_segment(a.largeBlock, a.numLarge, b);
        const int seg = a.largeSeg[l];
        const int first = (b - a.largeBlock[l]) * kChooseBlock + (int)(threadIdx.x & 3) * kWave;
        const int left = a.segs[seg].nOwn - first;
        a.open[(int64_t)b * 4 + (threadIdx.x & 3)] =
            left >= kWave ? ~uint64_t(0) : left > 0 ? (uint64_t(1) << left) - 1 : 0;
        if (first == 0) {
            a.segK[seg] = 0;
            a.base[l] = 0;
            a.cursor[l] = 0;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) *a.doneCount = 0;
}

// One wave per word of 64 samples: no block-wide work, so a word without open samples costs one
// load.  256 samples a block keep a 20k-point cloud on 80 CUs.
template <typename T, int DIM>
__global__ __launch_bounds__(kChooseBlock) void choose_filter_kernel(ChooseArgs<T> a, int block0, int fresh) {
    const int b = block0 + (int)blockIdx.x;
    const int l = block_segment(a.largeBlock, a.numLarge, b);
    const int seg = a.largeSeg[l];
    const int w = __builtin_amdgcn_readfirstlane((b - a.largeBlock[l]) * 4 + (int)(threadIdx.x / kWave));
    if (!fresh && w < a.cursor[l]) return;
    uint64_t* word = a.open + (int64_t)a.largeBlock[l] * 4 + w;
    const SegDesc sd = a.segs[seg];
    const int lane = lane_id();
    const int i = w * kWave + lane;
    const uint64_t was = fresh ? __ballot(i < sd.nOwn) : *word;
    if (was == 0) {
        if (fresh && lane == 0) *word = 0;
        return;
    }
    const int k0 = fresh ? 0 : a.base[l], K = a.segK[seg];
    const T rSqr = a.segRSqr[seg];
    const T* __restrict__ Sb = a.S + sd.sOff;
    const int64_t ss = a.sStride;
    bool live = (was >> lane) & 1;
    const int64_t src = point_of(a.pIndex, sd.pOff + (live ? i : 0));
    T p[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) p[d] = a.P[d * a.pStride + src];
    constexpr int kG = 8;   // chosen points per group of scalar loads
    int k = k0;
    for (; k + kG <= K; k += kG) {
        T s[kG][DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d)
#pragma unroll
            for (int j = 0; j < kG; ++j) s[j][d] = Sb[d * ss + k + j];
#pragma unroll
        for (int j = 0; j < kG; ++j) live = live && !(exact_sqdist<T, DIM>(p, s[j]) <= rSqr);
        if (!__ballot(live)) {
            k = K;   // all covered: nothing is left for the remainder either
            break;
        }
    }
    for (; k < K; ++k) {
        T s[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) s[d] = Sb[d * ss + k];
        live = live && !(exact_sqdist<T, DIM>(p, s) <= rSqr);
    }
    const uint64_t now = __ballot(live);
    if (lane == 0 && (fresh || now != was)) *word = now;
}

// One block per large segment: the first open samples in order, a batch at a time.
template <typename T, int DIM>
__global__ __launch_bounds__(kChooseBatch) void choose_resolve_kernel(ChooseArgs<T> a, int endSample,
                                                                      int maxBatches) {
    __shared__ TurnLds<T, DIM> sh;
    __shared__ int cand[kChooseBatch];
    __shared__ int wsum[kChooseBatch / kWave];
    __shared__ int lastWord;
    const int l = blockIdx.x;
    const int seg = a.largeSeg[l];
    const SegDesc sd = a.segs[seg];
    const int n = endSample >= 0 ? min(endSample, sd.nOwn) : sd.nOwn;
    const int words = (n + kWave - 1) / kWave;
    int w0 = a.cursor[l];
    if (w0 >= words) return;
    uint64_t* open = a.open + (int64_t)a.largeBlock[l] * 4;
    const T rSqr = a.segRSqr[seg];
    T* Sb = a.S + sd.sOff;
    int* cidx = a.chosenIdx + sd.sOff;
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const int kBase = a.segK[seg];   // every open sample has been tested against these
    int K = kBase;
    for (int batch = 0; w0 < words && (maxBatches == 0 || batch < maxBatches); ++batch) {
        // the first kChooseBatch open samples from word w0 on, in order
        constexpr int kPer = 2;
        int got = 0, w = w0;
        while (got < kChooseBatch && w < words) {
            uint64_t v[kPer];
            int c = 0;
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int x = w + tid * kPer + j;
                v[j] = x < words ? open[x] : 0;
                c += __popcll(v[j]);
            }
            int incl = c;
#pragma unroll
            for (int o = 1; o < kWave; o <<= 1) {
                const int y = __shfl_up(incl, o);
                if (lane >= o) incl += y;
            }
            if (lane == kWave - 1) wsum[wave] = incl;
            __syncthreads();
            int at = got + incl - c, total = 0;
#pragma unroll
            for (int u = 0; u < kChooseBatch / kWave; ++u) {
                at += u < wave ? wsum[u] : 0;
                total += wsum[u];
            }
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const int x = w + tid * kPer + j;
                uint64_t m = v[j];
                while (m && at < kChooseBatch) {
                    cand[at] = x * kWave + __builtin_ctzll(m);
                    if (at == kChooseBatch - 1) lastWord = x;
                    m &= m - 1;
                    ++at;
                }
                if (m != v[j]) open[x] = m;
            }
            got += total;
            w += kChooseBatch * kPer;
            __syncthreads();
        }
        const int m = min(got, kChooseBatch);
        w0 = got >= kChooseBatch ? lastWord : words;
        if (m == 0) break;
        bool live = tid < m;
        const int i = cand[live ? tid : 0];
        const int64_t src = point_of(a.pIndex, sd.pOff + i);
        T p[DIM];
#pragma unroll
        for (int d = 0; d < DIM; ++d) p[d] = a.P[d * a.pStride + src];
        live = drop_covered<T, DIM>(p, live, Sb, a.sStride, kBase, K, rSqr);
        K = resolve_batch<T, DIM>(p, i, live, (m + kWave - 1) / kWave, rSqr, Sb, a.sStride, cidx, K, sd.sCap, sh);
        if (K > sd.sCap) {
            if (tid == 0) atomicOr(a.overflow, 1);
            K = sd.sCap;
            w0 = words;
        }
    }
    if (tid == 0) {
        a.segK[seg] = K;
        a.base[l] = kBase;
        a.cursor[l] = w0;
        if (w0 >= words) atomicAdd(a.doneCount, 1);
    }
}

template <typename T>
hipError_t launch_choose_small(const ChooseArgs<T>& a, int dim, hipStream_t st) {
    if (a.numSegs <= 0) return hipSuccess;
    bool ok = false;
    // many segments (tiles) fill the GPU with small blocks; a few take the widest block each
    RD_DISPATCH_DIM(dim, {
        if (a.numSegs > 256)
            hipLaunchKernelGGL((choose_small_kernel<T, DIM, 256>), dim3(a.numSegs), dim3(256), 0, st, a);
        else
            hipLaunchKernelGGL((choose_small_kernel<T, DIM, 1024>), dim3(a.numSegs), dim3(1024), 0, st, a);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_choose_open(const ChooseArgs<T>& a, int numBlocks, hipStream_t st) {
    if (numBlocks <= 0) return hipSuccess;
    hipLaunchKernelGGL((choose_open_kernel<T>), dim3((unsigned)((numBlocks + 63) / 64)), dim3(256), 0, st, a,
                       numBlocks);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_choose_filter(const ChooseArgs<T>& a, int dim, int block0, int numBlocks, bool fresh,
                                hipStream_t st) {
    if (numBlocks <= 0) return hipSuccess;
    bool ok = false;
    RD_DISPATCH_DIM(dim, {
        hipLaunchKernelGGL((choose_filter_kernel<T, DIM>), dim3((unsigned)numBlocks), dim3(kChooseBlock), 0, st, a,
                           block0, fresh ? 1 : 0);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

template <typename T>
hipError_t launch_choose_resolve(const ChooseArgs<T>& a, int dim, int endSample, int maxBatches, hipStream_t st) {
    if (a.numLarge <= 0) return hipSuccess;
    bool ok = false;
    RD_DISPATCH_DIM(dim, {
        hipLaunchKernelGGL((choose_resolve_kernel<T, DIM>), dim3((unsigned)a.numLarge), dim3(kChooseBatch), 0, st, a,
                           endSample, maxBatches);
        ok = true;
    });
    return ok ? hipGetLastError() : hipErrorInvalidValue;
}

#define RD_CHOOSE_INSTANCES(T)                                                                           \
    template hipError_t launch_choose_small<T>(const ChooseArgs<T>&, int, hipStream_t);                  \
    template hipError_t launch_choose_open<T>(const ChooseArgs<T>&, int, hipStream_t);                   \
    template hipError_t launch_choose_filter<T>(const ChooseArgs<T>&, int, int, int, bool, hipStream_t); \
    template hipError_t launch_choose_resolve<T>(const ChooseArgs<T>&, int, int, int, hipStream_t);
RD_CHOOSE_INSTANCES(float)
RD_CHOOSE_INSTANCES(double)
#undef RD_CHOOSE_INSTANCES

}  // namespace rdhip
