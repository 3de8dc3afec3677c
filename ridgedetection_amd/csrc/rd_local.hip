// rd_local.hip -- evolve of small segments (tiles, small clouds of a batch), one
// workgroup per segment, every iteration inside the workgroup.
//
// The batch-wide iteration (rd_evolve.hip) pays about fifteen launches and a device-wide
// sort per iteration, however little work is left; a segment of up to a few ten thousand
// samples iterates much faster on one CU with its chosen points, running sums and member
// lists in LDS.  Per iteration the samples are taken in chunks of kLocalChunk, in order:
//   1. labels: nearest chosen point of every sample of the chunk (rd_nearest.hpp, chosen
//      points read from LDS), stored as int16 in LDS;
//   2. stable counting sort of the chunk by label: wave w owns a contiguous range of the
//      chunk; it counts the labels of its range (ballot match, one LDS add per distinct
//      label and 64 samples), a block scan turns the counts into per-(wave, label) bases,
//      and the wave walks its range again placing every sample at base + rank among the
//      equal labels of its 64-sample chunk -- so each chosen point's members are listed in
//      sample order;
//   3. ordered sums: one 16-lane row per (coordinate, chosen point) continues that
//      point's running sum with the chunk's members in sample order (rd_rowsum.hpp: the
//      reference's serial sum);
// then 4. the shift rule updates the chosen points in LDS, and the workgroup repeats until
// no coordinate moved (or the iteration cap).  Results are bit-identical to the batch-wide
// path: same labels, same member order, same additions.  Reference:
// rd/cpu/brute_force/evolve.hpp:32-77 (labels, sums), 129-179 (shift), 237-459 (loop).
#include "rd_local.hpp"
#include "rd_nearest.hpp"
#include "rd_rowsum.hpp"

#include <algorithm>
#include <type_traits>

namespace rdhip {

namespace {

constexpr int kSmallInts = 16;   // wave totals of the block scan + two moved flags
constexpr int kLocalRing = 4;    // steps in flight in the ordered sums (members are L2-resident)

__host__ __device__ inline size_t align16(size_t v) { return (v + 15) / 16 * 16; }

// LDS layout: chosen coordinates [dim][kStride] | running sums [dim][kStride] | total
// counts, chunk counts, chunk offsets [kStride] each | per-wave bases [waves][kStride] |
// small ints | labels int16 [chunk] | order uint16 [chunk]
__host__ __device__ inline size_t lds_bytes(int dim, size_t vb, int kStride, int chunk) {
    return 2 * align16((size_t)dim * kStride * vb) + 4 * (size_t)kStride * (3 + kLocalWaves) + 4 * kSmallInts +
           2 * align16(2 * (size_t)chunk);
}

// LDS arrays of the segment-local kernels
template <typename T>
struct LocalLds {
    T* sS;
    T* run;
    int* cntT;
    int* cnt;
    int* off;
    int* wbase;   // [wave][label]
    int* small;   // [0, waves): wave totals; [14], [15]: moved flags
    short* lab;
    unsigned short* order;
    int ks;
};

template <typename T, int DIM>
__device__ __forceinline__ LocalLds<T> local_lds(char* smem, int ks, int chunk) {
    LocalLds<T> L;
    L.ks = ks;
    L.sS = reinterpret_cast<T*>(smem);
    L.run = reinterpret_cast<T*>(smem + align16((size_t)DIM * ks * sizeof(T)));
    L.cntT = reinterpret_cast<int*>(smem + 2 * align16((size_t)DIM * ks * sizeof(T)));
    L.cnt = L.cntT + ks;
    L.off = L.cnt + ks;
    L.wbase = L.off + ks;
    L.small = L.wbase + kLocalWaves * ks;
    L.lab = reinterpret_cast<short*>(L.small + kSmallInts);
    L.order = reinterpret_cast<unsigned short*>(reinterpret_cast<char*>(L.lab) + align16(2 * (size_t)chunk));
    return L;
}

// With the labels of samples c0 .. c0+cn-1 of the segment in lab[0 .. cn) (local chosen
// index or -1) and wbase zeroed (barrier passed): stable counting sort of the chunk by
// label into order, chunk counts/offsets into cnt/off, totals added to cntT, then every
// (coordinate, chosen point) running sum in run continued with the chunk's members in
// sample order.  Ends with a barrier.
template <typename T, int DIM>
__device__ __forceinline__ void sort_and_fold_chunk(const LocalArgs<T>& a, const LocalLds<T>& Ld, const SegDesc& sd,
                                                    int K, int c0, int cn, int bits) {
    const int ks = Ld.ks;
    short* lab = Ld.lab;
    int* wbase = Ld.wbase;
    int* small = Ld.small;
    int* cnt = Ld.cnt;
    int* off = Ld.off;
    int* cntT = Ld.cntT;
    T* run = Ld.run;
    unsigned short* order = Ld.order;
    const int tid = threadIdx.x;
    const int lane = tid & (kWave - 1);
    const int wave = tid / kWave;
    const uint64_t below = lanes_below();
    const int64_t ps = a.pStride;
    // ballot match: lanes whose label equals this lane's (valid lanes only)
    auto match = [&](int Lb) {
        const bool v = Lb >= 0;
        uint64_t m = __ballot(v);
        for (int b = 0; b < bits; ++b) {
            const bool bit = (Lb >> b) & 1;
            const uint64_t bb = __ballot(v && bit);
            m &= bit ? bb : ~bb;
        }
        return m;
    };
    // 2a. per-wave label counts over the wave's range of the chunk
    const int range = ((cn + kLocalWaves - 1) / kLocalWaves + kWave - 1) / kWave * kWave;
    const int r0 = min(cn, wave * range), r1 = min(cn, r0 + range);
    for (int q0 = r0; q0 < r1; q0 += kWave) {
        const int i = q0 + lane;
        const int L = i < r1 ? lab[i] : -1;
        const uint64_t m = match(L);
        if (L >= 0 && (m & below) == 0) wbase[wave * ks + L] += __popcll(m);
    }
    __syncthreads();

    // 2b. chunk counts, offsets (block exclusive scan, two labels per thread), wave bases
    {
        const int k0 = 2 * tid, k1 = 2 * tid + 1;
        int t0 = 0, t1 = 0;
        if (k0 < K)
            for (int w = 0; w < kLocalWaves; ++w) t0 += wbase[w * ks + k0];
        if (k1 < K)
            for (int w = 0; w < kLocalWaves; ++w) t1 += wbase[w * ks + k1];
        const int s = t0 + t1;
        int x = s;
#pragma unroll
        for (int o = 1; o < kWave; o <<= 1) {
            const int y = __shfl_up(x, o);
            if (lane >= o) x += y;
        }
        if (lane == kWave - 1) small[wave] = x;
        __syncthreads();
        int pre = 0;
        for (int w = 0; w < wave; ++w) pre += small[w];
        const int ex = pre + x - s;
        if (k0 < K) {
            off[k0] = ex;
            cnt[k0] = t0;
            cntT[k0] += t0;
            int r = ex;
            for (int w = 0; w < kLocalWaves; ++w) {
                const int c = wbase[w * ks + k0];
                wbase[w * ks + k0] = r;
                r += c;
            }
        }
        if (k1 < K) {
            off[k1] = ex + t0;
            cnt[k1] = t1;
            cntT[k1] += t1;
            int r = ex + t0;
            for (int w = 0; w < kLocalWaves; ++w) {
                const int c = wbase[w * ks + k1];
                wbase[w * ks + k1] = r;
                r += c;
            }
        }
    }
    __syncthreads();

    // 2c. placement in sample order.  Within a wave LDS operations complete in
    // issue order, so every lane reads its label's base before the leader advances it.
    for (int q0 = r0; q0 < r1; q0 += kWave) {
        const int i = q0 + lane;
        const int L = i < r1 ? lab[i] : -1;
        const uint64_t m = match(L);
        if (L >= 0) order[wbase[wave * ks + L] + __popcll(m & below)] = (unsigned short)i;
        if (L >= 0 && (m & below) == 0) wbase[wave * ks + L] += __popcll(m);
    }
    __syncthreads();

    // 3. running sums, rows of 16 lanes over (coordinate, chosen point)
    for (int rb = 0; rb < DIM * K; rb += kLocalThreads / 16) {
        const int row = rb + tid / 16;
        const bool act = row < DIM * K;
        const int d = act ? row / K : 0;
        const int k = act ? row - d * K : 0;
        const int c = act ? cnt[k] : 0;
        const int o = act ? off[k] : 0;
        const T* __restrict__ Pd = a.P + (int64_t)d * ps;
        const T sum = row_ordered_sum<T, kLocalRing>(
            wave_row_max(c),
            [&](int i) {
                const int pos = c > 0 ? (int)order[o + min(i, c - 1)] : 0;
                const T x = Pd[point_of(a.pIndex, sd.pOff + c0 + pos)];
                return i < c ? x : T(0);
            },
            act ? run[d * ks + k] : T(0));
        if (act && (tid & 15) == 0) run[d * ks + k] = sum;
    }
    __syncthreads();
}

template <typename T, int DIM, int PPT>
__global__ __launch_bounds__(kLocalThreads) void local_evolve_kernel(LocalArgs<T> a) {
    extern __shared__ __align__(16) char smem[];
    const int ks = a.kStride;
    const LocalLds<T> Ld = local_lds<T, DIM>(smem, ks, a.pCap);
    const int chunk = a.pCap;
    T* sS = Ld.sS;
    T* run = Ld.run;
    int* cntT = Ld.cntT;
    int* wbase = Ld.wbase;
    short* lab = Ld.lab;
    int* moved = Ld.small + 14;

    const int seg = a.list[blockIdx.x];
    const SegDesc sd = a.segs[seg];
    const int K = a.segK[seg];
    const int nP = sd.nP;
    const T rSqr = a.segRSqr[seg];
    const int tid = threadIdx.x;
    const int64_t ps = a.pStride;

    // chosen points into LDS, the far-away sentinel after K up to the end of the last tile
    const int kt = (K + kChosenTile - 1) / kChosenTile * kChosenTile;
    for (int i = tid; i < DIM * kt; i += kLocalThreads) {
        const int d = i / kt, k = i - d * kt;
        sS[d * ks + k] = k < K ? a.S[d * a.sStride + sd.sOff + k] : FpTraits<T>::sentinel;
    }
    if (tid < 2) moved[tid] = 0;
    __syncthreads();

    int iter = 0;
    if (K > 0 && nP > 0) {
        const int bits = K > 1 ? 32 - __clz(K - 1) : 1;
        for (;;) {
            for (int i = tid; i < DIM * K; i += kLocalThreads) run[(i / K) * ks + i % K] = T(0);
            for (int i = tid; i < K; i += kLocalThreads) cntT[i] = 0;
            for (int c0 = 0; c0 < nP; c0 += chunk) {
                const int cn = min(chunk, nP - c0);
                // 1. labels of the chunk
                for (int base = 0; base < cn; base += kLocalThreads * PPT) {
                    T p[PPT][DIM];
                    bool valid[PPT];
#pragma unroll
                    for (int j = 0; j < PPT; ++j) {
                        const int pos = base + tid + j * kLocalThreads;
                        valid[j] = pos < cn;
                        const int64_t src = valid[j] ? point_of(a.pIndex, sd.pOff + c0 + pos) : 0;
#pragma unroll
                        for (int d = 0; d < DIM; ++d) p[j][d] = valid[j] ? a.P[d * ps + src] : T(0);
                    }
                    int label[PPT];
                    nearest_labels<T, DIM, PPT>(p, valid, K, sS, ks, rSqr, label);
#pragma unroll
                    for (int j = 0; j < PPT; ++j)
                        if (valid[j]) lab[base + tid + j * kLocalThreads] = (short)label[j];
                }
                for (int i = tid; i < kLocalWaves * K; i += kLocalThreads) wbase[(i / K) * ks + i % K] = 0;
                __syncthreads();
                if (tid == 0 && c0 == 0) moved[(iter + 1) & 1] = 0;

                sort_and_fold_chunk<T, DIM>(a, Ld, sd, K, c0, cn, bits);
            }

            // 4. shift toward the mass centres
            for (int i = tid; i < DIM * K; i += kLocalThreads) {
                const int d = i / K, k = i - d * K;
                const int c = cntT[k];
                if (c == 0) continue;
                const T fc = (T)c;
                const T mc = run[d * ks + k] / fc;
                T thr = T(2) * fabs(mc);
                thr = thr * fc;
                thr = thr * FpTraits<T>::eps;
                T& s = sS[d * ks + k];
                if (fabs(mc - s) > thr) {
                    s = mc;
                    moved[iter & 1] = 1;
                }
            }
            __syncthreads();
            const bool any = moved[iter & 1] != 0;
            ++iter;
            if (!any || (a.maxIter > 0 && iter >= a.maxIter)) break;
            if (iter >= a.guard) {
                if (tid == 0) *a.error = 1;
                break;
            }
        }
    } else {
        iter = 1;   // the reference loop runs one pass that moves nothing
    }

    for (int i = tid; i < DIM * K; i += kLocalThreads) {
        const int d = i / K, k = i - d * K;
        a.S[d * a.sStride + sd.sOff + k] = sS[d * ks + k];
    }
    if (tid == 0) {
        a.segIter[seg] = iter;
        atomicMax(a.maxIters, iter);
    }
}

// ---------------------------------------------------------------------------------
// The same loop with the segment's samples in LDS (segments that fit), and only the work the last
// iteration's moves call for.  Every sample keeps its nearest chosen point and that distance: while
// that point stays put, only the points that moved can replace it, so the sample is compared with
// those alone; the samples whose own point moved are listed and compared with every chosen point.
// Distances are the reference's and equal ones go to the lower index, which is the reference's
// first-index rule.  A chain whose members did not change has the sum it had, and its point cannot
// move, so only the other chains are sorted and summed.
//
// Bound: one CU's VALU rate over (listed samples) x K distances in the first iterations, then the
// latency of the phases' ~10 barriers.  2,000 2-D samples in double with 150-180 chosen points:
// 255 us per launch (24 us per iteration) against 498 us for the kernel above, which compares all
// pairs and gathers its members from memory.  Tiles of a 120,000-sample 4-D chain: 722 us against
// 1,001 us.  With chosen points one coordinate after the other and two samples a lane: 306 and 748.
// ---------------------------------------------------------------------------------
constexpr int kMemThreads = 1024;
constexpr int kMemWaves = kMemThreads / kWave;

// values between chosen points in LDS: a point's coordinates are one wide read
__host__ __device__ constexpr int mem_point_stride(int dim) { return dim == 3 ? 4 : dim; }

__host__ __device__ inline size_t mem_lds_bytes(int dim, size_t vb, int kStride, int pCap) {
    return align16((size_t)mem_point_stride(dim) * kStride * vb) + align16((size_t)dim * kStride * vb) + align16((size_t)dim * pCap * vb) + align16((size_t)pCap * vb) +
           4 * (size_t)kStride * (6 + kMemWaves) + 4 * 32 + 4 * align16(2 * (size_t)pCap);
}

template <typename T, int DIM>
__global__ __launch_bounds__(kMemThreads) void local_mem_kernel(LocalArgs<T> a) {
    extern __shared__ __align__(16) char smem[];
    const int ks = a.kStride, pc = a.pCap;
    char* at = smem;
    auto take = [&](size_t bytes) {
        char* q = at;
        at += align16(bytes);
        return q;
    };
    constexpr int kSt = mem_point_stride(DIM);
    T* sS = reinterpret_cast<T*>(take((size_t)kSt * ks * sizeof(T)));    // chosen points, one after the other
    T* sum = reinterpret_cast<T*>(take((size_t)DIM * ks * sizeof(T)));   // by place in `touched`
    T* x = reinterpret_cast<T*>(take((size_t)DIM * pc * sizeof(T)));     // samples
    T* dist = reinterpret_cast<T*>(take((size_t)pc * sizeof(T)));        // to the nearest chosen point
    int* cnt = reinterpret_cast<int*>(at);   // members, first member in `order`: touched chains
    int* off = cnt + ks;
    int* touched = off + ks;                 // chains whose members changed, in index order
    int* tflag = touched + ks;               // touched, then place in `touched` + 1
    int* movedL = tflag + ks;                // chosen points moved by the last iteration
    int* mflag = movedL + ks;
    int* wbase = mflag + ks;                 // [wave][ks]
    int* small = wbase + kMemWaves * ks;     // [0, 16): wave totals; then counters
    int* nList = small + 16;
    int* nMoved = small + 17;
    at = reinterpret_cast<char*>(small + 32);
    short* near = reinterpret_cast<short*>(take(2 * (size_t)pc));   // nearest chosen point, -1: none
    short* lab = reinterpret_cast<short*>(take(2 * (size_t)pc));    // the same within r, else -1
    unsigned short* order = reinterpret_cast<unsigned short*>(take(2 * (size_t)pc));
    unsigned short* list = reinterpret_cast<unsigned short*>(take(2 * (size_t)pc));

    const int seg = a.list[blockIdx.x];
    const SegDesc sd = a.segs[seg];
    const int K = a.segK[seg], nP = sd.nP;
    const T rSqr = a.segRSqr[seg];
    const int tid = threadIdx.x, lane = lane_id(), wave = tid / kWave;
    const uint64_t below = lanes_below();

    for (int i = tid; i < DIM * K; i += kMemThreads) sS[(i % K) * kSt + i / K] = a.S[(i / K) * a.sStride + sd.sOff + i % K];
    for (int i = tid; i < nP; i += kMemThreads) {
        const int64_t src = point_of(a.pIndex, sd.pOff + i);
#pragma unroll
        for (int d = 0; d < DIM; ++d) x[d * pc + i] = a.P[d * a.pStride + src];
        lab[i] = -1;
    }
    for (int k = tid; k < ks; k += kMemThreads) {
        tflag[k] = 1;   // the first iteration sums every chain
        mflag[k] = 0;
    }
    int iter = 0;
    if (K > 0 && nP > 0) {
        const int bits = K > 1 ? 32 - __clz(K - 1) : 1;
        auto sample = [&](int i, T(&p)[DIM]) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) p[d] = x[d * pc + i];
        };
        auto chosen = [&](int k, T(&s)[DIM]) {
#pragma unroll
            for (int d = 0; d < DIM; ++d) s[d] = sS[k * kSt + d];
        };
        // a sample's new nearest point; chains that lose or gain it are touched
        auto settle = [&](int i, T e, int k) {
            dist[i] = e;
            near[i] = (short)k;
            const int l = k >= 0 && e <= rSqr ? k : -1, was = lab[i];
            if (l == was) return;
            lab[i] = (short)l;
            if (was >= 0) tflag[was] = 1;
            if (l >= 0) tflag[l] = 1;
        };
        for (;;) {
            if (tid == 0) *nList = 0;
            for (int i = tid; i < kMemWaves * ks; i += kMemThreads) wbase[i] = 0;
            __syncthreads();
            // 1. labels: against the moved points, or listed
            const int nM = iter == 0 ? 0 : *nMoved;
            int n = nP;
            if (iter > 0) {
                for (int b = 0; b < nP; b += kMemThreads) {
                    const int i = b + tid;
                    const int k0 = i < nP ? near[i] : -1;
                    const bool full = k0 >= 0 && mflag[k0];
                    const uint64_t m = __ballot(full);
                    int base = 0;
                    if (lane == 0 && m) base = atomicAdd(nList, __popcll(m));
                    base = __shfl(base, 0);
                    if (full) {
                        list[base + __popcll(m & below)] = (unsigned short)i;
                    } else if (i < nP) {
                        T p[DIM];
                        sample(i, p);
                        T best = dist[i];
                        int k = k0;
                        for (int q = 0; q < nM; ++q) {
                            const int c = movedL[q];
                            T s[DIM];
                            chosen(c, s);
                            const T e = exact_sqdist<T, DIM>(p, s);
                            if (e < best || (e == best && c < k)) {
                                best = e;
                                k = c;
                            }
                        }
                        if (k != k0) settle(i, best, k);
                    }
                }
                __syncthreads();
                n = *nList;
            }
            // listed samples (all of them in the first iteration) against every chosen point; a wave
            // takes `per` samples a lane, which share the reads of the chosen points
            auto full_scan = [&](auto perC) {
                constexpr int kPer = decltype(perC)::value;
                for (int b = wave * kPer * kWave; b < n; b += kMemWaves * kPer * kWave) {
                    T p[kPer][DIM], best[kPer];
                    int i[kPer], k[kPer];
#pragma unroll
                    for (int j = 0; j < kPer; ++j) {
                        const int q = b + j * kWave + lane;
                        i[j] = q < n ? (iter == 0 ? q : (int)list[q]) : -1;
                        sample(max(i[j], 0), p[j]);
                        best[j] = FpTraits<T>::big;
                        k[j] = -1;
                    }
#pragma unroll 4
                    for (int c = 0; c < K; ++c) {
                        T s[DIM];
                        chosen(c, s);
#pragma unroll
                        for (int j = 0; j < kPer; ++j) {
                            const T e = exact_sqdist<T, DIM>(p[j], s);
                            const bool closer = e < best[j];
                            best[j] = closer ? e : best[j];
                            k[j] = closer ? c : k[j];
                        }
                    }
#pragma unroll
                    for (int j = 0; j < kPer; ++j)
                        if (i[j] >= 0) settle(i[j], best[j], k[j]);
                }
            };
            // as many samples a lane as leave every SIMD a wave
            if (n > 512 && DIM <= 3) full_scan(std::integral_constant<int, 4>{});
            else if (n > 256 && DIM <= 6) full_scan(std::integral_constant<int, 2>{});
            else full_scan(std::integral_constant<int, 1>{});
            __syncthreads();

            // 2. the touched chains in index order (K <= kMemThreads); tflag: their places
            int nT;
            {
                const bool t = tid < K && tflag[tid];
                const uint64_t m = __ballot(t);
                if (lane == 0) small[wave] = __popcll(m);
                __syncthreads();
                int o = __popcll(m & below);
                nT = 0;
                for (int w = 0; w < kMemWaves; ++w) {
                    o += w < wave ? small[w] : 0;
                    nT += small[w];
                }
                if (tid < K) {
                    tflag[tid] = t ? o + 1 : 0;
                    mflag[tid] = 0;
                }
                if (t) touched[o] = tid;
                if (tid == 0) *nMoved = 0;
            }
            __syncthreads();
            if (nT == 0) {   // every chain has its members, hence its sum: nothing moves
                ++iter;
                break;
            }

            // 3. their members in sample order: stable counting sort of the samples by place
            auto match = [&](int L) {
                const bool v = L >= 0;
                uint64_t m = __ballot(v);
                for (int b = 0; b < bits; ++b) {
                    const bool bit = (L >> b) & 1;
                    const uint64_t bb = __ballot(v && bit);
                    m &= bit ? bb : ~bb;
                }
                return m;
            };
            auto place = [&](int i) { return lab[i] >= 0 ? tflag[lab[i]] - 1 : -1; };
            const int range = ((nP + kMemWaves - 1) / kMemWaves + kWave - 1) / kWave * kWave;
            const int r0 = min(nP, wave * range), r1 = min(nP, r0 + range);
            for (int q0 = r0; q0 < r1; q0 += kWave) {
                const int i = q0 + lane;
                const int L = i < r1 ? place(i) : -1;
                const uint64_t m = match(L);
                if (L >= 0 && (m & below) == 0) wbase[wave * ks + L] += __popcll(m);
            }
            __syncthreads();
            {
                int tot = 0;
                if (tid < nT)
                    for (int w = 0; w < kMemWaves; ++w) tot += wbase[w * ks + tid];
                int incl = tot;
#pragma unroll
                for (int o = 1; o < kWave; o <<= 1) {
                    const int y = __shfl_up(incl, o);
                    if (lane >= o) incl += y;
                }
                if (lane == kWave - 1) small[wave] = incl;
                __syncthreads();
                int o = incl - tot;
                for (int w = 0; w < wave; ++w) o += small[w];
                if (tid < nT) {
                    cnt[tid] = tot;
                    off[tid] = o;
                    for (int w = 0; w < kMemWaves; ++w) {
                        const int c = wbase[w * ks + tid];
                        wbase[w * ks + tid] = o;
                        o += c;
                    }
                }
            }
            __syncthreads();
            for (int q0 = r0; q0 < r1; q0 += kWave) {
                const int i = q0 + lane;
                const int L = i < r1 ? place(i) : -1;
                const uint64_t m = match(L);
                // within a wave LDS operations complete in issue order: every lane reads its
                // place's base before the leader advances it
                if (L >= 0) order[wbase[wave * ks + L] + __popcll(m & below)] = (unsigned short)i;
                if (L >= 0 && (m & below) == 0) wbase[wave * ks + L] += __popcll(m);
            }
            __syncthreads();

            // 4. their sums, rows of 16 lanes over (coordinate, place)
            for (int rb = 0; rb < DIM * nT; rb += kMemThreads / 16) {
                const int row = rb + tid / 16;
                const bool act = row < DIM * nT;
                const int d = act ? row / nT : 0, t = act ? row - d * nT : 0;
                const int c = act ? cnt[t] : 0, o = act ? off[t] : 0;
                const T* xd = x + d * pc;
                const T v = row_ordered_sum<T, 2>(wave_row_max(c), [&](int i) {
                    const T y = xd[c > 0 ? (int)order[o + min(i, c - 1)] : 0];
                    return i < c ? y : T(0);
                });
                if (act && (tid & 15) == 0) sum[d * ks + t] = v;
            }
            __syncthreads();

            // 5. shift toward their mass centres
            if (tid < nT) {
                const int k = touched[tid], c = cnt[tid];
                tflag[k] = 0;
                bool moved = false;
                if (c > 0) {
                    const T fc = (T)c;
#pragma unroll
                    for (int d = 0; d < DIM; ++d) {
                        const T mc = sum[d * ks + tid] / fc;
                        T thr = T(2) * fabs(mc);
                        thr = thr * fc;
                        thr = thr * FpTraits<T>::eps;
                        T& s = sS[k * kSt + d];
                        if (fabs(mc - s) > thr) {
                            s = mc;
                            moved = true;
                        }
                    }
                }
                if (moved) {
                    mflag[k] = 1;
                    movedL[atomicAdd(nMoved, 1)] = k;
                }
            }
            __syncthreads();
            ++iter;
            if (*nMoved == 0 || (a.maxIter > 0 && iter >= a.maxIter)) break;
            if (iter >= a.guard) {
                if (tid == 0) *a.error = 1;
                break;
            }
        }
    } else {
        iter = 1;   // the reference loop runs one pass that moves nothing
    }
    for (int i = tid; i < DIM * K; i += kMemThreads) a.S[(i / K) * a.sStride + sd.sOff + i % K] = sS[(i % K) * kSt + i / K];
    if (tid == 0) {
        a.segIter[seg] = iter;
        atomicMax(a.maxIters, iter);
    }
}

// One evolve iteration of every segment with its labels taken from the batch-wide scan
// (global chosen slots, or -1): the counting sort and the ordered sums of the local kernel
// in one workgroup per segment, then the shift straight on the chosen points in HBM and the
// segment's moved flag.  Replaces the batch-wide sort, member gather and sums for batches
// of small segments.
template <typename T, int DIM>
__global__ __launch_bounds__(kLocalThreads) void segment_sums_kernel(LocalArgs<T> a) {
    if (*a.allDone) return;
    const int seg = blockIdx.x;
    if (a.segDone[seg]) return;
    extern __shared__ __align__(16) char smem[];
    const int ks = a.kStride;
    const LocalLds<T> Ld = local_lds<T, DIM>(smem, ks, a.pCap);
    const SegDesc sd = a.segs[seg];
    const int K = a.segK[seg];
    const int nP = sd.nP;
    if (K <= 0 || nP <= 0) return;   // no member: nothing moves
    const int tid = threadIdx.x;
    const int chunk = a.pCap;
    const int bits = K > 1 ? 32 - __clz(K - 1) : 1;
    for (int i = tid; i < DIM * K; i += kLocalThreads) Ld.run[(i / K) * ks + i % K] = T(0);
    for (int i = tid; i < K; i += kLocalThreads) Ld.cntT[i] = 0;
    for (int c0 = 0; c0 < nP; c0 += chunk) {
        const int cn = min(chunk, nP - c0);
        for (int i = tid; i < cn; i += kLocalThreads) {
            const int g = a.labelsIn[sd.pOff + c0 + i];
            Ld.lab[i] = (short)(g < 0 ? -1 : (int)(g - sd.sOff));
        }
        for (int i = tid; i < kLocalWaves * K; i += kLocalThreads) Ld.wbase[(i / K) * ks + i % K] = 0;
        __syncthreads();
        sort_and_fold_chunk<T, DIM>(a, Ld, sd, K, c0, cn, bits);
    }
    bool movedAny = false;
    for (int i = tid; i < DIM * K; i += kLocalThreads) {
        const int d = i / K, k = i - d * K;
        const int c = Ld.cntT[k];
        if (c == 0) continue;
        const T fc = (T)c;
        const T mc = Ld.run[d * ks + k] / fc;
        T thr = T(2) * fabs(mc);
        thr = thr * fc;
        thr = thr * FpTraits<T>::eps;
        T& s = a.S[d * a.sStride + sd.sOff + k];
        if (fabs(mc - s) > thr) {
            s = mc;
            movedAny = true;
        }
    }
    if (movedAny) a.segMoved[seg] = 1;
}

template <typename T, int DIM>
hipError_t launch_segment_dim(const LocalArgs<T>& a, int numSegs, hipStream_t st) {
    const size_t bytes = lds_bytes(DIM, sizeof(T), a.kStride, a.pCap);
    static bool attrSet = false;
    if (!attrSet) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&segment_sums_kernel<T, DIM>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLocalLdsBudget);
        if (e != hipSuccess) return e;
        attrSet = true;
    }
    hipLaunchKernelGGL((segment_sums_kernel<T, DIM>), dim3(numSegs), dim3(kLocalThreads), bytes, st, a);
    return hipGetLastError();
}

template <typename T, int DIM>
hipError_t launch_mem_dim(const LocalArgs<T>& a, hipStream_t st) {
    static bool attrSet = false;
    if (!attrSet) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&local_mem_kernel<T, DIM>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLocalLdsBudget);
        if (e != hipSuccess) return e;
        attrSet = true;
    }
    hipLaunchKernelGGL((local_mem_kernel<T, DIM>), dim3(a.count), dim3(kMemThreads),
                       mem_lds_bytes(DIM, sizeof(T), a.kStride, a.pCap), st, a);
    return hipGetLastError();
}

template <typename T, int DIM>
hipError_t launch_dim(const LocalArgs<T>& a, hipStream_t st) {
    constexpr int PPT = DIM <= 4 ? 2 : 1;
    const size_t bytes = lds_bytes(DIM, sizeof(T), a.kStride, a.pCap);
    static bool attrSet = false;
    if (!attrSet) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&local_evolve_kernel<T, DIM, PPT>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLocalLdsBudget);
        if (e != hipSuccess) return e;
        attrSet = true;
    }
    hipLaunchKernelGGL((local_evolve_kernel<T, DIM, PPT>), dim3(a.count), dim3(kLocalThreads), bytes, st, a);
    return hipGetLastError();
}

}  // namespace

size_t local_lds_bytes(int dim, size_t valueBytes, int kStride, int pCap) {
    return lds_bytes(dim, valueBytes, kStride, pCap);
}

bool local_fits_lds(int dim, size_t valueBytes, int kStride, int maxP) {
    return kStride <= kMemThreads && maxP <= kLocalChunk &&
           mem_lds_bytes(dim, valueBytes, kStride, maxP) <= kLocalLdsBudget;
}

template <typename T>
hipError_t launch_local_evolve(const LocalArgs<T>& a, int dim, hipStream_t st) {
    if (a.count <= 0) return hipSuccess;
    if (local_lds_bytes(dim, sizeof(T), a.kStride, a.pCap) > kLocalLdsBudget || a.pCap > kLocalChunk ||
        a.kStride > kLocalMaxK + kChosenTile)
        return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    if (a.samplesInLds) {
        if (mem_lds_bytes(dim, sizeof(T), a.kStride, a.pCap) > kLocalLdsBudget || a.kStride > kMemThreads)
            return hipErrorInvalidValue;
        RD_DISPATCH_DIM(dim, { e = launch_mem_dim<T, DIM>(a, st); });
        return e;
    }
    RD_DISPATCH_DIM(dim, { e = launch_dim<T, DIM>(a, st); });
    return e;
}

template <typename T>
hipError_t launch_segment_sums(const LocalArgs<T>& a, int dim, int numSegs, hipStream_t st) {
    if (numSegs <= 0) return hipSuccess;
    if (local_lds_bytes(dim, sizeof(T), a.kStride, a.pCap) > kLocalLdsBudget || a.pCap > kLocalChunk ||
        a.kStride > kLocalMaxK + kChosenTile)
        return hipErrorInvalidValue;
    hipError_t e = hipErrorInvalidValue;
    RD_DISPATCH_DIM(dim, { e = launch_segment_dim<T, DIM>(a, numSegs, st); });
    return e;
}

template hipError_t launch_segment_sums<float>(const LocalArgs<float>&, int, int, hipStream_t);
template hipError_t launch_segment_sums<double>(const LocalArgs<double>&, int, int, hipStream_t);
template hipError_t launch_local_evolve<float>(const LocalArgs<float>&, int, hipStream_t);
template hipError_t launch_local_evolve<double>(const LocalArgs<double>&, int, hipStream_t);

}  // namespace rdhip
