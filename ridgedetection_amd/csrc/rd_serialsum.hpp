// rd_serialsum.hpp -- the serial floating-point sum of a list of values, bit for bit, computed by
// a wave in parallel.
//
// While a running sum s stays inside one binade [2^e, 2^(e+1)), it is a whole multiple m U of that
// binade's unit U, and adding x rounds the exact m + x/U to a whole number: m grows by rint(x/U)
// whatever it was, unless x/U lies exactly between two whole numbers (then the even sum is taken,
// which depends on m).  So the steps of a run of values that stays inside a binade are whole
// numbers that can be added in any order.
//
// A tile gives each lane consecutive values.  The running sums at every lane are first predicted by
// a floating-point scan.  Every partial sum on the way is a difference of two running sums, so no
// rounding exceeds a unit of the largest running sum, and the serial ones' half of one: the
// predictions are off by less than 3/2 (values of the tile) + 100 units, and G below is more than
// that.  A half lane adds its values one after the other to its predicted start, and also to the
// number one unit above it, which has the other parity.  When every predicted running sum on the way
// is at least G inside one binade, the serial ones are inside that binade too, and the half lane's
// whole-number steps are those of the start that has the serial sum's parity.  A lane is clean when
// both halves are inside and take the same steps from either start; neighbouring clean lanes share
// their binade.  The sum advances from one dirty lane to the next by the steps of the clean lanes
// between them (a difference of an integer scan); a dirty lane's halves inside a binade are advanced
// by the steps of the right parity, the others' values are added one by one (every lane adds its own
// to the sum so far, and the dirty one's result is taken).  Sums of one sign are dirty where they
// cross a power of two and at about one tie in between; where a sum hovers around zero (the
// coordinate mean of a chosen point near an axis) most lanes are dirty, and after two such tiles in
// a row the caller gets the sum so far back and finishes it with four waves (block_speculative_sum).
//
// Bound: latency of one wave's dependent steps, and of a dirty lane's (about 350 cycles each; the
// first 2,000 values have five to ten).  Cycles per value of a list of 32,768 floats, one wave: 1.14,
// against 8.75 for additions fed by lane reads and 6.25 for additions fed from LDS; 3.2 for one of
// 2,048.  With half the values a tile, lone ties added one by one and a rint of every value: 1.63
// and 3.0, and 420 cycles a dirty lane.
#pragma once

#include "rd_common.hpp"

namespace rdhip {

template <typename T>
struct Binade;
template <>
struct Binade<float> {
    using Bits = unsigned;
    using Int = int;
    static constexpr int mant = 23, expMax = 255, expBias = 127, perHalf = 16;
    static constexpr float guard = 4.8828125e-4f;   // 2^-11: 4096 units, a tile has 2048 values
    static __device__ __forceinline__ Bits bits(float v) { return __float_as_uint(v); }
    static __device__ __forceinline__ float value(Bits b) { return __uint_as_float(b); }
    static __device__ __forceinline__ Int lane(Int v, int l) { return __builtin_amdgcn_readlane(v, l); }
    template <int kCtrl, int kRows>
    static __device__ __forceinline__ Int dpp(Int old, Int v) {   // old where the lane has no source
        return __builtin_amdgcn_update_dpp(old, v, kCtrl, kRows, 0xf, false);
    }
    template <int kCtrl, int kRows>
    static __device__ __forceinline__ float dpp(float old, float v) {
        return __int_as_float(dpp<kCtrl, kRows>(__float_as_int(old), __float_as_int(v)));
    }
};
template <>
struct Binade<double> {
    using Bits = unsigned long long;
    using Int = long long;
    static constexpr int mant = 52, expMax = 2047, expBias = 1023, perHalf = 8;
    static constexpr double guard = 9.094947017729282e-13;   // 2^-40: 4096 units, a tile has 1024 values
    static __device__ __forceinline__ Bits bits(double v) { return (Bits)__double_as_longlong(v); }
    static __device__ __forceinline__ double value(Bits b) { return __longlong_as_double((long long)b); }
    static __device__ __forceinline__ Int lane(Int v, int l) { return (Int)read_lane((uint64_t)v, l); }
    template <int kCtrl, int kRows>
    static __device__ __forceinline__ Int dpp(Int old, Int v) {
        const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp((int)(old & 0xffffffffLL), (int)(v & 0xffffffffLL),
                                                                  kCtrl, kRows, 0xf, false);
        const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp((int)(old >> 32), (int)(v >> 32), kCtrl, kRows, 0xf,
                                                                  false);
        return (Int)(((Bits)hi << 32) | lo);
    }
    template <int kCtrl, int kRows>
    static __device__ __forceinline__ double dpp(double old, double v) {
        return __longlong_as_double(dpp<kCtrl, kRows>((Int)__double_as_longlong(old), (Int)__double_as_longlong(v)));
    }
};

// Inclusive scan of the wave's lanes by `op` with identity `id` (lane 63: the reduction).
template <typename T, typename V, typename Op>
__device__ __forceinline__ V wave_scan(V v, V id, Op op) {
    using B = Binade<T>;
    v = op(v, B::template dpp<0x111, 0xf>(id, v));   // row_shr:1
    v = op(v, B::template dpp<0x112, 0xf>(id, v));   // row_shr:2
    v = op(v, B::template dpp<0x114, 0xf>(id, v));   // row_shr:4
    v = op(v, B::template dpp<0x118, 0xf>(id, v));   // row_shr:8
    v = op(v, B::template dpp<0x142, 0xa>(id, v));   // row_bcast:15 into rows 1 and 3
    v = op(v, B::template dpp<0x143, 0xc>(id, v));   // row_bcast:31 into rows 2 and 3
    return v;
}

// a 16-byte read
template <typename T>
struct WideOf;
template <>
struct WideOf<float> { using type = float4; static constexpr int n = 4; };
template <>
struct WideOf<double> { using type = double2; static constexpr int n = 2; };

// orders a wave's LDS accesses to a part of its own
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

constexpr int kSerialSlack = 4;

// LDS values wave_serial_sum takes: the values of half the wave's lanes, 16 bytes apart
template <typename T>
constexpr int serial_lds_elems() {
    return kWave / 2 * (2 * Binade<T>::perHalf + 16 / (int)sizeof(T));
}

// A running sum: `sum` holds the values before `done`.
template <typename T>
struct PartialSum {
    T sum;
    int done;
};

// +0 + src[0] + src[1] + ... + src[cnt - 1] added in that order, by a whole wave (cnt and src the
// same for every lane; every lane returns the sum).  Up to kSerialSlack values past the list are
// read (not used).  A sum that hovers is handed back unfinished while at least `hoverMin` values
// are left.
template <typename T>
__device__ __forceinline__ PartialSum<T> wave_serial_sum(const T* __restrict__ src, int cnt, int hoverMin, T* lds) {
    using B = Binade<T>;
    using Int = typename B::Int;
    using Bits = typename B::Bits;
    constexpr int kHalf = B::perHalf, kPer = 2 * kHalf, kTile = kPer * kWave;
    constexpr int kVec = 16 / sizeof(T), kLoads = kPer / kVec;
    static_assert(kVec <= kSerialSlack && kPer * sizeof(T) == 128, "a lane's values are one line");
    const int lane = lane_id();
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    struct __attribute__((packed, aligned(sizeof(T)))) Vec {
        T v[kVec];
    };
    // Loads are coalesced, 16 bytes a lane, and go through LDS to the lane that sums them, the first
    // half of the lanes' values and then the second's.  Every tile is loaded the same way, whole, so
    // that the loads of the next one stay in flight while this one is summed.
    const int lastVec = cnt > 0 ? (cnt - 1) / kVec * kVec : 0;
    T* const put = lds + (lane / kLoads) * (kPer + kVec) + lane % kLoads * kVec;
    const T* const get = lds + lane % (kWave / 2) * (kPer + kVec);
    auto load = [&](int t0, Vec* c) {
#pragma unroll
        for (int k = 0; k < kLoads; ++k)
            c[k] = *reinterpret_cast<const Vec*>(src + min(t0 + (k * kWave + lane) * kVec, lastVec));
    };
    T s = T(0);
    if (cnt <= 0) return {s, 0};
    constexpr Bits kExp = (Bits)B::expMax << B::mant;
    auto unit_of = [](T v) { return B::value((B::bits(v) & kExp) - ((Bits)B::mant << B::mant)); };
    Vec nxt[kLoads];
    load(0, nxt);
    int hover = 0;
    for (int t0 = 0; t0 < cnt; t0 += kTile) {
        // lane l: values kPer l .. kPer l + kPer - 1 of the tile, +0 past the end (adding it changes no
        // sum: a sum that starts at +0 is never -0)
        T x[kPer];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            wave_lds_sync();
#pragma unroll
            for (int k = 0; k < kLoads / 2; ++k)
                *reinterpret_cast<typename WideOf<T>::type*>(put + k * (kWave / kLoads) * (kPer + kVec)) =
                    __builtin_bit_cast(typename WideOf<T>::type, nxt[half * (kLoads / 2) + k]);
            wave_lds_sync();
            if (lane / (kWave / 2) == half) {
#pragma unroll
                for (int k = 0; k < kLoads; ++k) {
                    const Vec v = __builtin_bit_cast(Vec, reinterpret_cast<const typename WideOf<T>::type*>(get)[k]);
#pragma unroll
                    for (int j = 0; j < kVec; ++j) x[k * kVec + j] = v.v[j];
                }
            }
        }
        if (t0 + kTile > cnt) {
#pragma unroll
            for (int j = 0; j < kPer; ++j) x[j] = t0 + lane * kPer + j < cnt ? x[j] : T(0);
        }
        load(t0 + kTile, nxt);
        // the predicted sum at the start of each half of the lane, and the half's running sums from
        // there (their extremes) and from one unit higher
        T run[2] = {x[0], x[kHalf]}, at[2], unit[2], c0[2], c1[2], lo[2], hi[2];
#pragma unroll
        for (int j = 1; j < kHalf; ++j)
            for (int h = 0; h < 2; ++h) run[h] = run[h] + x[h * kHalf + j];
        const T both = run[0] + run[1];
        at[0] = s + (wave_scan<T>(both, T(0), [](T a, T b) { return a + b; }) - both);
        at[1] = at[0] + run[0];
        for (int h = 0; h < 2; ++h) {
            unit[h] = unit_of(at[h]);
            c1[h] = at[h] + unit[h];
            c0[h] = lo[h] = hi[h] = at[h];
        }
#pragma unroll
        for (int j = 0; j < kHalf; ++j)
            for (int h = 0; h < 2; ++h) {
                c0[h] = c0[h] + x[h * kHalf + j];
                c1[h] = c1[h] + x[h * kHalf + j];
                lo[h] = fmin(lo[h], c0[h]);
                hi[h] = fmax(hi[h], c0[h]);
            }
        T big[2];
        for (int h = 0; h < 2; ++h) big[h] = fmax(fabs(lo[h]), fabs(hi[h]));
        const T most = fmax(big[0], big[1]);
        const T g = B::guard * read_lane(wave_scan<T>(most, T(0), [](T a, T b) { return fmax(a, b); }), kWave - 1);
        bool inside[2], clean[2];
        Int up0[2], up1[2];
        for (int h = 0; h < 2; ++h) {
            // the sums' magnitudes between near and far lie in one binade
            const T near = fmin(fabs(lo[h]), fabs(hi[h])) - g, far = big[h] + g;
            const int ex = (int)((B::bits(near) >> B::mant) & (Bits)B::expMax);
            inside[h] = lo[h] * hi[h] > T(0) && near > T(0) && (B::bits(near) >> B::mant) == (B::bits(far) >> B::mant) &&
                        ex > B::mant && ex < B::expMax - 1;
            // units the magnitude grows by, counted by the bits of the one binade
            up0[h] = (Int)(B::bits(c0[h]) - B::bits(at[h]));
            up1[h] = (Int)(B::bits(c1[h]) - B::bits(at[h] + unit[h]));
            clean[h] = inside[h] && up0[h] == up1[h];
        }
        const Int steps = wave_scan<T>(clean[0] && clean[1] ? up0[0] + up0[1] : Int(0), Int(0),
                                       [](Int a, Int b) { return a + b; });
        const int lanes = min(kWave, (cnt - t0 + kPer - 1) / kPer);
        const uint64_t in0 = __ballot(inside[0]), in1 = __ballot(inside[1]);
        uint64_t dirty = __ballot(!(clean[0] && clean[1]) && lane < lanes);
        if (s == T(0) && __ballot(!(most == T(0))) == 0) dirty = 0;   // zeros leave a sum of zero
        if (__popcll(dirty) > kWave / 2) {
            if (++hover >= 2 && cnt - t0 >= hoverMin) return {s, t0};
        } else {
            hover = 0;
        }
        auto advance = [](T from, Int by) { return B::value(B::bits(from) + (Bits)by); };   // in one binade
        Int before = 0;   // steps taken so far
        int from = 0;     // lanes in s
        for (;;) {
            const int to = dirty ? __builtin_ctzll(dirty) : lanes;
            if (to > from) {
                const Int upto = B::lane(steps, to - 1);
                if (upto != before) s = advance(s, upto - before);
                before = upto;
            }
            if (!dirty) break;
            T v = s;   // every lane takes its own values; lane `to` started from the right sum
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (((h ? in1 : in0) >> to) & 1) {
                    // what a tie rounds to follows from the start's parity
                    v = advance(v, (B::bits(v) ^ B::bits(at[h])) & 1 ? up1[h] : up0[h]);
                } else {
#pragma unroll
                    for (int j = 0; j < kHalf; ++j) v = v + x[h * kHalf + j];
                }
            }
            s = read_lane(v, to);
            from = to + 1;
            dirty &= dirty - 1;
        }
    }
    return {s, cnt};
}

// Serial sum start + src[0] + ... + src[cnt - 1] by a whole wave whose lanes may start from
// different values (each lane returns its own sum; a start must not be -0).  cnt is the same for
// every lane.  A lane holds one value in 64 of a tile, and each value reaches all lanes by
// v_readlane, two values ahead of its add: 8.75 cycles a value (the issue of the readlane and the
// add; double 14.2) on each of a CU's four SIMDs at once.
template <typename T>
__device__ __forceinline__ T wave_lane_sums(const T* __restrict__ src, int cnt, T start) {
    constexpr int kPer = 4;                // 256 values a tile: ~2200 cycles of adds hide
    constexpr int kTile = kPer * kWave;    // the loads of the next
    constexpr int kStep = 32;              // values between end tests
    constexpr int kAhead = 2;
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    const int lane = lane_id(), last = max(cnt - 1, 0);
    auto load = [&](int i0, T(&r)[kPer]) {
#pragma unroll
        for (int c = 0; c < kPer; ++c) {
            const int i = i0 + c * kWave + lane;
            const T x = src[min(i, last)];
            r[c] = i < cnt ? x : T(0);
        }
    };
    T sum = start, reg[kPer], nxt[kPer];
    if (cnt <= 0) return sum;
    load(0, reg);
    for (int i0 = 0; i0 < cnt; i0 += kTile) {
        load(i0 + kTile, nxt);
#pragma unroll
        for (int h = 0; h < kTile / kStep; ++h) {
            if (i0 + h * kStep >= cnt) break;
            const T r = reg[h * kStep / kWave];
            T s[kAhead];
#pragma unroll
            for (int j = 0; j < kAhead; ++j) s[j] = read_lane(r, h * kStep % kWave + j);
#pragma unroll
            for (int j = 0; j < kStep; ++j) {
                T x = T(0);
                if (j + kAhead < kStep) x = read_lane(r, h * kStep % kWave + j + kAhead);
                __builtin_amdgcn_sched_barrier(0);
                sum = sum + s[j % kAhead];
                __builtin_amdgcn_sched_barrier(0);
                s[j % kAhead] = x;
            }
        }
#pragma unroll
        for (int c = 0; c < kPer; ++c) reg[c] = nxt[c];
    }
    return sum;
}

// Ordered integer of a value (the order of the values, -0 and +0 both 0) and back (never -0).
__device__ __forceinline__ int64_t ord_of(float x) {
    const int i = __float_as_int(x);
    return i >= 0 ? (int64_t)i : -(int64_t)(i & 0x7fffffff);
}
__device__ __forceinline__ int64_t ord_of(double x) {
    const long long i = __double_as_longlong(x);
    return i >= 0 ? (int64_t)i : -(int64_t)(i & 0x7fffffffffffffffLL);
}
template <typename T>
__device__ __forceinline__ T from_ord(int64_t o);
template <>
__device__ __forceinline__ float from_ord<float>(int64_t o) {
    return __int_as_float(o >= 0 ? (int)o : (int)(0x80000000u | (unsigned)(-o)));
}
template <>
__device__ __forceinline__ double from_ord<double>(int64_t o) {
    return __longlong_as_double(o >= 0 ? (long long)o : (long long)(0x8000000000000000ULL | (unsigned long long)(-o)));
}

// start + src[0] + ... + src[cnt - 1] in that order by a block of kRuns waves (arguments and result
// the same for the whole block): the values are cut into kRuns runs, one per wave, summed at the
// same time.  Wave p cannot know the exact sum its run starts from, so each of its 64 lanes sums
// the run from its own start, the 64 consecutive values of the type centred on the correctly
// rounded sum of everything before the run (from sums in W's wider type).  The runs are then
// walked in order: run p's result is that of the lane whose start equals, bit for bit, the exact
// sum through run p - 1.  When no lane started there (the rounding errors of the serial sum before
// run p exceed 32 units of its last place), every wave sums run p again from it.  The result never
// depends on the estimate; only the time does.
constexpr int kRuns = 4;

template <typename T, typename W>
struct RunLds {
    typename W::Acc wide[kRuns];
    int64_t centre[kRuns];
    T result[kRuns][kWave];
    T start[kRuns][kWave];
};

template <typename T, typename W>
__device__ __forceinline__ T block_speculative_sum(const T* __restrict__ src, int cnt, T start, RunLds<T, W>& sh) {
    using B = Binade<T>;
    const int w = threadIdx.x / kWave, lane = lane_id();
    auto run_start = [&](int p) { return (int)((int64_t)cnt * p / kRuns); };
    const int b0 = run_start(w), n = run_start(w + 1) - b0;
    typename W::Acc acc[4] = {W::zero(), W::zero(), W::zero(), W::zero()};
    constexpr int kAtOnce = 16;
    for (int i0 = 0; i0 < n; i0 += kAtOnce * kWave) {
        T v[kAtOnce];
#pragma unroll
        for (int c = 0; c < kAtOnce; ++c) {
            const int i = i0 + c * kWave + lane;
            v[c] = i < n ? src[b0 + i] : T(0);
        }
#pragma unroll
        for (int c = 0; c < kAtOnce; ++c) acc[c & 3] = W::add(acc[c & 3], v[c]);
    }
    typename W::Acc wide = W::add(W::add(acc[0], acc[1]), W::add(acc[2], acc[3]));
#pragma unroll
    for (int m = kWave / 2; m >= 1; m /= 2) wide = W::add(wide, W::xorShfl(wide, m));
    if (lane == 0) sh.wide[w] = wide;
    __syncthreads();
    T mine = start;
    if (w > 0) {
        typename W::Acc est = W::add(W::zero(), start);
        for (int q = 0; q < w; ++q) est = W::add(est, sh.wide[q]);
        const T e0 = (T)W::value(est);
        const int64_t oe = ord_of(e0);
        mine = isfinite(e0) ? from_ord<T>(oe + lane - kWave / 2) : T(0);
        if (lane == 0) sh.centre[w] = oe;
    }
    sh.result[w][lane] = wave_lane_sums(src + (n > 0 ? b0 : 0), n, mine);
    sh.start[w][lane] = mine;
    __syncthreads();
    T x = sh.result[0][0];
    for (int p = 1; p < kRuns; ++p) {
        const int64_t o = ord_of(x) - sh.centre[p] + kWave / 2;
        if (o >= 0 && o < kWave && B::bits(sh.start[p][o]) == B::bits(x))
            x = sh.result[p][o];
        else
            x = wave_lane_sums(src + run_start(p), run_start(p + 1) - run_start(p), x);
    }
    __syncthreads();   // sh may be used again
    return x;
}

}  // namespace rdhip
