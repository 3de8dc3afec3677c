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
// a floating-point scan; they differ from the serial ones by less than (values of the tile) / 2 + 40
// units of the largest of them, and G below is more than that.  A lane is clean when every predicted
// running sum from its start to its end is at least G inside one binade and none of its values lies
// between two whole numbers: then the serial running sums are inside that binade too, its unit is
// theirs, and neighbouring clean lanes share it.  The sum then advances from one dirty lane to the
// next by the whole-number steps of the clean lanes between them (a difference of an integer scan),
// and a dirty lane's values are added one by one.  Sums of one sign are dirty where they cross a
// power of two and at about one value in between; where a sum hovers around zero (the coordinate
// mean of a chosen point near an axis) most lanes are dirty, and after two such tiles in a row the
// caller gets the sum so far back and finishes it with four waves (block_speculative_sum).
//
// Bound: latency of one wave's dependent steps.  Cycles per value of a long list, one wave: 1.95
// float and 3.9 double, against 8.75 and 14.2 for additions fed by lane reads and 6.25 and 22.8 for
// additions fed from LDS.
#pragma once

#include "rd_common.hpp"

namespace rdhip {

template <typename T>
struct Binade;
template <>
struct Binade<float> {
    using Bits = unsigned;
    using Int = int;
    static constexpr int mant = 23, expMax = 255, expBias = 127, perLane = 16;
    static constexpr float guard = 1.220703125e-4f;   // 2^-13: 1024 units, a tile has 1024 values
    static __device__ __forceinline__ Bits bits(float v) { return __float_as_uint(v); }
    static __device__ __forceinline__ float value(Bits b) { return __uint_as_float(b); }
    static __device__ __forceinline__ float round(float v) { return __builtin_rintf(v); }
    static __device__ __forceinline__ Bits first_lane(Bits b) { return (Bits)__builtin_amdgcn_readfirstlane((int)b); }
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
    static constexpr int mant = 52, expMax = 2047, expBias = 1023, perLane = 8;
    static constexpr double guard = 9.094947017729282e-13;   // 2^-40
    static __device__ __forceinline__ Bits bits(double v) { return (Bits)__double_as_longlong(v); }
    static __device__ __forceinline__ double value(Bits b) { return __longlong_as_double((long long)b); }
    static __device__ __forceinline__ double round(double v) { return __builtin_rint(v); }
    static __device__ __forceinline__ Bits first_lane(Bits b) {
        const unsigned lo = (unsigned)__builtin_amdgcn_readfirstlane((int)(b & 0xffffffffULL));
        const unsigned hi = (unsigned)__builtin_amdgcn_readfirstlane((int)(b >> 32));
        return ((Bits)hi << 32) | lo;
    }
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

constexpr int kSerialSlack = 16;

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
__device__ __forceinline__ PartialSum<T> wave_serial_sum(const T* __restrict__ src, int cnt, int hoverMin) {
    using B = Binade<T>;
    using Int = typename B::Int;
    using Bits = typename B::Bits;
    constexpr int kPer = B::perLane, kTile = kPer * kWave;
    static_assert(kPer <= kSerialSlack, "a lane's last chunk may start at the list's last value");
    const int lane = lane_id();
    cnt = __builtin_amdgcn_readfirstlane(cnt);
    struct __attribute__((packed, aligned(sizeof(T)))) Chunk {
        T v[kPer];
    };
    // lane l: values kPer l .. kPer l + kPer - 1 of the tile, +0 past the end (adding it changes no
    // sum: a sum that starts at +0 is never -0).  Every tile is loaded the same way, whole, so that
    // the loads of the next one stay in flight while this one is summed.
    const int lastChunk = cnt > 0 ? (cnt - 1) / kPer * kPer : 0;
    auto load = [&](int t0, Chunk& c) {
        c = *reinterpret_cast<const Chunk*>(src + min(t0 + lane * kPer, lastChunk));
    };
    T s = T(0);
    if (cnt <= 0) return {s, 0};
    Chunk nxt;
    load(0, nxt);
    int hover = 0;
    for (int t0 = 0; t0 < cnt; t0 += kTile) {
        T x[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) x[j] = t0 + lane * kPer + j < cnt ? nxt.v[j] : T(0);
        load(t0 + kTile, nxt);
        // predicted running sums: extremes inside the lane, start of the lane, largest of the tile
        T run = T(0), mn = T(0), mx = T(0);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            run = run + x[j];
            mn = fmin(mn, run);
            mx = fmax(mx, run);
        }
        const T upTo = wave_scan<T>(run, T(0), [](T a, T b) { return a + b; });
        const T at = s + (upTo - run);
        const T lo = at + mn, hi = at + mx;
        const T big = fmax(fabs(lo), fabs(hi));
        const T most = B::value(B::first_lane(B::bits(
            read_lane(wave_scan<T>(big, T(0), [](T a, T b) { return fmax(a, b); }), kWave - 1))));
        const T g = B::guard * most;
        // the lane's binade, if it has one (the sums' magnitudes between near and far)
        const T near = fmin(fabs(lo), fabs(hi)) - g, far = big + g;
        const int ex = (int)((B::bits(near) >> B::mant) & (Bits)B::expMax);
        bool clean = lo * hi > T(0) && near > T(0) && (B::bits(near) >> B::mant) == (B::bits(far) >> B::mant) &&
                     ex > B::mant && ex < B::expMax - 1 && fabs(run) < far;   // run: no NaN on the way
        const T inv = B::value((Bits)(2 * B::expBias + B::mant - (clean ? ex : B::expBias)) << B::mant);
        T step = T(0), half = T(0);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const T f = x[j] * inv;
            const T r = B::round(f);
            half = fmax(half, fabs(f - r));
            step = step + r;
        }
        clean = clean && half < T(0.5);
        const Int own = clean ? (Int)step : 0;
        const Int steps = wave_scan<T>(own, Int(0), [](Int a, Int b) { return a + b; });
        const int lanes = min(kWave, (cnt - t0 + kPer - 1) / kPer);
        uint64_t dirty = __ballot(!clean && lane < lanes);
        if (s == T(0) && __ballot(!(big == T(0))) == 0) dirty = 0;   // zeros leave a sum of zero
        if (__popcll(dirty) > kWave / 2) {
            if (++hover >= 2 && cnt - t0 >= hoverMin) return {s, t0};
        } else {
            hover = 0;
        }
        Int before = 0;   // steps taken so far
        int from = 0;     // lanes in s
        for (;;) {
            const int to = dirty ? __builtin_ctzll(dirty) : lanes;
            if (to > from) {
                const Int upto = B::lane(steps, to - 1);
                if (upto != before) {
                    const Bits sb = B::first_lane(B::bits(s));
                    constexpr Bits kMant = ((Bits)1 << B::mant) - 1;
                    const Bits signBit = (Bits)1 << (8 * sizeof(T) - 1);
                    const Int m = (Int)((sb & kMant) | ((Bits)1 << B::mant));
                    // x / U carries the sign of x: a negative sum's magnitude falls by it
                    const Int now = (sb & signBit) ? m - (upto - before) : m + (upto - before);
                    const Bits ue = ((sb & ~signBit) >> B::mant) - B::mant;
                    s = (T)now * B::value((ue << B::mant) | (sb & signBit));
                }
                before = upto;
            }
            if (!dirty) break;
            T v[kPer];
#pragma unroll
            for (int j = 0; j < kPer; ++j) v[j] = read_lane(x[j], to);
#pragma unroll
            for (int j = 0; j < kPer; ++j) s = s + v[j];
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
