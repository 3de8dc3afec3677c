// rd_noalloc.hip -- rdhip_choose_noalloc: the greedy choose of rdhip_choose on caller-owned
// device buffers, for callers that cannot allocate device memory (code under HIP graph
// capture, serving loops, harnesses that forbid hipMalloc).
//
// The choose kernels (rd_choose.hip) need, beyond the points (input) and the chosen points,
// indices and count (outputs), a few device words (the segment description, its radius, the
// running count and cursor, an overflow flag) and one "open" bit per sample.  Here they live in
// `scratch`, a fixed device array of this library, instead of
// buffers a context allocates.  Every call on a device shares that device's copy of the array:
// calls that overlap on one device (different streams, or threads) race and must be ordered by
// the caller.  A call rewrites all of the array it reads before reading it, so nothing is
// carried over from an earlier call.  The entry point only launches kernels (no allocation,
// copy or synchronisation), so it may also be captured into a graph.
#include "../../include/rdhip.h"
#include "rd_choose.hpp"

#include <algorithm>
#include <mutex>
#include <string>

namespace rdhip {
namespace {

constexpr int64_t kOpenOff = 4096;   // after the header, one bit per sample
constexpr int64_t kScratchBytes = kOpenOff + RDHIP_NOALLOC_MAX_POINTS / 8;

__device__ __align__(256) unsigned char scratch[kScratchBytes];

struct Header {
    SegDesc seg;
    int segK;
    int overflow;
    int largeSeg;       // 0: the one segment
    int largeBlock[2];  // its filter blocks
    int base;
    int cursor;
    int doneCount;
    double rSqr;   // read through segRSqr as the value type (float in the first 4 bytes)
};
static_assert(sizeof(Header) <= kOpenOff, "header layout");

template <typename T>
__global__ void noalloc_setup_kernel(unsigned char* base, int n, T rSqr) {
    if (threadIdx.x != 0) return;
    Header* h = reinterpret_cast<Header*>(base);
    SegDesc s{};
    s.pOff = 0;
    s.nP = n;
    s.nOwn = n;
    s.sOff = 0;
    s.sCap = n;   // the kernels write slots [0, sCap) only
    s.group = 0;
    h->seg = s;
    h->segK = 0;
    h->overflow = 0;
    h->largeSeg = 0;
    h->largeBlock[0] = 0;
    h->largeBlock[1] = (n + kChooseBlock - 1) / kChooseBlock;
    h->base = 0;
    h->cursor = 0;
    h->doneCount = 0;
    *reinterpret_cast<T*>(&h->rSqr) = rSqr;
}

__global__ void noalloc_finish_kernel(const unsigned char* base, int32_t* count) {
    if (threadIdx.x == 0) *count = reinterpret_cast<const Header*>(base)->segK;
}

// hipGetSymbolAddress once per device, with that device current.
constexpr int kMaxDevices = 64;
std::mutex g_mu;
unsigned char* g_scratch[kMaxDevices] = {};

hipError_t scratch_for_current_device(unsigned char** out) {
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_mu);
    if (!g_scratch[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch[dev] = static_cast<unsigned char*>(p);
    }
    *out = g_scratch[dev];
    return hipSuccess;
}

template <typename T>
hipError_t choose_noalloc(int dim, const T* points, int64_t n, int64_t stride, T r, T* chosen, int64_t chosenStride,
                          int32_t* indices, int32_t* count, hipStream_t st) {
    unsigned char* base = nullptr;
    hipError_t e = scratch_for_current_device(&base);
    if (e != hipSuccess) return e;
    Header* h = reinterpret_cast<Header*>(base);
    constexpr int kOneBlock = 4096;   // up to here one block takes the whole cloud (as Engine::choose)
    const int nn = (int)n;
    hipLaunchKernelGGL((noalloc_setup_kernel<T>), dim3(1), dim3(64), 0, st, base, nn, r * r);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    const ChooseArgs<T> a{points, stride, nullptr, chosen, chosenStride, &h->seg, 1, &h->segK,
                          reinterpret_cast<const T*>(&h->rSqr), indices, &h->overflow, nullptr, 1, &h->largeSeg,
                          h->largeBlock, reinterpret_cast<uint64_t*>(base + kOpenOff), &h->base, &h->cursor,
                          &h->doneCount};
    if (nn <= kOneBlock) {
        if ((e = launch_choose_small<T>(a, dim, st)) != hipSuccess) return e;
    } else {
        // the number of rounds depends on the data and cannot be read back here: a fixed list of
        // chunks instead, each filtered against every chosen point before it, then decided by one
        // block however many batches that takes
        for (int c = 0; choose_chunk_start(c) < nn; ++c) {
            const int c0 = choose_chunk_start(c), c1 = std::min(choose_chunk_start(c + 1), nn);
            const int blocks = (c1 - c0 + kChooseBlock - 1) / kChooseBlock;
            if ((e = launch_choose_filter<T>(a, dim, c0 / kChooseBlock, blocks, true, st)) != hipSuccess) return e;
            if ((e = launch_choose_resolve<T>(a, dim, c1, 0, st)) != hipSuccess) return e;
        }
    }
    hipLaunchKernelGGL(noalloc_finish_kernel, dim3(1), dim3(64), 0, st, base, count);
    return hipGetLastError();
}

int fail(int code, const char* msg) {
    set_last_error(msg);
    return code;
}

}  // namespace
}  // namespace rdhip

extern "C" int rdhip_choose_noalloc(int dtype, int dim, const void* points, int64_t n, int64_t stride, double r,
                                    void* chosen, int64_t chosen_stride, int32_t* indices, int32_t* count,
                                    void* hip_stream) {
    using namespace rdhip;
    if (dtype != RDHIP_F32 && dtype != RDHIP_F64) return fail(RDHIP_ERR_INVALID, "dtype must be RDHIP_F32 or RDHIP_F64");
    if (dim < 1 || dim > kMaxDim) return fail(RDHIP_ERR_INVALID, "dimension must be in [1, 12]");
    if (n < 1 || n > RDHIP_NOALLOC_MAX_POINTS)
        return fail(RDHIP_ERR_INVALID, "rdhip_choose_noalloc: n must be in [1, RDHIP_NOALLOC_MAX_POINTS = 2^24]");
    if (!points || !chosen || !indices || !count) return fail(RDHIP_ERR_INVALID, "null device buffer");
    if (stride != 0 && stride < n) return fail(RDHIP_ERR_INVALID, "point stride smaller than the point count");
    if (chosen_stride != 0 && chosen_stride < n) return fail(RDHIP_ERR_INVALID, "chosen stride smaller than the point count");
    if (!(r >= 0)) return fail(RDHIP_ERR_INVALID, "radius must be non-negative");
    const int64_t ps = stride ? stride : n, cs = chosen_stride ? chosen_stride : n;
    hipStream_t st = static_cast<hipStream_t>(hip_stream);
    const hipError_t e =
        dtype == RDHIP_F32
            ? choose_noalloc<float>(dim, static_cast<const float*>(points), n, ps, (float)r, static_cast<float*>(chosen),
                                    cs, indices, count, st)
            : choose_noalloc<double>(dim, static_cast<const double*>(points), n, ps, r, static_cast<double*>(chosen), cs,
                                     indices, count, st);
    if (e != hipSuccess) {
        set_last_error((std::string("rdhip_choose_noalloc: ") + hipGetErrorString(e)).c_str());
        return RDHIP_ERR_HIP;
    }
    return RDHIP_OK;
}
