// sgemm_launch_noalloc: sgemm_launch for callers that cannot allocate device
// memory (code under HIP graph capture, serving loops, harnesses that forbid
// hipMalloc).  A split-K or stream-K launch needs a workspace -- partial tiles
// and their tickets -- which sgemm_launch allocates on the handle's first
// launch that needs it; here it lives in a fixed device array, `scratch`,
// compiled into this library, one copy per device, held until the process
// ends.  Nothing on this path calls hipMalloc, hipFree or any allocating
// routine.
//
// Host code never uses the array's name as a device address: the address of
// each device's copy is looked up once, with that device current, through
// hipGetSymbolAddress, and that pointer is what the kernels receive.  The
// lookup runs in sgemm_open (noalloc_prepare) for the handle's device, so a
// launch -- even the first one on a device, even under graph capture -- only
// reads the stored pointer.

#include "bf16x6_plan.hpp"
#include "noalloc_slots.hpp"
#include "sgemm_internal.hpp"

#include <hip/hip_runtime.h>

#include <cstdio>
#include <functional>
#include <mutex>
#include <thread>

static_assert(bf16x6::kMaxPartialBytes <= SGEMM_NOALLOC_PARTIAL_BYTES && bf16x6::kMaxTickets <= SGEMM_NOALLOC_MAX_TILES,
              "every split-BF16 plan fits the static scratch");

namespace {

constexpr size_t kTicketBytes = (size_t)SGEMM_NOALLOC_MAX_TILES * 4u;
constexpr size_t kScratchBytes = (size_t)SGEMM_NOALLOC_PARTIAL_BYTES + kTicketBytes;

// Split-K partials (the first SGEMM_NOALLOC_PARTIAL_BYTES bytes), then the
// tickets.  Every call on a device shares that device's copy and leaves its
// partials behind and its tickets zero.
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

// Zeroes the tickets of one launch (a kernel rather than a memset, so that a
// caller may capture the call in a HIP graph).
__global__ void __launch_bounds__(256) clear_tickets(uint32_t* __restrict__ t, uint32_t count) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < count) t[i] = 0u;
}

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
void* g_scratch[kMaxDevices];  // device address of each device's `scratch`, null until looked up

// Who uses each device's scratch: noalloc_slots.hpp.  A slot holds an eighth of
// the partials and tickets, so calls of up to eight streams run side by side;
// every launch leaves its tickets zero and a slot's launches are ordered by
// its stream, so a call on the slot its stream owns needs no clearing kernel of
// its own (333 x 129 x 517 in 4 K ranges: 7.7 -> 4.9 us; one slot for all with a
// wait between streams took 18.6 us where three streams took turns).
// Captured calls, whose replays are not seen here, clear their tickets, and
// so does every call on a device once one has been captured.
constexpr size_t kSlotBytes = (size_t)SGEMM_NOALLOC_PARTIAL_BYTES / noalloc::kSlots;
constexpr size_t kSlotTickets = (size_t)SGEMM_NOALLOC_MAX_TILES / noalloc::kSlots;

// The runtime that noalloc::Slots speaks to, on one device.
struct HipStreams {
    typedef hipStream_t Stream;
    hipEvent_t moment = nullptr;                 // recorded and waited for within one order()
    hipEvent_t marks[noalloc::kSlots] = {};

    bool capturing(hipStream_t s, uint64_t* id) {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        unsigned long long n = 0;
        // an error: the null stream while another one captures
        const bool on = hipStreamGetCaptureInfo(s, &cs, &n) != hipSuccess || cs != hipStreamCaptureStatusNone;
        *id = n;
        return on;
    }
    bool per_thread(hipStream_t s) { return s == hipStreamPerThread; }
    uint64_t thread() { return std::hash<std::thread::id>()(std::this_thread::get_id()) | 1u; }
    int order(hipStream_t before, hipStream_t after) {
        hipError_t e = hipEventRecord(moment, before);
        if (e != hipSuccess) return (int)e;
        uint64_t x = 0, y = 0;
        if (capturing(before, &x) && !(capturing(after, &y) && x == y)) return noalloc::kBusy;
        return (int)hipStreamWaitEvent(after, moment, 0);
    }
    int mark(int slot, hipStream_t s) { return (int)hipEventRecord(marks[slot], s); }
    int wait(int slot, hipStream_t s) { return (int)hipStreamWaitEvent(s, marks[slot], 0); }
    int sync(hipStream_t s) { return (int)hipStreamSynchronize(s); }
    hipError_t create() {
        hipError_t e = moment ? hipSuccess : hipEventCreateWithFlags(&moment, hipEventDisableTiming);
        for (hipEvent_t& m : marks)
            if (e == hipSuccess && !m) e = hipEventCreateWithFlags(&m, hipEventDisableTiming);
        return e;
    }
};

struct Use {
    noalloc::Slots<HipStreams> slots;
    HipStreams streams;
    bool captured = false;
};
std::mutex g_use_mutex;
Use g_use[kMaxDevices];

// Address of `scratch` on device `dev`, looked up once per device with that
// device current (the calling thread's current device is restored).
int scratch_address(int dev, void** out) {
    if (dev < 0 || dev >= kMaxDevices) return sgemm_internal::set_error(SGEMM_E_INVALID, "device id out of range");
    std::lock_guard<std::mutex> lock(g_mutex);
    if (!g_scratch[dev]) {
        int cur = 0;
        hipError_t e = hipGetDevice(&cur);
        if (e == hipSuccess && cur != dev) e = hipSetDevice(dev);
        void* p = nullptr;
        if (e == hipSuccess) e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e == hipSuccess) e = g_use[dev].streams.create();
        if (cur != dev) (void)hipSetDevice(cur);
        if (e != hipSuccess || !p) {
            char msg[256];
            snprintf(msg, sizeof(msg), "preparing the static scratch on device %d failed: %s (%d)", dev,
                     hipGetErrorString(e), (int)e);
            return sgemm_internal::set_error(e != hipSuccess ? (int)e : SGEMM_E_NO_DEVICE, msg);
        }
        g_scratch[dev] = p;
    }
    *out = g_scratch[dev];
    return SGEMM_OK;
}

int launch_failed(hipError_t e, const char* what) {
    char msg[256];
    snprintf(msg, sizeof(msg), "%s failed: %s (%d)", what, hipGetErrorString(e), (int)e);
    return sgemm_internal::set_error((int)e, msg);
}

// One call's part of a device's scratch.
struct Scratch {
    float* partials = nullptr;
    uint32_t* tickets = nullptr;
    bool all = false;
    int first = 0;
};

// Partials (`bytes`) and tickets (`count`, zero) on h's device for the launch
// that the caller enqueues on `s` next, with `lock` still held, before it calls
// give_scratch.  noalloc::kBusy: none now.
int take_scratch(const sgemm_handle* h, size_t bytes, size_t count, hipStream_t s, std::unique_lock<std::mutex>& lock,
                 Scratch* out) {
    const int dev = sgemm_internal::device(h);
    void* base = nullptr;
    const int r = scratch_address(dev, &base);
    if (r != SGEMM_OK) return r;
    if (!lock.owns_lock()) lock.lock();
    Use& u = g_use[dev];
    out->all = bytes > kSlotBytes || count > kSlotTickets;
    bool fresh = false, captured = false;
    int e = u.slots.take(u.streams, s, out->all, &out->first, &fresh, &captured);
    u.captured = u.captured || captured;
    if (e == noalloc::kBusy) return e;
    if (e) return launch_failed((hipError_t)e, "ordering two streams' calls");
    unsigned char* const bytes0 = static_cast<unsigned char*>(base);
    out->partials = reinterpret_cast<float*>(bytes0 + (size_t)out->first * kSlotBytes);
    out->tickets = reinterpret_cast<uint32_t*>(bytes0 + SGEMM_NOALLOC_PARTIAL_BYTES) + (size_t)out->first * kSlotTickets;
    if (!fresh && !u.captured) return SGEMM_OK;
    uint32_t n = (uint32_t)count;
    void* args[] = {&out->tickets, &n};
    e = (int)hipLaunchKernel(reinterpret_cast<const void*>(&clear_tickets), dim3((n + 255) / 256), dim3(256), args, 0, s);
    return e == 0 ? SGEMM_OK : launch_failed((hipError_t)e, "clear_tickets launch");
}

// After the launch that take_scratch was called for (its result `r`).
int give_scratch(const sgemm_handle* h, hipStream_t s, const Scratch& t, int r) {
    Use& u = g_use[sgemm_internal::device(h)];
    const int e = u.slots.done(u.streams, s, t.all, t.first);
    return r != SGEMM_OK || !e ? r : launch_failed((hipError_t)e, "ordering two streams' calls");
}

}  // namespace

int sgemm_internal::noalloc_prepare(int dev) {
    void* p = nullptr;
    return scratch_address(dev, &p);
}

void sgemm_internal::noalloc_forget(int dev, hipStream_t stream) {
    if (dev < 0 || dev >= kMaxDevices) return;
    std::lock_guard<std::mutex> lock(g_use_mutex);
    (void)g_use[dev].slots.forget(g_use[dev].streams, stream);
}

extern "C" int sgemm_launch_noalloc(sgemm_handle* h, const float* dA, const float* dB, const float* dC, float* dD,
                                    uint32_t m, uint32_t n, uint32_t k, uint32_t lda, uint32_t ldb, uint32_t ldc,
                                    uint32_t ldd, float alpha, float beta) {
    if (!h) return sgemm_internal::set_error(SGEMM_E_INVALID, "sgemm_launch_noalloc: null handle");
    int r = sgemm_internal::check_launch(h, dA, dB, dC, dD, m, n, k, lda, ldb, ldc, ldd, beta);
    if (r != SGEMM_OK || m == 0 || n == 0) return r;
    hipStream_t s = sgemm_internal::stream(h);
    const thin::Shape ts = sgemm_internal::thin_shape(h, m, n, k, lda, ldb);
    if (ts.on)
        return sgemm_internal::thin_launch(ts, sgemm_internal::trans_a(h), sgemm_internal::trans_b(h), dA, dB, dC, dD, m,
                                           n, k, lda, ldb, ldc, ldd, alpha, beta, s);
    sgemm_internal::Part parts[3];
    // the split-BF16 plan never needs more than the scratch
    sgemm_internal::SplitPlan sp = sgemm_internal::split_plan(h, m, n, k, lda, ldb, ldc, ldd, alpha, beta);
    int count = sp.tile >= 0 ? sgemm_internal::split_strips(h, sp, m, n, lda, ldb, ldc, ldd, parts)
                             : sgemm_internal::decompose(h, m, n, k, lda, ldb, ldc, ldd, parts);
    // every part's needs are checked before anything is launched
    for (int q = 0; q < count; ++q) {
        const sgemm_internal::Part& pt = parts[q];
        if (pt.kh != h && (r = sgemm_check_shape(pt.kh, pt.m, pt.n, k, lda, ldb, ldc, ldd)) != SGEMM_OK) return r;
        const sgemm_internal::Plan p = sgemm_internal::plan(pt.kh, pt.m, pt.n, k);
        if (p.partial_bytes > (size_t)SGEMM_NOALLOC_PARTIAL_BYTES || p.ticket_count > (size_t)SGEMM_NOALLOC_MAX_TILES) {
            char msg[256];
            snprintf(msg, sizeof(msg),
                     "sgemm_launch_noalloc: a %ux%ux%u launch (%u K ranges, %u stream-K tiles) needs %zu bytes of "
                     "partials and %zu tickets; the static scratch holds %u bytes and %u tickets", pt.m, pt.n, k,
                     p.splits, p.sk_tiles, p.partial_bytes, p.ticket_count, (unsigned)SGEMM_NOALLOC_PARTIAL_BYTES,
                     (unsigned)SGEMM_NOALLOC_MAX_TILES);
            return sgemm_internal::set_error(SGEMM_E_SHAPE, msg);
        }
    }
    std::unique_lock<std::mutex> lock(g_use_mutex, std::defer_lock);
    bool whole = false;   // no scratch for this call: every tile's K in one work-group, by the FP32 kernels
    if (sp.tile >= 0) {
        Scratch t;
        if (sp.partial_bytes && (r = take_scratch(h, sp.partial_bytes, sp.ticket_count, s, lock, &t)) != SGEMM_OK) {
            if (r != noalloc::kBusy) return r;
            whole = true;
            parts[0] = sgemm_internal::Part{h, m, n, 0, 0, 0, 0};
            count = 1;
        } else {
            r = sgemm_internal::bf16x6_launch(sp.tile, sp.splits, sgemm_internal::trans_a(h), sgemm_internal::trans_b(h), dA,
                                              dB, dC, dD, sp.m, sp.n, k, lda, ldb, ldc, ldd, alpha, beta, t.partials,
                                              t.tickets, s);
            if (sp.partial_bytes) r = give_scratch(h, s, t, r);
            if (r != SGEMM_OK) return r;
        }
    }
    for (int q = 0; q < count; ++q) {
        const sgemm_internal::Part& pt = parts[q];
        const float* a = dA ? dA + pt.a_off : dA;
        const float* b = dB ? dB + pt.b_off : dB;
        const float* c = dC ? dC + pt.c_off : dC;
        float* d = dD + pt.d_off;
        const sgemm_internal::Plan p = sgemm_internal::plan(pt.kh, pt.m, pt.n, k);
        // the parts run in order on one stream, so they share the scratch
        Scratch t;
        bool taken = false;
        if (p.partial_bytes && !whole) {
            r = take_scratch(h, p.partial_bytes, p.ticket_count, s, lock, &t);
            if (r != SGEMM_OK && r != noalloc::kBusy) return r;
            taken = r == SGEMM_OK;
        }
        const sgemm_internal::Workspace ws{t.partials, p.partial_bytes, t.tickets, p.ticket_count};
        r = sgemm_internal::launch(pt.kh, a, b, c, d, pt.m, pt.n, k, lda, ldb, ldc, ldd, alpha, beta, taken ? &ws : nullptr,
                                   s, !taken);
        if (taken) r = give_scratch(h, s, t, r);
        if (r != SGEMM_OK) return r;
    }
    return SGEMM_OK;
}
