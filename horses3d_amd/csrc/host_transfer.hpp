// Transfers between host arrays and the device for the hx3d engine (host code only).
#pragma once
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstddef>
#include <cstring>

namespace hxt {

// Results leave for host arrays through a ring of pinned chunks, the copy of one chunk by the host
// overlapping the transfer of the next: 13.7 MB to pageable memory took 759 us with hipMemcpyAsync (18
// GB/s); the link does 55 GB/s to pinned memory and a host core copies 75 GB/s.  hx3d_get_state into an
// array that is kept: 13.7 MB 0.88 -> 0.57 ms, 20.5 MB 1.30 -> 0.85, 320 MB 18.8 -> 12.7.  Four chunks of
// 1 MB: the first waits 20 us, and 4 MB stay pinned per engine that reads such arrays back.  Memory the
// runtime knows (the caller's own pinned arrays) goes directly, and so does everything if the ring
// cannot be had.  The other way the runtime's own staging is as good (36 GB/s), and setting a state through the
// ring measured slower: 8.6 MB 0.27 -> 0.32 ms, 20.5 MB 0.74 -> 0.82, 320 MB 11.5 -> 12.1.
// From RING_MIN bytes on: hx3d_get_state of 0.16 MB 29 us directly and 35 through the ring (67 the first time, which
// makes it), 0.88 MB 57 and 63 (87), 1.9 MB 116 and 101 (130), 2.6 MB 163 and 131 (160).
constexpr int RING_SLOTS = 4;
constexpr size_t RING_CHUNK = 1 << 20, RING_MIN = 2 << 20;

struct Ring {
    char *mem = nullptr;   // RING_SLOTS chunks, from the first transfer on
    hipEvent_t ev[RING_SLOTS] = {};
};

// Whether a transfer to `host` takes the ring, which is made if need be.  Its events must belong to the
// stream's device (hipEventRecord refuses others), so that device is made current for it: the caller
// may have another one.
inline bool use_ring(Ring &r, int device, const void *host)
{
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, host) != hipSuccess) (void)hipGetLastError();   // unknown: pageable
    else if (at.type != hipMemoryTypeUnregistered) return false;
    if (r.mem) return true;
    int current = device;
    bool ok = hipGetDevice(&current) == hipSuccess && (current == device || hipSetDevice(device) == hipSuccess);
    char *p = nullptr;
    ok = ok && hipHostMalloc((void **)&p, RING_SLOTS * RING_CHUNK, hipHostMallocDefault) == hipSuccess;
    for (int s = 0; s < RING_SLOTS && ok; ++s)
        if (!r.ev[s]) ok = hipEventCreateWithFlags(&r.ev[s], hipEventDisableTiming) == hipSuccess;
    if (!ok) {
        (void)hipGetLastError();
        if (p) (void)hipHostFree(p);
        p = nullptr;
    }
    if (current != device) (void)hipSetDevice(current);
    r.mem = p;
    return ok;
}

// With the stream idle
inline void destroy_ring(Ring &r)
{
    if (r.mem) (void)hipHostFree(r.mem);
    for (hipEvent_t e : r.ev)
        if (e) (void)hipEventDestroy(e);
    r = Ring{};
}

// bytes from the device to the host array dst, in the order of the stream (of `device`); complete on return.
// An error that the launches before it left (the kernel that packs src) is this call's result: the
// look at the pointer, which fails for every pageable array, would take its place.
inline hipError_t copy_to_host(Ring &r, int device, hipStream_t stream, void *dst, const void *src, size_t bytes)
{
    if (const hipError_t e = hipGetLastError(); e != hipSuccess) return e;
    if (bytes < RING_MIN || !use_ring(r, device, dst)) {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
        return e != hipSuccess ? e : hipStreamSynchronize(stream);
    }
    const size_t n = (bytes + RING_CHUNK - 1) / RING_CHUNK;
    auto size = [&](size_t c) { return std::min(RING_CHUNK, bytes - c * RING_CHUNK); };
    for (size_t c = 0; c < n + RING_SLOTS; ++c) {
        if (c >= RING_SLOTS) {   // chunk c - RING_SLOTS has arrived: out of its slot
            const size_t b = c - RING_SLOTS;
            if (b >= n) break;
            const hipError_t e = hipEventSynchronize(r.ev[b % RING_SLOTS]);
            if (e != hipSuccess) return e;
            std::memcpy((char *)dst + b * RING_CHUNK, r.mem + (b % RING_SLOTS) * RING_CHUNK, size(b));
        }
        if (c < n) {
            hipError_t e = hipMemcpyAsync(r.mem + (c % RING_SLOTS) * RING_CHUNK, (const char *)src + c * RING_CHUNK, size(c),
                                          hipMemcpyDeviceToHost, stream);
            if (e == hipSuccess) e = hipEventRecord(r.ev[c % RING_SLOTS], stream);
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

}  // namespace hxt
