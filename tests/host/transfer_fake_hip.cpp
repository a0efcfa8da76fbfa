// The engine's host transfers (csrc/host_transfer.hpp) over a small stand-in for the HIP runtime: two
// devices, pageable memory, and asynchronous copies that run only when something waits for them, so that
// a missing wait moves wrong data.  argv[1] names the check; exit status 0 means it held.
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <string>
#include <vector>

#include "host_transfer.hpp"

struct ihipStream_t {
    int device;
    std::vector<std::function<void()>> work;
    size_t done = 0;
    void run(size_t until)
    {
        for (; done < until; ++done) work[done]();
    }
};
struct ihipEvent_t {
    int device;
    ihipStream_t *stream = nullptr;
    size_t at = 0;
};

static int current = 0, events = 0, pinned = 0;
static hipError_t last = hipSuccess;
static hipError_t set(hipError_t e) { return e == hipSuccess ? e : last = e; }   // success leaves the last error

extern "C" {
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipGetDevice(int *d) { *d = current; return hipSuccess; }
hipError_t hipSetDevice(int d) { current = d; return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *, const void *) { return set(hipErrorInvalidValue); }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = std::malloc(n); ++pinned; return hipSuccess; }
hipError_t hipHostFree(void *p) { std::free(p); --pinned; return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = new ihipEvent_t{current};
    ++events;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) { delete e; --events; return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    if (e->device != s->device) return set(hipErrorInvalidHandle);
    e->stream = s;
    e->at = s->work.size();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (e->stream) e->stream->run(e->at);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { s->run(s->work.size()); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    st->work.push_back([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}
}

#define CHECK(x) do { if (!(x)) { std::printf("line %d: %s\n", __LINE__, #x); return 1; } } while (0)

// sizes below, at and past the ring's least, the chunks and the slots
static const size_t SIZES[] = {1, hxt::RING_MIN - 1, hxt::RING_MIN, hxt::RING_MIN + 1, 3 * hxt::RING_CHUNK - 1,
                               4 * hxt::RING_CHUNK, 4 * hxt::RING_CHUNK + 7, 11 * hxt::RING_CHUNK - 3};

static std::vector<char> bytes(size_t n, unsigned seed)
{
    std::vector<char> v(n);
    for (char &c : v) c = (char)((seed = seed * 1664525u + 1013904223u) >> 24);
    return v;
}

// twice through one ring, with another device current than the engine's
static int transfers(int caller, int device)
{
    ihipStream_t s{device};
    hxt::Ring r;
    for (int pass = 0; pass < 2; ++pass)
        for (size_t n : SIZES) {
            current = caller;
            const std::vector<char> dev = bytes(n, (unsigned)n + pass);
            std::vector<char> host(n);
            CHECK(hxt::copy_to_host(r, device, &s, host.data(), dev.data(), n) == hipSuccess);
            CHECK(host == dev);
            CHECK(current == caller);
        }
    CHECK(pinned == 1 && events == hxt::RING_SLOTS);
    hxt::destroy_ring(r);
    CHECK(pinned == 0 && events == 0);
    return 0;
}

// results below the ring's least make none
static int small_results()
{
    ihipStream_t s{0};
    hxt::Ring r;
    for (size_t n : {(size_t)1, hxt::RING_MIN - 1}) {
        const std::vector<char> dev = bytes(n, (unsigned)n);
        std::vector<char> host(n);
        CHECK(hxt::copy_to_host(r, 0, &s, host.data(), dev.data(), n) == hipSuccess);
        CHECK(host == dev && pinned == 0 && events == 0);
    }
    return 0;
}

// a failed launch before a transfer is the transfer's result, with and without a ring in place
static int failed_launch(size_t n)
{
    ihipStream_t s{0};
    hxt::Ring r;
    std::vector<char> a(n), b(n);
    for (int pass = 0; pass < 2; ++pass) {
        last = hipErrorLaunchFailure;
        CHECK(hxt::copy_to_host(r, 0, &s, a.data(), b.data(), a.size()) == hipErrorLaunchFailure);
        CHECK(hxt::copy_to_host(r, 0, &s, a.data(), b.data(), a.size()) == hipSuccess);
        CHECK(last == hipSuccess);
    }
    return 0;
}

int main(int argc, char **argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "same device") return transfers(0, 0);
    if (what == "another device current") return transfers(1, 0);
    if (what == "small results") return small_results();
    if (what == "failed launch") return failed_launch(100) || failed_launch(hxt::RING_MIN);
    return 2;
}
