// The library's scratch table (km_runtime.cpp) on the CPU: the HIP calls that it
// makes are the ones below, which count and, when told to, fail.
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstdlib>
#include <functional>

#include "km_runtime.hpp"

static int g_mallocs, g_frees, g_drains;
static bool g_full;                       // hipMalloc fails
static std::function<void()> g_between;   // runs once, in the capture-mode exchange

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t) {
    if (g_full) return hipErrorOutOfMemory;
    ++g_mallocs;
    *p = std::malloc(16);
    return hipSuccess;
}
hipError_t hipFree(void *p) {
    ++g_frees;
    std::free(p);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { ++g_drains; return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) {
    *s = hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *) {
    if (g_between) {
        auto f = std::move(g_between);
        g_between = nullptr;
        f();
    }
    return hipSuccess;
}
}

using km::Workspace;
using km::WsUse;
static hipStream_t stream(long i) { return reinterpret_cast<hipStream_t>(4096 + 64 * i); }
#define CHECK(c) do { if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; } } while (0)

int main() {
    const size_t mb = size_t(1) << 20;
    // An allocation that fails leaves nothing in the table of 64: with 62 other
    // blocks there is room for two more, whatever failed before.
    for (int i = 0; i < 62; ++i) CHECK(Workspace::reserve(mb, stream(i), WsUse::Block));
    g_full = true;
    for (int i = 100; i < 110; ++i) {
        CHECK(!Workspace::try_reserve(mb, stream(i), WsUse::Scan1DSegments));
        CHECK(!Workspace::reserve(mb, stream(i), WsUse::Block));
    }
    g_full = false;
    CHECK(Workspace::reserve(mb, stream(62), WsUse::Block));
    CHECK(Workspace::try_reserve(mb, stream(62), WsUse::Scan1DSegments));
    CHECK(g_frees == 0 && g_drains == 0);
    for (int i = 0; i < 62; ++i) CHECK(Workspace::find(stream(i), WsUse::Block));
    // A full table: optional scratch is not to be had, no block is dropped.
    CHECK(!Workspace::try_reserve(mb, stream(63), WsUse::Scan1DSegments));
    CHECK(g_frees == 0 && g_drains == 0);
    // Nor when another thread takes the last place in between.
    CHECK(Workspace::release(stream(62)) == 2 * mb);
    CHECK(Workspace::reserve(mb, stream(62), WsUse::Block));
    g_frees = g_drains = 0;
    g_between = [] { Workspace::reserve(1, stream(64), WsUse::Block); };
    CHECK(!Workspace::try_reserve(mb, stream(63), WsUse::Scan1DSegments));
    CHECK(g_frees == 0 && g_drains == 0);
    // A block that cannot grow stays, and serves calls that it is enough for.
    CHECK(Workspace::release(stream(64)) == mb);
    void *p = Workspace::try_reserve(mb, stream(62), WsUse::Scan1DSegments);
    const size_t held = Workspace::held();
    g_full = true;
    CHECK(p && !Workspace::try_reserve(2 * mb, stream(62), WsUse::Scan1DSegments));
    CHECK(Workspace::try_reserve(mb, stream(62), WsUse::Scan1DSegments) == p);
    CHECK(Workspace::held() == held);
    g_full = false;
    CHECK(Workspace::try_reserve(2 * mb, stream(62), WsUse::Scan1DSegments));
    CHECK(Workspace::held() == held + mb);
    // Mandatory scratch still takes the least recently used block's place.
    CHECK(Workspace::reserve(mb, stream(65), WsUse::Block));
    CHECK(!Workspace::find(stream(0), WsUse::Block) && Workspace::find(stream(1), WsUse::Block));
    std::puts("ok");
    for (int i = 0; i < 66; ++i) Workspace::release(stream(i));
    return Workspace::held() == 0 ? 0 : 1;
}
