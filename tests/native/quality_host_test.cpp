// quality_host_test.cpp -- the host side of the pooled quality calls
// (goofy_amd/csrc/codec_api.cpp) on the CPU: the HIP runtime and the kernel
// launchers are stand-ins that count what is queued and write a launch's words
// when a test says so.  Arguments: the names of the tests to run (none: all).
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>

#include "internal.h"

using namespace goofy_impl;

static int g_errors = 0;
#define CHECK(cond, ...)                                           \
    do {                                                           \
        if (!(cond)) {                                             \
            ++g_errors;                                            \
            std::printf("%s:%d: %s: ", __FILE__, __LINE__, #cond); \
            std::printf(__VA_ARGS__);                              \
            std::printf("\n");                                     \
        }                                                          \
    } while (0)

namespace {

struct Counts {
    int memset, launch, record, sync, copy;
    int all() const { return memset + launch + record + sync + copy; }
} g_n;
bool g_capturing = false;
bool g_writes = true;  // launches write their words

hipError_t launched(const QualityDest& dest)
{
    ++g_n.launch;
    if (g_writes && dest.host)
        for (uint32_t k = 0; k < kQualityWords; ++k) dest.host->word[k] = k + 1;
    return hipSuccess;
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::malloc(n), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)16, hipSuccess; }
hipError_t hipMemsetAsync(void* p, int v, size_t n, hipStream_t)
{
    ++g_n.memset;
    std::memset(p, v, n);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return ++g_n.record, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return ++g_n.sync, hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* st)
{
    *st = g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void*, size_t n, hipMemcpyKind, hipStream_t)
{
    ++g_n.copy;
    std::memset(d, 0, n);
    return hipSuccess;
}
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace goofy_impl {
int fail(int code, const std::string&) { return code; }
int fail_hip(hipError_t, const char*) { return GOOFY_ERR_HIP; }
void clear_error() {}
int device_info(DeviceInfo* out)
{
    *out = DeviceInfo{};
    out->num_cus = 256;
    return GOOFY_OK;
}
LaunchCfg auto_cfg(uint64_t, int) { return LaunchCfg{1, 4, 0, 1, 0}; }
hipError_t launch_decode(int, const void*, void*, uint32_t, uint32_t, size_t, hipStream_t) { return hipSuccess; }
hipError_t launch_sqerr(int, const void*, const void*, size_t, uint32_t, uint32_t, const QualityDest& d, bool,
                        hipStream_t)
{
    return launched(d);
}
hipError_t launch_sqerr_images(const void*, size_t, const void*, size_t, uint32_t, uint32_t, const QualityDest& d,
                               hipStream_t)
{
    return launched(d);
}
hipError_t noalloc_scratch_address(int, void**) { return hipSuccess; }
hipError_t launch_rgb565_baseline(const void*, size_t, void*, size_t, uint32_t, uint32_t, hipStream_t, hipEvent_t,
                                  hipEvent_t)
{
    return hipSuccess;
}
hipError_t launch_traffic_probe(const void*, size_t, void*, uint32_t, uint32_t, uint32_t, hipStream_t, hipEvent_t,
                                hipEvent_t)
{
    return hipSuccess;
}
}  // namespace goofy_impl

namespace {

void* const kMem = (void*)(uintptr_t)4096;

int images(goofy_quality* q) { return goofy_hip_quality_images_device(kMem, 1024, kMem, 1024, 256, 64, nullptr, q); }
int noalloc(goofy_quality* q)
{
    return goofy_hip_quality_device_noalloc(0, kMem, kMem, 256, 64, 1024, nullptr, q);
}
int blocks(goofy_quality* q) { return goofy_hip_quality_device(0, kMem, kMem, 256, 64, 1024, nullptr, q); }

void right(int (*call)(goofy_quality*), const char* what)
{
    goofy_quality q{};
    CHECK(call(&q) == GOOFY_OK, "%s", what);
    for (int i = 0; i < 4; ++i) CHECK(q.sse_byte[i] == (uint64_t)i + 1, "%s: byte %d", what, i);
    CHECK(q.sse_luma == (5.0 + 6.0 * 4294967296.0) / 1e4, "%s: luma", what);
}

// On a capturing stream nothing is queued: neither the kernel nor the clearing
// of a new work area may become a node of the caller's graph.
void capture()
{
    for (auto call : {images, blocks})
        for (int round = 0; round < 2; ++round) {  // with a new work area and a kept one
            goofy_quality q{};
            g_capturing = true;
            g_n = {};
            CHECK(call(&q) == GOOFY_ERR_HIP, "under capture");
            CHECK(g_n.all() == 0, "queued under capture: %d memsets, %d launches, %d records, %d waits", g_n.memset,
                  g_n.launch, g_n.record, g_n.sync);
            g_capturing = false;
            right(call, "after a capture");
        }
    goofy_quality q{};
    g_capturing = true;
    g_n = {};
    CHECK(noalloc(&q) == GOOFY_ERR_HIP, "under capture");
    CHECK(g_n.all() == 0, "queued under capture: %d launches, %d copies, %d waits", g_n.launch, g_n.copy, g_n.sync);
    g_capturing = false;
    CHECK(noalloc(&q) == GOOFY_OK && g_n.launch == 1 && g_n.copy == 1, "after a capture");
}

// Words that are still unwritten when the stream has drained are an error, not
// figures; the next call clears the work area and is right.
void unwritten()
{
    for (auto call : {images, blocks}) {
        goofy_quality q{};
        q.pixels = 7;
        g_writes = false;
        CHECK(call(&q) == GOOFY_ERR_HIP, "no words");
        CHECK(q.pixels == 7, "figures from no words");
        g_writes = true;
        g_n = {};
        right(call, "after a call without words");
        CHECK(g_n.memset == 1, "%d memsets", g_n.memset);
    }
}

const struct {
    const char* name;
    void (*go)();
} kTests[] = {{"capture", capture}, {"unwritten", unwritten}};

}  // namespace

int main(int argc, char** argv)
{
    for (const auto& t : kTests) {
        bool want = argc < 2;
        for (int i = 1; i < argc; ++i) want |= !std::strcmp(argv[i], t.name);
        if (want) t.go();
    }
    std::printf("errors=%d\n", g_errors);
    return g_errors != 0;
}
