// dropin_host_test.cpp -- the host side of the drop-in (goofy_amd/csrc/capi.cpp)
// on the CPU.  The HIP runtime is a stand-in whose "fed kernel" is a thread:
// launched before the rows are staged, it waits for the parts that each group
// of blocks lies in, writes a digest of every block's 64 bytes and marks the
// group, as k_encode_fed does.  A part marked before its rows are staged, or
// blocks collected before they are marked, is a data race (ThreadSanitizer) or
// a wrong digest.  Arguments: the names of the tests to run (none: all).
#include <hip/hip_runtime_api.h>

#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>


#include "internal.h"

using namespace goofy_impl;

static std::atomic<int> g_errors{0};
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

std::mutex g_mu;
std::map<hipStream_t, std::vector<std::thread>> g_running;
size_t g_largest_part = 0, g_largest_launch = 0, g_launches = 0;  // bytes of pixels
bool g_late = false;                                              // fed kernels give up at once
std::atomic<int> g_fed_us{0};                                      // how long kernels take that are launched before staging
std::atomic<int> g_unstaged{0}, g_most_unstaged{0};               // kernels that wait for their hosts
uintptr_t g_next = 0x1000;

uint64_t digest(const uint8_t* src, size_t pitch, uint64_t bx, uint64_t by, int fmt)
{
    uint64_t h = 1469598103934665603ull + (uint64_t)fmt;
    for (int y = 0; y < 4; ++y)
        for (int i = 0; i < 2; ++i) {
            uint64_t v;
            std::memcpy(&v, src + (by * 4 + (uint64_t)y) * pitch + bx * 16 + 8 * i, 8);
            h = (h ^ v) * 1099511628211ull;
        }
    return h;
}

size_t bytes_per_block(int fmt) { return fmt == kFeedDualAlpha ? 16 : fmt == kFeedDual ? 8 : block_bytes(fmt); }

void write_block(int fmt, uint8_t* dst, uint8_t* dst2, uint64_t b, uint64_t h)
{
    const size_t bb = bytes_per_block(fmt);
    for (size_t i = 0; i < bb; i += 8) std::memcpy(dst + b * bb + i, &h, 8);
    const uint64_t h2 = ~h;
    if (fmt >= kFeedDual)
        for (size_t i = 0; i < bb; i += 8) std::memcpy(dst2 + b * bb + i, &h2, 8);
}

void wait(hipStream_t s)
{
    std::vector<std::thread> t;
    {
        std::lock_guard<std::mutex> lock(g_mu);
        t.swap(g_running[s]);
    }
    for (std::thread& x : t) x.join();
}

}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int* n) { return *n = 1, hipSuccess; }
hipError_t hipGetDevice(int* d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int)
{
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return *p = std::aligned_alloc(256, (n + 255) & ~(size_t)255), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned)
{
    std::lock_guard<std::mutex> lock(g_mu);
    return *s = (hipStream_t)(g_next += 16), hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return wait(s), hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)16, hipSuccess; }
hipError_t hipEventCreate(hipEvent_t* e) { return *e = (hipEvent_t)16, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { return *ms = 1, hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
}

namespace goofy_impl {
hipError_t launch_fed(int fmt, const void* src, size_t pitch, void* dst, void* dst2, uint32_t bw, uint32_t nblocks,
                      HostFeed* feed, uint64_t call, uint32_t part_blocks, uint64_t, hipStream_t stream)
{
    if (nblocks == 0 || (part_blocks && (nblocks - 1u) / part_blocks >= kFeedParts)) return hipErrorInvalidValue;
    wait(stream);  // one kernel of a stream at a time: every earlier one's rows are staged
    std::lock_guard<std::mutex> lock(g_mu);
    ++g_launches;
    g_largest_launch = std::max(g_largest_launch, (size_t)nblocks * 64);
    if (part_blocks) g_largest_part = std::max(g_largest_part, (size_t)part_blocks * 64);
    const bool late = g_late && part_blocks;
    if (part_blocks) g_most_unstaged = std::max(g_most_unstaged.load(), ++g_unstaged);
    g_running[stream].emplace_back([=] {
        for (uint32_t group = 0; group < feed_groups(nblocks); ++group) {
            const uint32_t first = group * kFeedBlocks, end = std::min(first + kFeedBlocks, nblocks);
            if (part_blocks)
                for (uint32_t p = first / part_blocks; p <= (end - 1) / part_blocks; ++p)
                    while (__atomic_load_n(&feed->part[p].staged, __ATOMIC_ACQUIRE) != call) {
                        if (late) {
                            --g_unstaged;
                            __atomic_store_n(&feed->gave_up, call, __ATOMIC_RELEASE);
                            return;
                        }
                        std::this_thread::yield();
                    }
            if (part_blocks && end == nblocks) --g_unstaged;
            if (part_blocks && end == nblocks) std::this_thread::sleep_for(std::chrono::microseconds(g_fed_us));
            for (uint32_t b = first; b < end; ++b)
                write_block(fmt, (uint8_t*)dst, (uint8_t*)dst2, b,
                            digest((const uint8_t*)src, pitch, b % bw, b / bw, fmt));
            if (group < kFeedMarks) __atomic_store_n(&feed->done[group], call, __ATOMIC_RELEASE);
        }
    });
    return hipSuccess;
}
static hipError_t launch_now(int fmt, const void* src, size_t pitch, void* dst, void* dst2, uint32_t bw, uint32_t n,
                             hipStream_t s)
{
    wait(s);
    for (uint32_t b = 0; b < n; ++b)
        write_block(fmt, (uint8_t*)dst, (uint8_t*)dst2, b, digest((const uint8_t*)src, pitch, b % bw, b / bw, fmt));
    return hipSuccess;
}
hipError_t launch_plain(int fmt, const LaunchCfg&, const void* src, size_t pitch, void* dst, uint32_t bw, uint32_t n,
                        hipStream_t s, hipEvent_t, hipEvent_t)
{
    return launch_now(fmt, src, pitch, dst, nullptr, bw, n, s);
}
hipError_t launch_dual(const LaunchCfg&, const void* src, size_t pitch, void* a, void* b, uint32_t bw, uint32_t n,
                       hipStream_t s, hipEvent_t, hipEvent_t)
{
    return launch_now(kFeedDual, src, pitch, a, b, bw, n, s);
}
hipError_t launch_dual_alpha(const LaunchCfg&, const void* src, size_t pitch, void* a, void* b, uint32_t bw, uint32_t n,
                             hipStream_t s, hipEvent_t, hipEvent_t)
{
    return launch_now(kFeedDualAlpha, src, pitch, a, b, bw, n, s);
}
hipError_t launch_synth(const void*, void*, uint32_t, uint32_t, size_t, hipStream_t) { return hipSuccess; }
}  // namespace goofy_impl

namespace {

// One call; every block has to be the digest of its own pixels, and nothing
// may be written behind the last.
void compare(int fmt, unsigned w, unsigned h, unsigned extra)
{
    const size_t stride = (size_t)w * 4 + extra, n = (size_t)(w / 4) * (h / 4), bb = bytes_per_block(fmt);
    std::vector<uint8_t> img(stride * h), a(n * bb + 64, 0xCD), b(n * bb + 64, 0xCD);
    uint64_t x = 88172645463325252ull + w + h;
    for (size_t i = 0; i + 8 <= img.size(); i += 8) {
        x ^= x << 13, x ^= x >> 7, x ^= x << 17;
        std::memcpy(&img[i], &x, 8);
    }
    const int rc = fmt == kFeedDual ? goofy_hip_compress_dual(a.data(), b.data(), img.data(), w, h, (unsigned)stride)
                   : fmt == kFeedDualAlpha
                       ? goofy_hip_compress_dual_alpha(a.data(), b.data(), img.data(), w, h, (unsigned)stride)
                       : goofy_hip_compress(fmt, a.data(), img.data(), w, h, (unsigned)stride);
    CHECK(rc == GOOFY_OK, "%ux%u format %d: %d", w, h, fmt, rc);
    for (size_t i = 0; i < n; ++i) {
        const uint64_t want = digest(img.data(), stride, i % (w / 4), i / (w / 4), fmt), want2 = ~want;
        if (std::memcmp(&a[i * bb], &want, 8) || (fmt >= kFeedDual && std::memcmp(&b[i * bb], &want2, 8))) {
            CHECK(false, "%ux%u format %d: block %zu of %zu", w, h, fmt, i, n);
            break;
        }
    }
    for (size_t i = n * bb; i < a.size(); ++i) CHECK(a[i] == 0xCD && b[i] == 0xCD, "written behind the blocks");
}

// Every path of the staging: small, one chunk, several, very wide rows.
void sizes()
{
    const unsigned list[][3] = {{16, 4, 0},       {128, 256, 16},   {2048, 32, 0},    {32768, 16, 64},  {65536, 4, 0},
                                {65552, 12, 0},   {2048, 2052, 0},  {262144, 16, 0},  {262160, 8, 16},  {524288, 4, 0},
                                {524304, 8, 0},   {1048592, 8, 32}, {2097152, 4, 0},  {4194288, 4, 0}};
    for (const auto& s : list)
        for (int late : {0, 1}) {
            g_late = late;
            const size_t px = (size_t)s[0] * s[1];
            compare(0, s[0], s[1], s[2]);
            if (px > (1u << 22)) continue;  // the time under ThreadSanitizer
            for (int fmt : {(int)GOOFY_FORMAT_DXT5, kFeedDual, kFeedDualAlpha}) compare(fmt, s[0], s[1], s[2]);
        }
    g_late = false;
}

// However wide the rows, a thread copies about a MiB at a time, so that the
// kernel can start early and the threads share the work, and no launch is
// larger than its marks reach.
void wide()
{
    for (unsigned w : {262144u, 524288u, 524304u, 1048592u, 2097152u, 4194288u}) {
        g_largest_part = g_largest_launch = g_launches = 0;
        compare(0, w, 4, 0);
        CHECK(g_largest_part && g_largest_part <= (5u << 18), "%u pixels a row: a part of %zu KiB", w,
              g_largest_part >> 10);
        CHECK(g_largest_launch <= (size_t)kFeedMarks * kFeedBlocks * 64, "%u pixels a row: a launch of %zu KiB", w,
              g_largest_launch >> 10);
    }
}

// Several threads at once: of all callers, one kernel of 2 MiB and more at a
// time waits for its host thread, or three smaller ones, and the turns for that
// come back from calls of every kind.
void threads()
{
    for (int run : {0, 1, 2, 3}) {
        const bool mixed = run & 1;
        g_late = run & 2;
        g_most_unstaged = 0;
        std::vector<std::thread> t;
        for (unsigned i = 0; i < 4; ++i)
            t.emplace_back([i, mixed] {
                for (unsigned r = 0; r < 3; ++r) {
                    compare(0, 2048, 516 + 1024 * (i & 1), 0);
                    compare(0, 64, 64, 0);
                    for (unsigned k = 0; mixed && k < 20; ++k) compare(GOOFY_FORMAT_ETC1, 128 + 16 * i, 256, 16);
                }
            });
        for (std::thread& x : t) x.join();
        CHECK(g_most_unstaged >= 1 && g_most_unstaged <= (mixed ? 3 : 1), "%d kernels waited for their hosts at once",
              g_most_unstaged.load());
    }
    g_late = false;
    for (unsigned h : {512u, 2048u}) {
        g_most_unstaged = 0;
        compare(0, 512, h, 0);
        CHECK(g_most_unstaged == 1, "a turn was lost");
    }
}

// A caller with a new context does not wait for a kernel whose rows another
// caller has not staged, or which takes long.
void waiting()
{
    const unsigned w = 1024, h = 512;  // 2 MiB
    std::vector<uint8_t> img((size_t)w * h * 4, 1), out((size_t)w * h / 2), out2(out.size());
    const auto call = [&](std::vector<uint8_t>& o) {
        CHECK(goofy_hip_compress(0, o.data(), img.data(), w, h, w * 4) == GOOFY_OK, "call");
    };
    g_fed_us = 1500000;
    std::thread other([&] { call(out2); });  // has the turn meanwhile
    std::this_thread::sleep_for(std::chrono::milliseconds(50));
    const auto t0 = std::chrono::steady_clock::now();
    for (int i = 0; i < 5; ++i) call(out);
    const double wall = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    CHECK(wall < 1.2, "%.0f ms: waited for the other caller", wall * 1e3);
    other.join();
    g_fed_us = 0;
}

const struct {
    const char* name;
    void (*go)();
} kTests[] = {{"sizes", sizes}, {"wide", wide}, {"threads", threads}, {"waiting", waiting}};

}  // namespace

int main(int argc, char** argv)
{
    for (const auto& t : kTests) {  // "waiting" in a process of its own: it needs new contexts
        bool want = argc < 2 && t.go != waiting;
        for (int i = 1; i < argc; ++i) want |= !std::strcmp(argv[i], t.name);
        if (want) t.go();
    }
    for (auto& r : g_running)
        for (std::thread& t : r.second) t.join();
    std::printf("errors=%d\n", g_errors.load());
    return g_errors != 0;
}
