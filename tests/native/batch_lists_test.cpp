// batch_lists_test.cpp -- the batch planner (goofy_amd/csrc/batch.cpp) on the
// CPU, against a device that runs nothing until it is told to: every launch is
// kept, with the work-list pointer and counts it was given, and "runs" when its
// stream is waited for (or when a captured one is replayed).  Running reads the
// list the way the kernel does, but with every index checked, and marks the
// blocks it covers.  So a list that is rewritten, resized or freed while a
// launch or a captured graph still reads it shows as an error here, with no
// GPU.  Arguments: the names of the tests to run.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <vector>

#include "internal.h"

using namespace goofy_impl;

static int g_errors = 0;
#define CHECK(cond, ...)                                         \
    do {                                                         \
        if (!(cond)) {                                           \
            ++g_errors;                                          \
            std::printf("%s:%d: %s: ", __FILE__, __LINE__, #cond); \
            std::printf(__VA_ARGS__);                            \
            std::printf("\n");                                   \
        }                                                        \
    } while (0)

// ---- the device ------------------------------------------------------------------

namespace {

std::map<const void*, size_t> g_memory;  // live device allocations
struct Launch {
    const TexDesc* descs;
    uint32_t ntex, ntiles, tile;
    hipEvent_t done;
};
struct Op {
    bool kernel;
    Launch l;
    hipEvent_t event;
    uint64_t ticket;
};
std::map<hipStream_t, std::vector<Op>> g_queue;  // not yet run
std::map<hipEvent_t, std::pair<uint64_t, uint64_t>> g_event;  // recorded, reached
std::map<hipEvent_t, hipStream_t> g_event_stream;
std::set<hipStream_t> g_capturing;
std::vector<Launch> g_captured;
hipStream_t g_per_thread = nullptr;  // what hipStreamPerThread names now
uint64_t g_ticket = 0, g_runs = 0, g_events_made = 0;
uintptr_t g_next_event = 0x1000;
std::vector<int> g_hits;  // of each block (by destination address / 8)

void run(const Launch& l)
{
    ++g_runs;
    const auto it = g_memory.find(l.descs);
    CHECK(it != g_memory.end(), "launch reads a freed work-list");
    if (it == g_memory.end()) return;
    CHECK(it->second >= worklist_bytes(l.ntex), "work-list of %zu bytes, launch reads %zu", it->second,
          worklist_bytes(l.ntex));
    if (it->second < worklist_bytes(l.ntex)) return;
    const uint32_t* tb = worklist_tile_begin(l.descs, l.ntex);
    CHECK(tb[l.ntex] == l.ntiles, "launch of %u tiles over a list of %u", l.ntiles, tb[l.ntex]);
    for (uint32_t t = 0; t < l.ntiles; ++t) {
        uint32_t i = 0;
        while (i < l.ntex && t >= tb[i + 1]) ++i;
        if (i == l.ntex) {
            CHECK(false, "tile %u is past the list's end", t);
            return;
        }
        const TexDesc& d = l.descs[i];
        const uint64_t first = (uint64_t)(t - tb[i]) * l.tile;
        CHECK(first < d.nblocks, "tile %u starts at block %llu of %u", t, (unsigned long long)first, d.nblocks);
        for (uint64_t b = first; b < first + l.tile && b < d.nblocks; ++b) ++g_hits[d.dst / 8 - 1 + b];
    }
}

void advance(hipStream_t s, uint64_t ticket)
{
    auto& q = g_queue[s];
    while (!q.empty() && q.front().ticket <= ticket) {
        const Op op = q.front();
        q.erase(q.begin());
        if (op.kernel) run(op.l);
        if (op.event && g_event.count(op.event)) g_event[op.event].second = op.ticket;
    }
}

bool reached(hipEvent_t e) { return g_event[e].second >= g_event[e].first; }

hipError_t push(hipStream_t s, bool kernel, const Launch& l, hipEvent_t e)
{
    if (s == hipStreamPerThread) s = g_per_thread;
    if (g_capturing.count(s)) {
        if (kernel) g_captured.push_back(l);
        return hipSuccess;
    }
    ++g_ticket;
    if (e) {
        g_event[e].first = g_ticket;
        g_event_stream[e] = s;
    }
    g_queue[s].push_back(Op{kernel, l, e, g_ticket});
    return hipSuccess;
}

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t n)
{
    *p = std::malloc(n);
    g_memory[*p] = n;
    return hipSuccess;
}
hipError_t hipFree(void* p)
{
    if (!p) return hipSuccess;
    CHECK(g_memory.erase(p) == 1, "free of unknown memory");
    std::memset(p, 0xEE, 1);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);  // orders no stream, as for non-blocking ones
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned)
{
    *e = (hipEvent_t)g_next_event++;
    g_event[*e] = {0, 0};
    ++g_events_made;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    CHECK(g_event.erase(e) == 1, "destroy of an unknown event");
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return push(s, false, Launch{}, e); }
hipError_t hipEventQuery(hipEvent_t e) { return reached(e) ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (!reached(e)) advance(g_event_stream[e], g_event[e].first);
    return hipSuccess;
}
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st)
{
    *st = g_capturing.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
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
    std::snprintf(out->arch, sizeof out->arch, "test");
    return GOOFY_OK;
}
LaunchCfg auto_cfg(uint64_t, int) { return LaunchCfg{1, 4, 0, 1, 0}; }
bool cfg_valid(const LaunchCfg& c) { return c.blocks_per_lane == 1 || c.blocks_per_lane == 2 || c.blocks_per_lane == 4; }
hipError_t launch_plain(int, const LaunchCfg&, const void*, size_t, void*, uint32_t, uint32_t, hipStream_t, hipEvent_t,
                        hipEvent_t)
{
    return hipSuccess;
}
hipError_t launch_batch(const LaunchCfg& c, const TexDesc* d, uint32_t ntex, uint32_t ntiles, int, hipStream_t s, bool,
                        hipEvent_t done)
{
    return push(s, true, Launch{d, ntex, ntiles, (uint32_t)tile_blocks(c), done}, done);
}
hipError_t launch_batch(const LaunchCfg& c, const TexDesc* d, uint32_t ntex, uint32_t ntiles, int n, hipStream_t s,
                        bool alpha)
{
    return launch_batch(c, d, ntex, ntiles, n, s, alpha, nullptr);
}
}  // namespace goofy_impl

// ---- tests -----------------------------------------------------------------------

namespace {

const hipStream_t kA = (hipStream_t)0x100, kB = (hipStream_t)0x200;

// 8-byte formats; sizes whose last tiles are ragged at every tile size
goofy_batch* make_plan()
{
    const unsigned sizes[][2] = {{64, 64}, {68, 20}, {260, 132}, {4, 4}, {1028, 4}};
    std::vector<goofy_texture_desc> t;
    uint64_t at = 8;  // "address" of the first block
    for (const auto& s : sizes) {
        t.push_back(goofy_texture_desc{(void*)16, (void*)(uintptr_t)at, s[0], s[1], (size_t)s[0] * 4, GOOFY_FORMAT_DXT1});
        at += (uint64_t)(s[0] / 4) * (s[1] / 4) * 8;
    }
    g_hits.assign(at / 8 - 1, 0);
    goofy_batch* b = nullptr;
    CHECK(goofy_batch_create(t.data(), t.size(), nullptr, &b) == GOOFY_OK, "create");
    return b;
}

goofy_launch_config shape(int bpl) { return goofy_launch_config{bpl, 4, 0, 1, 0}; }

void covered(int times, const char* what)
{
    for (size_t i = 0; i < g_hits.size(); ++i)
        if (g_hits[i] != times) {
            CHECK(false, "%s: block %zu written %d times, not %d", what, i, g_hits[i], times);
            break;
        }
    g_hits.assign(g_hits.size(), 0);
}

void finish(goofy_batch* b)
{
    CHECK(goofy_batch_destroy(b) == GOOFY_OK, "destroy");
    CHECK(g_memory.empty(), "%zu allocations left", g_memory.size());
    CHECK(g_event.empty(), "%zu events left", g_event.size());
    g_queue.clear();
    g_captured.clear();
    g_events_made = 0;
}

// A captured launch reads its list whatever the plan does afterwards.
void captured()
{
    goofy_batch* b = make_plan();
    g_capturing = {kA};
    CHECK(goofy_batch_launch(b, kA) == GOOFY_OK, "launch under capture");
    g_capturing.clear();
    for (int bpl : {4, 2, 1, 4}) {
        goofy_launch_config c = shape(bpl);
        CHECK(goofy_batch_set_config(b, &c) == GOOFY_OK, "set_config");
        for (const Launch& l : g_captured) run(l);
        covered((int)g_captured.size(), "replay after set_config");
        g_capturing = {kA};  // a second graph with the new shape
        CHECK(goofy_batch_launch(b, kA) == GOOFY_OK, "launch under capture");
        g_capturing.clear();
    }
    CHECK(goofy_batch_autotune(b, kB, 1, nullptr, nullptr) == GOOFY_OK, "autotune");
    advance(kB, g_ticket);
    g_hits.assign(g_hits.size(), 0);
    for (const Launch& l : g_captured) run(l);
    covered((int)g_captured.size(), "replay after autotune");
    CHECK(g_memory.size() <= 3, "%zu work-lists for three tile sizes", g_memory.size());
    finish(b);
}

uint64_t left(hipStream_t s)
{
    uint64_t n = 0;
    for (const Op& op : g_queue[s]) n += op.kernel;
    return n;
}

// set_config, autotune and destroy wait for the launches of every stream.
void streams()
{
    goofy_batch* b = make_plan();
    const goofy_launch_config same = shape(1), other = shape(4);
    for (const goofy_launch_config* c : {&same, &other, &same}) {
        for (hipStream_t s : {kA, kA, kB, (hipStream_t) nullptr})
            CHECK(goofy_batch_launch(b, s) == GOOFY_OK, "launch");
        CHECK(left(kA) == 2 && left(kB) == 1 && left(nullptr) == 1, "launches wait for nothing");
        CHECK(goofy_batch_set_config(b, c) == GOOFY_OK, "set_config");
        CHECK(left(kA) + left(kB) + left(nullptr) == 0, "launches left after set_config: %d %d %d", (int)left(kA),
              (int)left(kB), (int)left(nullptr));
        covered(4, "launches on three streams");
    }
    for (hipStream_t s : {kB, kA}) CHECK(goofy_batch_launch(b, s) == GOOFY_OK, "launch");
    CHECK(goofy_batch_autotune(b, kB, 1, nullptr, nullptr) == GOOFY_OK, "autotune");
    CHECK(left(kA) == 0, "launches left after autotune");
    advance(kB, g_ticket);
    for (hipStream_t s : {kA, kB}) CHECK(goofy_batch_launch(b, s) == GOOFY_OK, "launch");
    CHECK(goofy_batch_destroy(b) == GOOFY_OK, "destroy");
    CHECK(left(kA) + left(kB) == 0, "launches left after destroy: %d %d", (int)left(kA), (int)left(kB));
    CHECK(g_memory.empty() && g_event.empty(), "%zu allocations, %zu events left", g_memory.size(), g_event.size());
    g_queue.clear();
}

// The handle of the per-thread default stream names another stream in every
// thread: here its launches alternate between two.
void per_thread()
{
    goofy_batch* b = make_plan();
    for (hipStream_t s : {kA, kB}) {
        g_per_thread = s;
        CHECK(goofy_batch_launch(b, hipStreamPerThread) == GOOFY_OK, "launch");
    }
    const goofy_launch_config c = shape(2);
    CHECK(goofy_batch_set_config(b, &c) == GOOFY_OK, "set_config");
    CHECK(left(kA) + left(kB) == 0, "launches left after set_config: %d %d", (int)left(kA), (int)left(kB));
    covered(2, "launches on two threads' streams");
    finish(b);
}

// As many events as streams with unfinished launches, or a few more, not as
// launches or streams.
void events()
{
    goofy_batch* b = make_plan();
    for (int i = 0; i < 1000; ++i) {
        CHECK(goofy_batch_launch(b, kA) == GOOFY_OK, "launch");
        CHECK(goofy_batch_launch(b, kB) == GOOFY_OK, "launch");
    }
    CHECK(g_events_made == 2, "%d events for two streams", (int)g_events_made);
    for (int i = 0; i < 1000; ++i) {
        const hipStream_t s = (hipStream_t)(uintptr_t)(0x1000 + 16 * i);
        CHECK(goofy_batch_launch(b, s) == GOOFY_OK, "launch");
        advance(s, g_ticket);
    }
    CHECK(g_events_made <= 8, "%d events for three streams at a time", (int)g_events_made);
    finish(b);
}

// The tuning file (GOOFY_TUNE_CACHE): rows of a build whose shapes meant
// something else are left alone, those of this one are taken.  One process each,
// as the file is read once.
void expect(const char* what, const goofy_launch_config& want)
{
    goofy_batch* b = make_plan();
    goofy_launch_config c{};
    CHECK(goofy_batch_get_config(b, &c) == GOOFY_OK && !std::memcmp(&c, &want, sizeof c),
          "%s: %d blocks per lane, %d waves, %d per CU, streaming %d, order %d", what, c.blocks_per_lane, c.wg_waves,
          c.waves_per_cu, c.nontemporal, c.tile_order);
    finish(b);
}
void tune_file_foreign() { expect("shape after a foreign file", shape(1)); }
void tune_file_write()
{
    goofy_batch* b = make_plan();
    CHECK(goofy_batch_autotune(b, nullptr, 1, nullptr, nullptr) == GOOFY_OK, "autotune");
    advance(nullptr, g_ticket);
    finish(b);
}
void tune_file_read() { expect("shape after our file", goofy_launch_config{1, 2, 0, 0, 0}); }  // all alike: the first

const struct {
    const char* name;
    void (*go)();
} kTests[] = {{"captured", captured}, {"streams", streams}, {"per_thread", per_thread}, {"events", events},
             {"tune_file_foreign", tune_file_foreign}, {"tune_file_write", tune_file_write},
             {"tune_file_read", tune_file_read}};

}  // namespace

int main(int argc, char** argv)
{
    for (const auto& t : kTests) {
        bool want = false;
        for (int i = 1; i < argc; ++i) want |= !std::strcmp(argv[i], t.name);
        if (want) t.go();
    }
    std::printf("errors=%d\n", g_errors);
    return g_errors != 0;
}
