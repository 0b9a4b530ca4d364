// capi.cpp -- single-image entry points of libgoofy_hip.so: the drop-in
// goofy::compressDXT1 / compressETC1 (host memory, synchronous), the device
// pointer / stream variant, error reporting and the synthetic-input fill.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "goofy_hip.h"
#include "goofy_tc.h"
#include "copy_pool.h"
#include "internal.h"
#include "synth.h"

namespace goofy_impl {

// ---- errors -----------------------------------------------------------------

static thread_local std::string t_last_error;

int fail(int code, const std::string& msg)
{
    t_last_error = msg;
    return code;
}

int fail_hip(hipError_t e, const char* what)
{
    const int code = (e == hipErrorOutOfMemory || e == hipErrorMemoryAllocation) ? GOOFY_ERR_OUT_OF_MEMORY
                     : (e == hipErrorNoDevice)                                     ? GOOFY_ERR_NO_DEVICE
                                                                                   : GOOFY_ERR_HIP;
    return fail(code, std::string(what) + ": " + hipGetErrorString(e));
}

void clear_error() { t_last_error.clear(); }

// ---- device -------------------------------------------------------------------

constexpr int kMaxDevices = 64;

int device_info(DeviceInfo* out)
{
    static std::mutex mu;
    static DeviceInfo cache[kMaxDevices];
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
        (void)hipGetLastError();
        return fail(GOOFY_ERR_NO_DEVICE, "no GPU visible");
    }
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return fail_hip(e, "hipGetDevice");
    if (dev < 0 || dev >= kMaxDevices) return fail(GOOFY_ERR_INVALID, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (cache[dev].device != dev) {
        hipDeviceProp_t prop;
        e = hipGetDeviceProperties(&prop, dev);
        if (e != hipSuccess) return fail_hip(e, "hipGetDeviceProperties");
        cache[dev].num_cus = prop.multiProcessorCount;
        cache[dev].total_mem = prop.totalGlobalMem;
        std::snprintf(cache[dev].arch, sizeof(cache[dev].arch), "%s", prop.gcnArchName);
        cache[dev].device = dev;
    }
    *out = cache[dev];
    return GOOFY_OK;
}

// The shape of small and middling launches, and what wide_cfg starts from for
// large ones: one block per lane (4 lose ~10% at 8192^2), streaming loads and
// stores, linear tile order, and the largest workgroup (8, 4, 2 or 1 waves)
// that still leaves two workgroups per CU: up to 8192 tiles 8-wave workgroups
// are the fastest linear shape (3000x2052 DXT1 5.7 us, 5.8 / 5.9 / 6.0 in 4- /
// 2- / 1-wave ones), while a texture of a few hundred tiles needs smaller ones
// to reach every CU.
LaunchCfg auto_cfg(uint64_t blocks, int num_cus)
{
    const uint64_t tiles = (blocks + 63u) / 64u;
    const uint64_t want = 2u * (uint64_t)(num_cus > 0 ? num_cus : 1);
    int wg = 8;
    while (wg > 1 && (tiles + (uint64_t)wg - 1) / (uint64_t)wg < want) wg >>= 1;
    return LaunchCfg{1, wg, 0, 1, 0};
}

bool cfg_valid(const LaunchCfg& c)
{
    const bool bpl = c.blocks_per_lane == 1 || c.blocks_per_lane == 2 || c.blocks_per_lane == 4;
    const bool wg = c.wg_waves == 1 || c.wg_waves == 2 || c.wg_waves == 4 || c.wg_waves == 8;
    return bpl && wg && c.waves_per_cu >= 0 && c.waves_per_cu <= 256 && (c.nontemporal == 0 || c.nontemporal == 1) &&
           (c.tile_order == 0 || c.tile_order == 1);
}

// ---- host-memory drop-in: pinned staging, read by the kernels themselves ------
//
// goofy::compressDXT1/ETC1 take pageable host buffers.  The image goes in
// chunks of at most 8 MiB of pixels through three pinned staging slots.  A chunk's kernel (k_encode_fed) is launched before any of its
// rows is staged, reads the slot over PCIe part by part as the host marks the
// parts, writes its blocks to pinned memory over PCIe and marks them group by
// group, so that the link runs from the first part staged to the last block,
// and the host copies rows in and blocks out meanwhile (a caller's chunks behind
// the one that is so launched, and other callers' chunks: StagingLink).  DXT1 /
// ETC2 RGBA8 in us per call; in the middle images up to 8 MiB with a fed kernel
// and a stream synchronisation before the blocks were copied out, larger ones by
// copy engines both ways (8 MiB chunks, plain kernels); on the left images up to
// 8 MiB with a plain kernel per 512 KiB staged:
//     64x64      18 / 18     ->    17 / 17     ->    14 / 15
//    512x512     55 / 59     ->    45 / 49     ->    38 / 40
//   1440x1448   274 / 328    ->   227 / 274    ->   194 / 198
//   2048x2048   490 / 532    ->   494 / 535    ->   400 / 405
//   4096x4096  1485 / 1540   ->  1490 / 1545   ->  1350 / 1385
//   8192x8192  5455 / 5860   ->  5450 / 5820   ->  5140 / 5170
// The kernels read 52 GB/s over the link.  With the first chunk fed and copy
// engines for the others the calls were bound by the host (4096x4096 1473 /
// 1617, 8192x8192 5530 / 6790).
//   A slot is refilled after its chunk's blocks are collected.  Between a fed
// launch and the mark of the chunk's last part the host calls nothing that
// could wait for the device, so the kernel's wait ends whatever other threads
// and streams do.  Should this thread stand still for `patience` ticks, the
// kernel ends unfinished, and the chunk, all staged by then, is encoded by a
// plain launch.  Images below 128 KiB are staged first: a look at a mark over
// PCIe costs more than it hides there; so is every chunk where a launch returns
// only after its kernel.
//   Contexts (streams, events, pinned buffers) come from a process-wide pool:
// concurrent callers never share one, and nothing is freed at thread exit (the
// HIP runtime may already be gone then).

constexpr int kSlots = 3;
constexpr uint64_t kFeedPatience = 2000000;  // 20 ms in 10 ns ticks
constexpr size_t kWidePart = (size_t)1 << 20;

// Whether a launch returns only when its kernel has ended.
static bool launches_block()
{
    for (const char* name : {"HIP_LAUNCH_BLOCKING", "AMD_SERIALIZE_KERNEL"}) {
        const char* v = std::getenv(name);
        if (v && *v && std::strcmp(v, "0") != 0) return true;
    }
    return false;
}

// A device's link, and who of its callers may have a kernel there that waits for
// its host thread (a turn, from the launch to the last block collected): one
// chunk of 2 MiB and more at a time, on stream[0], or up to three smaller ones.
// Chunks that get no turn are staged first; the large ones then follow one
// another on stream[1], so that two at most share the link.  With the kernels
// of all callers beside each other, callers that had started together ended
// together, and the link stood still while they staged their next images.  In
// us per image with 1 / 2 / 4 threads, copy engines -> every chunk launched
// before it is staged -> with turns:
//    512x512      53 / 44 / 29       ->    35 / 30 / 22       ->    36 / 30 / 22
//   1024x1024    150 / 115 / 97      ->   107 / 97 / 86       ->   107 / 94 / 83
//   2048x2048    498 / 324 / 326     ->   410 / 365 / 335     ->   408 / 318 / 318
//   4096x4096   1508 / 1300 / 1308   ->  1390 / 1355 / 1340   ->  1370 / 1250 / 1250
// 512x512 with all chunks in turn on the two streams: 35 / 36 / 24.
struct StagingLink {
    std::atomic<int> turns{0};
    hipStream_t stream[2] = {};
};

struct StagingCtx {
    int device = -1;
    StagingLink* link = nullptr;
    hipStream_t stream = nullptr;  // of chunks below 2 MiB
    hipEvent_t ended[2] = {};
    struct Slot {
        uint8_t* in = nullptr;     // staged rows
        uint8_t* out = nullptr;    // blocks, a pair's second format behind the first
        HostFeed* feed = nullptr;  // the marks of the slot's parts and groups
    } slot[kSlots];
    size_t in_cap = 0, out_cap = 0;
    uint64_t call = 0;  // the number of the last launch
    bool turn = false;  // this call has one of the link's turns
    const bool stage_first = launches_block();

    bool take_turn(int limit)  // false too where an earlier chunk of this call has one
    {
        if (turn) return false;
        if (link->turns.fetch_add(1, std::memory_order_acquire) < limit) return turn = true;
        link->turns.fetch_sub(1, std::memory_order_relaxed);
        return false;
    }
    bool others_have_turns() const { return link->turns.load(std::memory_order_relaxed) > (turn ? 1 : 0); }
    void give_turn()
    {
        if (turn) link->turns.fetch_sub(1, std::memory_order_release);
        turn = false;
    }
};

class StagingPool {
public:
    StagingCtx* acquire(int device)
    {
        std::lock_guard<std::mutex> lock(mu_);
        for (size_t i = 0; i < free_.size(); ++i)
            if (free_[i]->device == device) {
                StagingCtx* c = free_[i];
                free_.erase(free_.begin() + (long)i);
                return c;
            }
        StagingCtx* c = new StagingCtx();
        c->device = device;
        c->link = &links_[device];
        return c;
    }
    // Makes the streams of a link.
    hipError_t ensure_link(StagingLink* l)
    {
        std::lock_guard<std::mutex> lock(mu_);
        hipError_t e = hipSuccess;
        for (hipStream_t& s : l->stream)
            if (!s && e == hipSuccess) e = hipStreamCreateWithFlags(&s, hipStreamNonBlocking);
        return e;
    }
    void release(StagingCtx* c)
    {
        std::lock_guard<std::mutex> lock(mu_);
        free_.push_back(c);
    }

private:
    std::mutex mu_;
    std::vector<StagingCtx*> free_;
    StagingLink links_[kMaxDevices];
};

static StagingPool& staging_pool()
{
    static StagingPool* pool = new StagingPool();  // never destroyed
    return *pool;
}

static int ensure_ctx(StagingCtx* c, size_t in_bytes, size_t out_bytes)
{
    hipError_t e;
    if (!c->stream) {
        if ((e = staging_pool().ensure_link(c->link)) != hipSuccess ||
            (e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess)
            return fail_hip(e, "hipStreamCreate");
    }
    for (hipEvent_t& ev : c->ended)
        if (!ev && (e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) != hipSuccess)
            return fail_hip(e, "hipEventCreate");
    if (c->in_cap < in_bytes || c->out_cap < out_bytes) {
        if (c->in_cap)  // its last kernels have marked their blocks, but may not have ended
            for (hipStream_t s : {c->stream, c->link->stream[0], c->link->stream[1]}) (void)hipStreamSynchronize(s);
        const size_t ni = std::max(in_bytes, c->in_cap), no = std::max(out_bytes, c->out_cap);
        for (StagingCtx::Slot& s : c->slot) {
            if (s.in) (void)hipHostFree(s.in);
            if (s.out) (void)hipHostFree(s.out);
            s.in = s.out = nullptr;
        }
        c->in_cap = c->out_cap = 0;
        for (StagingCtx::Slot& s : c->slot) {
            // coherent: kernels and host read and write it while both run
            if ((e = hipHostMalloc((void**)&s.in, ni, hipHostMallocCoherent)) != hipSuccess ||
                (e = hipHostMalloc((void**)&s.out, no, hipHostMallocCoherent)) != hipSuccess)
                return fail_hip(e, "hipHostMalloc(staging)");
            if (!s.feed) {
                if ((e = hipHostMalloc((void**)&s.feed, sizeof(HostFeed), hipHostMallocCoherent)) != hipSuccess)
                    return fail_hip(e, "hipHostMalloc(staging)");
                *s.feed = HostFeed{};
            }
        }
        c->in_cap = ni;
        c->out_cap = no;
    }
    return GOOFY_OK;
}

// Copy `rows` rows of `bytes` from src to dst, which are `stride` and `pitch`
// apart.
static void copy_rows(uint8_t* dst, size_t pitch, const uint8_t* src, size_t stride, size_t bytes, size_t rows)
{
    if (stride == bytes && pitch == bytes) std::memcpy(dst, src, bytes * rows);
    else
        for (size_t r = 0; r < rows; ++r) std::memcpy(dst + r * pitch, src + r * stride, bytes);
}

// Marks every part of a launched chunk on the way out: all are marked already
// unless the staging was left by an exception.
struct FeedGuard {
    HostFeed* feed;
    uint64_t call;
    unsigned parts;
    void mark(unsigned p) const { __atomic_store_n(&feed->part[p].staged, call, __ATOMIC_RELEASE); }
    ~FeedGuard()
    {
        for (unsigned p = 0; p < parts; ++p) mark(p);
    }
};

// One launch of a format or pair over an image, or chunk of one, whose rows
// are row_bytes apart: blocks to `out`, a pair's second format to `out2`.
static hipError_t launch_any(int fmt, const LaunchCfg& cfg, const void* in, size_t row_bytes, void* out, void* out2,
                             uint32_t bw, uint32_t nblocks, hipStream_t stream)
{
    return fmt == kFeedDualAlpha
               ? launch_dual_alpha(cfg, in, row_bytes, out, out2, bw, nblocks, stream)
           : fmt == kFeedDual ? launch_dual(cfg, in, row_bytes, out, out2, bw, nblocks, stream)
                              : launch_plain(fmt, cfg, in, row_bytes, out, bw, nblocks, stream);
}

// What the chunks of one image share.
struct HostImage {
    StagingCtx* ctx;
    int fmt;
    LaunchCfg cfg;  // of a plain launch
    unsigned char* result;
    unsigned char* result2;  // a pair's second format, or null
    const unsigned char* input;
    size_t stride, block_bytes;
    uint32_t bw;
    size_t part_bytes;  // about what a part of a chunk holds
    uint64_t patience;
};

// The k-th chunk: `rows` block rows from the y0-th on, of them the `cols` block
// columns from the x0-th on (all of them unless rows is 1), launched as number
// `call` on `stream`; of its groups of kFeedBlocks blocks the first `got` are in
// the caller's memory.  fed: it has a turn.
struct HostChunk {
    uint32_t k = 0, y0 = 0, rows = 0, x0 = 0, cols = 0;
    hipStream_t stream = nullptr;
    uint64_t call = 0;
    uint32_t got = 0;
    bool fed = false;
};

static const StagingCtx::Slot& slot_of(const HostImage& im, const HostChunk& c) { return im.ctx->slot[c.k % kSlots]; }

// Copies blocks [first, last) of a chunk from its slot to the caller, large
// ranges split over the copy pool.
static void collect(const HostImage& im, const HostChunk& c, uint32_t first, uint32_t last)
{
    const uint8_t* const out = slot_of(im, c).out;
    const size_t bb = im.block_bytes;
    const auto copy = [&](uint32_t a, uint32_t b) {
        const size_t to = ((size_t)c.y0 * im.bw + c.x0 + a) * bb, n = (size_t)(b - a) * bb;
        std::memcpy(im.result + to, out + a * bb, n);
        if (im.result2) std::memcpy(im.result2 + to, out + ((size_t)c.cols * c.rows + a) * bb, n);
    };
    constexpr uint32_t kPiece = 8192;  // blocks
    if (last - first < 4u * kPiece) return copy(first, last);
    CopyPool::get().run((int)((last - first + kPiece - 1) / kPiece), [&](int i) {
        const uint32_t a = first + (uint32_t)i * kPiece;
        copy(a, last - a < kPiece ? last : a + kPiece);
    });
}

// Launches a chunk's kernel and stages its rows, in this order if it gets a
// turn.
static hipError_t start_chunk(const HostImage& im, HostChunk& c)
{
    const StagingCtx::Slot& slot = slot_of(im, c);
    const uint32_t nblocks = c.cols * c.rows;
    const size_t row_bytes = (size_t)c.cols * 16, bytes = row_bytes * 4 * c.rows;
    const uint8_t* const rows = im.input + (size_t)c.y0 * 4 * im.stride + (size_t)c.x0 * 16;
    const bool large = bytes >= (2u << 20) && !im.ctx->stage_first;
    c.fed = bytes >= (128u << 10) && !im.ctx->stage_first && im.ctx->take_turn(large ? 1 : 3);
    c.stream = large ? im.ctx->link->stream[c.fed ? 0 : 1] : im.ctx->stream;
    // Parts of whole block rows; where those have more than kWidePart, of
    // blocks in order, so that several threads copy what one row holds and the
    // kernel starts before all of it is staged (us per call, with parts of whole
    // rows / so: 524288x16 1250 / 780, 4194288x8 5900 / 2730).
    const bool wide = row_bytes * 4 > kWidePart;
    const uint32_t want =
        (uint32_t)(wide ? (bytes + kWidePart - 1) / kWidePart
                        : std::max<size_t>(1, std::min<size_t>(kFeedParts, bytes / im.part_bytes)));
    const uint32_t part_blocks = wide ? (nblocks + want - 1) / want : c.cols * ((c.rows + want - 1) / want);
    const uint32_t parts = (nblocks + part_blocks - 1) / part_blocks;
    const auto stage = [&](uint32_t p) {
        uint32_t b = p * part_blocks;
        for (const uint32_t end = std::min(b + part_blocks, nblocks); b < end;) {
            const uint32_t y = b / c.cols, x = b % c.cols;
            // the rest of a block row, or all block rows of the part
            const uint32_t n = wide ? std::min(end - b, c.cols - x) : end - b;
            copy_rows(slot.in + (size_t)y * 4 * row_bytes + (size_t)x * 16, row_bytes,
                      rows + (size_t)y * 4 * im.stride + (size_t)x * 16, im.stride,
                      wide ? (size_t)n * 16 : row_bytes, wide ? 4 : (size_t)n / c.cols * 4);
            b += n;
        }
    };
    // one thread copies an image of 1 MiB at the link's rate, and waking others
    // takes longer (512x512: 38 us with one, 43 with them)
    const auto each_part = [&](auto&& f) {
        if (bytes >= (2u << 20)) CopyPool::get().run((int)parts, [&](int p) { f((uint32_t)p); });
        else
            for (uint32_t p = 0; p < parts; ++p) f(p);
    };
    if (!c.fed) each_part(stage);
    c.call = ++im.ctx->call;
    const hipError_t e =
        launch_fed(im.fmt, slot.in, row_bytes, slot.out, slot.out + nblocks * im.block_bytes, c.cols, nblocks,
                   slot.feed, c.call, c.fed ? part_blocks : 0u, im.patience, c.stream);
    if (e != hipSuccess || !c.fed) return e;
    const FeedGuard guard{slot.feed, c.call, parts};
    each_part([&](uint32_t p) {
        stage(p);
        guard.mark(p);
    });
    return hipSuccess;
}

// Collects the groups of a chunk that are marked, in order.
static bool collect_marked(const HostImage& im, HostChunk& c)
{
    const uint32_t nblocks = c.cols * c.rows, groups = feed_groups(nblocks);
    const HostFeed* const feed = slot_of(im, c).feed;
    uint32_t to = c.got;
    while (to < groups && __atomic_load_n(&feed->done[to], __ATOMIC_ACQUIRE) == c.call) ++to;
    if (to != c.got) collect(im, c, c.got * kFeedBlocks, std::min(to * kFeedBlocks, nblocks));
    c.got = to;
    return c.got == groups;
}

// Waits for a chunk and collects it: by its marks, looking all the time for 2 ms
// and then now and then; or, where its kernel gave up or no mark comes for 200
// ms, by its stream.  Behind other callers' chunks it yields the CPU to the
// threads that copy after 0.1 ms, and sleeps after 1 ms.  1024x1024 from 8 / 12 /
// 16 / 24 threads on 16 CPUs, us per image: 91 / 92 / 87 / 95 with 2 ms of
// looking, 93 / 96 / 93 / 87 so (94 / 94 / 95 / 107 with copy engines); 99th
// percentiles 1.2 / 2.1 / 5.1 / 11 ms, 1.1 / 2.0 / 2.5 / 3.4 so (1.1 / 1.8 / 2.5 /
// 11).  Sleeping from 0.1 ms on takes 7.5 CPUs instead of 11.7 but 99 us per
// image with 12 threads.
static hipError_t finish_chunk(const HostImage& im, HostChunk& c)
{
    using std::chrono::microseconds;
    const StagingCtx::Slot& slot = slot_of(im, c);
    const uint32_t nblocks = c.cols * c.rows;
    const auto gave_up = [&] { return __atomic_load_n(&slot.feed->gave_up, __ATOMIC_ACQUIRE) == c.call; };
    const auto start = std::chrono::steady_clock::now();
    hipError_t e = hipSuccess;
    for (uint32_t look = 1; !collect_marked(im, c); ++look) {
        if (look % 64 != 0) continue;
        const auto waited = std::chrono::steady_clock::now() - start;
        const bool behind = !c.fed && im.ctx->others_have_turns();
        if (waited < microseconds(behind ? 1000 : 2000)) {
            if (behind && waited > microseconds(100)) std::this_thread::yield();
            continue;
        }
        if (gave_up() || waited > microseconds(200000)) {
            e = hipStreamSynchronize(c.stream);
            if (e == hipSuccess && gave_up()) {
                e = launch_any(im.fmt, im.cfg, slot.in, (size_t)c.cols * 16, slot.out,
                               slot.out + nblocks * im.block_bytes, c.cols, nblocks, c.stream);
                if (e == hipSuccess) e = hipStreamSynchronize(c.stream);
            }
            if (e == hipSuccess) collect(im, c, c.got * kFeedBlocks, nblocks);
            break;
        }
        std::this_thread::sleep_for(microseconds(20));
        look = 63;
    }
    if (c.fed) im.ctx->give_turn();
    return e;
}

// fmt: one format into `result`, or kFeedDual: DXT1 into `result` and ETC1S
// into `result2` from one pass over the image, or kFeedDualAlpha: DXT5 and
// ETC2 RGBA8 the same way.
static int compress_host(int fmt, unsigned char* result, const unsigned char* input, unsigned width,
                         unsigned height, unsigned stride, unsigned char* result2 = nullptr,
                         uint64_t patience = kFeedPatience)
{
    clear_error();
    const bool dual_alpha = fmt == kFeedDualAlpha;
    const bool dual = fmt == kFeedDual || dual_alpha;
    if (!format_valid(fmt) && !dual) return fail(GOOFY_ERR_INVALID, "unknown format");
    // Same checks, same order as the reference (GoofyTC/goofy_tc.h:1500-1508).
    if (width % 16 != 0) return fail(GOOFY_ERR_WIDTH, "width must be a multiple of 16");
    if (height % 4 != 0) return fail(GOOFY_ERR_HEIGHT, "height must be a multiple of 4");
    if (width == 0 || height == 0) return GOOFY_OK;
    if (!result || !input || (dual && !result2)) return fail(GOOFY_ERR_INVALID, "null buffer");
    if ((size_t)stride < (size_t)width * 4) return fail(GOOFY_ERR_INVALID, "stride smaller than 4*width");
    const uint32_t bw = width / 4, bh = height / 4;
    const uint32_t max_rows = max_stripe_brows(bw);  // per chunk: chunks are launched one by one
    if (max_rows == 0) return fail(GOOFY_ERR_TOO_LARGE, "image too wide (4,194,304 pixels or more per row)");

    DeviceInfo di;
    int rc = device_info(&di);
    if (rc != GOOFY_OK) return rc;
    StagingCtx* ctx = staging_pool().acquire(di.device);
    struct Release {  // on every path, the kernels are through with the context first
        StagingCtx* c;
        bool done = false;
        ~Release()
        {
            for (hipStream_t s : {c->stream, c->link->stream[0], c->link->stream[1]})
                if (s && !done) (void)hipStreamSynchronize(s);
            c->give_turn();
            staging_pool().release(c);
        }
    } rel{ctx};

    // Chunks of at most 8 MiB, as far as a launch's marks reach: block rows, or,
    // where one has more, pieces of one.
    const size_t row_bytes = (size_t)width * 4, chunk = (size_t)kFeedMarks * kFeedBlocks * 64;
    const unsigned cb = std::min(std::min((unsigned)std::max<size_t>(1, chunk / (row_bytes * 4)), bh), max_rows);
    const uint32_t pieces = (uint32_t)((row_bytes * 4 + chunk - 1) / chunk), cols = (bw + pieces - 1) / pieces;
    // dual: a chunk's staging output holds its blocks of the first format, then
    // those of the second
    const size_t outs = dual ? 2 : 1;
    const size_t bb = dual_alpha ? 16 : (dual ? 8 : block_bytes(fmt));
    if ((rc = ensure_ctx(ctx, (size_t)cols * 64 * cb, outs * cols * cb * bb)) != GOOFY_OK) return rc;
    // Parts of an image of one chunk: 64 KiB, or a thirty-second of it, so that
    // the kernel can start early.  Of larger ones: 1 MiB, copied as streams by
    // the threads; pieces of 256 KiB take 2 to 3 times as long from an image
    // that others have just written (first call on a new 4096x4096 image 2.1-3.4
    // ms, in 1 MiB pieces 1.5) and are 1-2% faster on one that lies in the
    // caches.
    const size_t part_bytes = cb < bh ? (size_t)1 << 20 : (size_t)1 << 16;
    const HostImage im{ctx, fmt, auto_cfg((uint64_t)cols * cb, di.num_cus), result, dual ? result2 : nullptr, input,
                       stride, bb, bw, part_bytes, patience};
    HostChunk ring[kSlots];  // chunks [oldest, k) are launched and not yet collected
    hipError_t e = hipSuccess;
    uint32_t k = 0, oldest = 0;
    for (uint64_t y0 = 0, x0 = 0; y0 < bh && e == hipSuccess; ++k) {
        if (k - oldest == kSlots && (e = finish_chunk(im, ring[oldest++ % kSlots])) != hipSuccess) break;
        ring[k % kSlots] = HostChunk{k, (uint32_t)y0, std::min<uint32_t>(cb, bh - (uint32_t)y0), (uint32_t)x0,
                                     std::min<uint32_t>(cols, bw - (uint32_t)x0)};
        e = start_chunk(im, ring[k % kSlots]);
        if (oldest < k) collect_marked(im, ring[oldest % kSlots]);
        if ((x0 += cols) >= bw) {
            x0 = 0;
            y0 += cb;
        }
    }
    // a marker behind the last kernels while they run, for a caller that goes on
    // to wait for the device
    for (uint32_t i = 0; i < std::min(k, 2u); ++i) (void)hipEventRecord(ctx->ended[i], ring[(k - 1u - i) % kSlots].stream);
    while (e == hipSuccess && oldest < k) e = finish_chunk(im, ring[oldest++ % kSlots]);
    if (e != hipSuccess) return fail_hip(e, "drop-in staging");
    rel.done = true;
    return GOOFY_OK;
}

static int compress_device(int fmt, void* d_result, const void* d_input, unsigned width, unsigned height,
                           size_t pitch, void* stream, const goofy_launch_config* ucfg, void* ev_start = nullptr,
                           void* ev_stop = nullptr)
{
    clear_error();
    if (!format_valid(fmt)) return fail(GOOFY_ERR_INVALID, "unknown format");
    if (width % 4 != 0) return fail(GOOFY_ERR_WIDTH, "width must be a multiple of 4");
    if (height % 4 != 0) return fail(GOOFY_ERR_HEIGHT, "height must be a multiple of 4");
    if (width == 0 || height == 0) return GOOFY_OK;
    if (!d_result || !d_input) return fail(GOOFY_ERR_INVALID, "null buffer");
    if (pitch < (size_t)width * 4 || pitch % 16 != 0)
        return fail(GOOFY_ERR_INVALID, "pitch must be >= 4*width and a multiple of 16");
    const size_t bb = block_bytes(fmt);
    if ((uintptr_t)d_input % 16 != 0 || (uintptr_t)d_result % bb != 0)
        return fail(GOOFY_ERR_INVALID, "input must be 16-byte and result block-size (8 or 16 byte) aligned");
    const uint32_t bw = width / 4, bh = height / 4;
    const uint32_t max_rows = max_stripe_brows(bw);
    if (max_rows == 0) return fail(GOOFY_ERR_TOO_LARGE, "image too wide (4,194,304 pixels or more per row)");
    LaunchCfg cfg{};
    int num_cus = 0;
    if (ucfg) {
        cfg = to_cfg(*ucfg);
        if (!cfg_valid(cfg)) return fail(GOOFY_ERR_INVALID, "invalid launch config");
    } else {
        DeviceInfo di;
        int rc = device_info(&di);
        if (rc != GOOFY_OK) return rc;
        num_cus = di.num_cus;
    }
    // One launch, or horizontal stripes for images beyond one launch's index
    // range; the start event goes with the first launch, the stop event with
    // the last, so the interval covers them all.
    for (uint32_t y0 = 0; y0 < bh;) {
        const uint32_t rows = std::min(max_rows, bh - y0);
        const uint32_t nb = rows * bw;  // <= 0xFFFFFFFF by max_stripe_brows
        const LaunchCfg c = ucfg ? cfg : wide_cfg(nb, num_cus);
        hipError_t e = launch_plain(fmt, c, static_cast<const uint8_t*>(d_input) + (size_t)y0 * 4 * pitch, pitch,
                                    static_cast<uint8_t*>(d_result) + (size_t)y0 * bw * bb, bw, nb,
                                    (hipStream_t)stream, y0 == 0 ? (hipEvent_t)ev_start : nullptr,
                                    y0 + rows == bh ? (hipEvent_t)ev_stop : nullptr);
        if (e != hipSuccess) return fail_hip(e, "encode kernel launch");
        y0 += rows;
    }
    return GOOFY_OK;
}

}  // namespace goofy_impl

using namespace goofy_impl;

extern "C" {

const char* goofy_hip_last_error(void) { return t_last_error.c_str(); }

const char* goofy_hip_status_string(int s)
{
    switch (s) {
    case GOOFY_OK: return "ok";
    case GOOFY_ERR_WIDTH: return "bad width";
    case GOOFY_ERR_HEIGHT: return "bad height";
    case GOOFY_ERR_HIP: return "HIP runtime error";
    case GOOFY_ERR_INVALID: return "invalid argument";
    case GOOFY_ERR_OUT_OF_MEMORY: return "out of memory";
    case GOOFY_ERR_NO_DEVICE: return "no GPU";
    case GOOFY_ERR_TOO_LARGE: return "image too large";
    case GOOFY_ERR_BUSY: return "busy";
    case GOOFY_ERR_CANCELLED: return "cancelled";
    case GOOFY_ERR_DEADLINE: return "deadline passed";
    default: return "unknown status";
    }
}

const char* goofy_hip_version(void) { return "goofy_hip 0.1 (gfx950)"; }

int goofy_hip_device_count(void)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return n;
}

int goofy_hip_compress(int format, unsigned char* result, const unsigned char* input, unsigned int width,
                       unsigned int height, unsigned int stride)
{
    return compress_host(format, result, input, width, height, stride);
}

// goofy_hip_compress with another limit for a fed kernel's wait (10 ns ticks):
// for the test of a host that stages too late.
GOOFY_HIP_API int goofy_impl_compress_with_patience(int format, unsigned char* result, const unsigned char* input,
                                                    unsigned int width, unsigned int height, unsigned int stride,
                                                    uint64_t patience)
{
    return compress_host(format, result, input, width, height, stride, nullptr, patience);
}

int goofy_hip_compress_dxt1(unsigned char* result, const unsigned char* input, unsigned int width, unsigned int height,
                            unsigned int stride)
{
    return compress_host(GOOFY_FORMAT_DXT1, result, input, width, height, stride);
}

int goofy_hip_compress_etc1(unsigned char* result, const unsigned char* input, unsigned int width, unsigned int height,
                            unsigned int stride)
{
    return compress_host(GOOFY_FORMAT_ETC1, result, input, width, height, stride);
}

int goofy_hip_compress_dxt5(unsigned char* result, const unsigned char* input, unsigned int width, unsigned int height,
                            unsigned int stride)
{
    return compress_host(GOOFY_FORMAT_DXT5, result, input, width, height, stride);
}

int goofy_hip_compress_etc2(unsigned char* result, const unsigned char* input, unsigned int width, unsigned int height,
                            unsigned int stride)
{
    return compress_host(GOOFY_FORMAT_ETC2, result, input, width, height, stride);
}

unsigned int goofy_format_block_bytes(int format) { return format_valid(format) ? (unsigned)block_bytes(format) : 0u; }

int goofy_hip_compress_device(int format, void* d_result, const void* d_input, unsigned int width,
                              unsigned int height, size_t pitch, void* stream)
{
    return compress_device(format, d_result, d_input, width, height, pitch, stream, nullptr);
}

int goofy_hip_compress_device_cfg(int format, void* d_result, const void* d_input, unsigned int width,
                                  unsigned int height, size_t pitch, void* stream, const goofy_launch_config* cfg)
{
    return compress_device(format, d_result, d_input, width, height, pitch, stream, cfg);
}

int goofy_hip_compress_device_timed(int format, void* d_result, const void* d_input, unsigned int width,
                                    unsigned int height, size_t pitch, void* stream, const goofy_launch_config* cfg,
                                    void* start_event, void* stop_event)
{
    return compress_device(format, d_result, d_input, width, height, pitch, stream, cfg, start_event, stop_event);
}

int goofy_hip_compress_dual(unsigned char* result_dxt1, unsigned char* result_etc1, const unsigned char* input,
                            unsigned int width, unsigned int height, unsigned int stride)
{
    return compress_host(kFeedDual, result_dxt1, input, width, height, stride, result_etc1);
}

static int compress_device_pair(bool alpha, void* d_a, void* d_b, const void* d_input, unsigned int width,
                                unsigned int height, size_t pitch, void* stream, void* start_event, void* stop_event)
{
    clear_error();
    if (width % 4 != 0) return fail(GOOFY_ERR_WIDTH, "width must be a multiple of 4");
    if (height % 4 != 0) return fail(GOOFY_ERR_HEIGHT, "height must be a multiple of 4");
    if (width == 0 || height == 0) return GOOFY_OK;
    if (!d_a || !d_b || !d_input) return fail(GOOFY_ERR_INVALID, "null buffer");
    if (pitch < (size_t)width * 4 || pitch % 16 != 0)
        return fail(GOOFY_ERR_INVALID, "pitch must be >= 4*width and a multiple of 16");
    const size_t bb = alpha ? 16 : 8;
    if ((uintptr_t)d_input % 16 != 0 || (uintptr_t)d_a % bb != 0 || (uintptr_t)d_b % bb != 0)
        return fail(GOOFY_ERR_INVALID, "input must be 16-byte and results block-size (8 or 16 byte) aligned");
    const uint32_t bw = width / 4, bh = height / 4;
    const uint32_t max_rows = max_stripe_brows(bw);
    if (max_rows == 0) return fail(GOOFY_ERR_TOO_LARGE, "image too wide (4,194,304 pixels or more per row)");
    DeviceInfo di;
    int rc = device_info(&di);
    if (rc != GOOFY_OK) return rc;
    for (uint32_t y0 = 0; y0 < bh;) {  // stripes for images beyond one launch's index range
        const uint32_t rows = std::min(max_rows, bh - y0);
        const uint32_t nb = rows * bw;
        const size_t out_off = (size_t)y0 * bw * bb;
        const uint8_t* in = static_cast<const uint8_t*>(d_input) + (size_t)y0 * 4 * pitch;
        uint8_t* a = static_cast<uint8_t*>(d_a) + out_off;
        uint8_t* b = static_cast<uint8_t*>(d_b) + out_off;
        hipEvent_t e0 = y0 == 0 ? (hipEvent_t)start_event : nullptr;
        hipEvent_t e1 = y0 + rows == bh ? (hipEvent_t)stop_event : nullptr;
        const LaunchCfg c = wide_cfg(nb, di.num_cus);
        hipError_t e = alpha ? launch_dual_alpha(c, in, pitch, a, b, bw, nb, (hipStream_t)stream, e0, e1)
                             : launch_dual(c, in, pitch, a, b, bw, nb, (hipStream_t)stream, e0, e1);
        if (e != hipSuccess) return fail_hip(e, "dual encode kernel launch");
        y0 += rows;
    }
    return GOOFY_OK;
}

int goofy_hip_compress_device_dual(void* d_dxt1, void* d_etc1, const void* d_input, unsigned int width,
                                   unsigned int height, size_t pitch, void* stream, void* start_event,
                                   void* stop_event)
{
    return compress_device_pair(false, d_dxt1, d_etc1, d_input, width, height, pitch, stream, start_event,
                                stop_event);
}

int goofy_hip_compress_device_dual_alpha(void* d_dxt5, void* d_etc2, const void* d_input, unsigned int width,
                                         unsigned int height, size_t pitch, void* stream, void* start_event,
                                         void* stop_event)
{
    return compress_device_pair(true, d_dxt5, d_etc2, d_input, width, height, pitch, stream, start_event,
                                stop_event);
}

int goofy_hip_compress_dual_alpha(unsigned char* result_dxt5, unsigned char* result_etc2, const unsigned char* input,
                                  unsigned int width, unsigned int height, unsigned int stride)
{
    return compress_host(kFeedDualAlpha, result_dxt5, input, width, height, stride, result_etc2);
}

int goofy_hip_tune_device(int format, void* d_result, const void* d_input, unsigned int width, unsigned int height,
                          size_t pitch, void* stream, int reps, goofy_launch_config* best, float* best_ms)
{
    // validates the arguments and warms the device with the default shape
    int rc = compress_device(format, d_result, d_input, width, height, pitch, stream, nullptr);
    if (rc != GOOFY_OK) return rc;
    if (width == 0 || height == 0) return fail(GOOFY_ERR_INVALID, "empty image");
    if (reps < 1) reps = 1;
    hipEvent_t ev[2] = {nullptr, nullptr};
    for (hipEvent_t& x : ev) {
        hipError_t e = hipEventCreate(&x);
        if (e != hipSuccess) {
            for (hipEvent_t y : ev)
                if (y) (void)hipEventDestroy(y);
            return fail_hip(e, "hipEventCreate");
        }
    }
    LaunchCfg top{1, 8, 0, 1, 0};
    float top_ms = 1e30f;
    const int bpls[] = {1, 2, 4}, wgs[] = {1, 2, 4, 8}, orders[] = {0, 1};
    for (int bpl : bpls)
        for (int wg : wgs)
            for (int order : orders) {
                const goofy_launch_config c = to_public(LaunchCfg{bpl, wg, 0, 1, order});
                std::vector<float> ts;
                for (int r = 0; r <= reps && rc == GOOFY_OK; ++r) {  // r == 0: warm-up
                    rc = compress_device(format, d_result, d_input, width, height, pitch, stream, &c, ev[0], ev[1]);
                    hipError_t e = rc == GOOFY_OK ? hipEventSynchronize(ev[1]) : hipSuccess;
                    if (e != hipSuccess) rc = fail_hip(e, "hipEventSynchronize");
                    float ms = 0;
                    if (rc == GOOFY_OK && r > 0 && hipEventElapsedTime(&ms, ev[0], ev[1]) == hipSuccess)
                        ts.push_back(ms);
                }
                if (rc != GOOFY_OK) break;
                if (ts.empty()) continue;
                std::sort(ts.begin(), ts.end());
                if (ts[ts.size() / 2] < top_ms) {
                    top_ms = ts[ts.size() / 2];
                    top = to_cfg(c);
                }
            }
    for (hipEvent_t y : ev) (void)hipEventDestroy(y);
    if (rc != GOOFY_OK) return rc;
    if (best) *best = to_public(top);
    if (best_ms) *best_ms = top_ms;
    return GOOFY_OK;
}

int goofy_synth_fill_host(int kind, uint64_t seed, uint32_t texture_id, uint32_t noise, unsigned char* dst,
                          unsigned int width, unsigned int height, size_t pitch, int threads)
{
    clear_error();
    if (kind < 0 || kind > 2) return fail(GOOFY_ERR_INVALID, "unknown synth kind");
    if (width == 0 || height == 0) return GOOFY_OK;
    if (!dst || pitch < (size_t)width * 4) return fail(GOOFY_ERR_INVALID, "bad destination");
    const goofy_synth::Params P = goofy_synth::make_params((uint32_t)kind, seed, texture_id, noise);
    if (threads <= 0) threads = (int)std::min(16u, std::max(1u, std::thread::hardware_concurrency()));
    threads = (int)std::min<unsigned>((unsigned)threads, height);
    auto rows = [&](unsigned y0, unsigned y1) {
        for (unsigned y = y0; y < y1; ++y) {
            uint32_t* row = reinterpret_cast<uint32_t*>(dst + (size_t)y * pitch);
            for (unsigned x = 0; x < width; ++x) {
                const uint32_t v = goofy_synth::pixel(P, x, y);
                std::memcpy(row + x, &v, 4);
            }
        }
    };
    std::vector<std::thread> pool;
    for (int t = 1; t < threads; ++t)
        pool.emplace_back(rows, (unsigned)((uint64_t)height * t / threads), (unsigned)((uint64_t)height * (t + 1) / threads));
    rows(0, (unsigned)((uint64_t)height / threads));
    for (auto& th : pool) th.join();
    return GOOFY_OK;
}

int goofy_synth_fill_device(int kind, uint64_t seed, uint32_t texture_id, uint32_t noise, void* d_dst,
                            unsigned int width, unsigned int height, size_t pitch, void* stream)
{
    clear_error();
    if (kind < 0 || kind > 2) return fail(GOOFY_ERR_INVALID, "unknown synth kind");
    if (width == 0 || height == 0) return GOOFY_OK;
    if (!d_dst || pitch < (size_t)width * 4 || pitch % 4 != 0 || (uintptr_t)d_dst % 4 != 0)
        return fail(GOOFY_ERR_INVALID, "bad destination");
    if (height > 65535u) return fail(GOOFY_ERR_TOO_LARGE, "height above 65535");
    const goofy_synth::Params P = goofy_synth::make_params((uint32_t)kind, seed, texture_id, noise);
    hipError_t e = launch_synth(&P, d_dst, width, height, pitch, (hipStream_t)stream);
    if (e != hipSuccess) return fail_hip(e, "synth kernel launch");
    return GOOFY_OK;
}

}  // extern "C"

// The drop-in C++ API (include/goofy_tc.h).
namespace goofy {
__attribute__((visibility("default"))) int compressDXT1(unsigned char* result, const unsigned char* input, unsigned int width, unsigned int height,
                 unsigned int stride)
{
    return goofy_impl::compress_host(GOOFY_FORMAT_DXT1, result, input, width, height, stride);
}
__attribute__((visibility("default"))) int compressETC1(unsigned char* result, const unsigned char* input,
                                                        unsigned int width, unsigned int height, unsigned int stride)
{
    return goofy_impl::compress_host(GOOFY_FORMAT_ETC1, result, input, width, height, stride);
}
__attribute__((visibility("default"))) int compressDXT5(unsigned char* result, const unsigned char* input,
                                                        unsigned int width, unsigned int height, unsigned int stride)
{
    return goofy_impl::compress_host(GOOFY_FORMAT_DXT5, result, input, width, height, stride);
}
__attribute__((visibility("default"))) int compressETC2(unsigned char* result, const unsigned char* input,
                                                        unsigned int width, unsigned int height, unsigned int stride)
{
    return goofy_impl::compress_host(GOOFY_FORMAT_ETC2, result, input, width, height, stride);
}
}  // namespace goofy
