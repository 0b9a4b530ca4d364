// batch.cpp -- many textures in one launch.
//
// A plan turns n device-resident textures of uneven sizes into one flattened
// work-list: texture t owns wave tiles [tile_begin(t), tile_begin(t+1)), a
// prefix sum over ceil(blocks(t) / tile).  Tiles never straddle textures, so
// a wave's loads stay contiguous and its format is uniform.  One kernel launch
// walks the whole list (kernels.hip, k_encode_batch), one wave per tile or a
// persistent grid of waves that each take a contiguous run of tiles.  The
// launch shape (blocks per lane, workgroup size, persistent waves per CU,
// streaming hints) comes from an autotuner that times the candidates on the
// plan itself and caches the winner per shape class for the process (and, with
// GOOFY_TUNE_CACHE=<file>, across processes).
//
// The reference has no batching: its driver encodes one image with one
// nested loop (GoofyTC/goofy_tc.h:1514-1524).
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "goofy_hip.h"
#include "internal.h"

using namespace goofy_impl;

// A work-list in device memory: the descriptors and prefix sums of one tile
// size.  Written once, before the first launch that reads it, and freed with
// the plan: launches that still run and graphs that captured one keep reading
// theirs, whatever shape the plan has taken since.
struct Worklist {
    TexDesc* d = nullptr;
    uint32_t ntex = 0, ntiles = 0;
};

struct goofy_batch {
    int device = -1;
    int num_cus = 0;
    std::string arch;
    std::vector<goofy_texture_desc> textures;  // non-empty textures, caller order
    Worklist lists[3];              // for 1, 2 and 4 blocks per lane, each made when first needed
    const Worklist* list = nullptr;  // the one of cfg's tile size
    uint64_t blocks = 0, pixels = 0;
    bool alpha = false;  // holds DXT5 / ETC2 RGBA8 textures
    LaunchCfg cfg{};
    // The launches that the plan's other calls wait for: of each stream the
    // last one, by an event that its own dispatch records.
    struct Launched {
        hipStream_t stream;
        hipEvent_t ended;
        bool pending;
    };
    std::vector<Launched> launched;
    std::mutex launch_mu;  // of `launched`, for launches from several threads
};

namespace {

// Waits for the plan's launches, on whatever stream.
int wait_launched(goofy_batch* b)
{
    std::lock_guard<std::mutex> lock(b->launch_mu);
    for (goofy_batch::Launched& l : b->launched) {
        if (!l.pending) continue;
        const hipError_t e = hipEventSynchronize(l.ended);
        if (e != hipSuccess) return fail_hip(e, "hipEventSynchronize(batch launch)");
        l.pending = false;
    }
    return GOOFY_OK;
}

// The entry for a launch on stream s: the stream's own, whose earlier launches
// end before this one; else one whose launch has ended; else a new one.  The
// per-thread default stream's handle names another stream in each thread, so
// it never has one of its own.  Events are looked at only from the eighth entry
// on: a plan that is launched on a few streams makes no call for them here.
hipError_t launch_entry(goofy_batch* b, hipStream_t s, goofy_batch::Launched** out)
{
    constexpr size_t kLook = 8;
    goofy_batch::Launched* found = nullptr;
    if (s != hipStreamPerThread)
        for (goofy_batch::Launched& l : b->launched)
            if (l.stream == s) found = &l;
    for (size_t i = 0; !found && i < b->launched.size(); ++i)
        if (!b->launched[i].pending) found = &b->launched[i];
    for (size_t i = 0; !found && b->launched.size() >= kLook && i < b->launched.size(); ++i) {
        if (hipEventQuery(b->launched[i].ended) == hipSuccess) found = &b->launched[i];
        else (void)hipGetLastError();
    }
    if (!found) {
        hipEvent_t ev;
        const hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming);
        if (e != hipSuccess) return e;
        b->launched.push_back({s, ev, false});
        found = &b->launched.back();
    } else if (found->stream != s || s == hipStreamPerThread) {
        found->stream = s;
        found->pending = false;
    }
    *out = found;
    return hipSuccess;
}

// Makes the work-list of tiles of `tile` blocks.
int make_worklist(const goofy_batch* b, uint64_t tile, Worklist* out)
{
    std::vector<TexDesc> descs;
    uint64_t tiles = 0;
    for (const goofy_texture_desc& t : b->textures) {
        // one entry per horizontal stripe of at most max_stripe_brows block
        // rows (a single stripe unless the texture is beyond the kernel's
        // index range)
        const uint32_t bw = t.width / 4, bh = t.height / 4, max_rows = max_stripe_brows(bw);
        for (uint32_t y0 = 0; y0 < bh;) {
            const uint32_t rows = std::min(max_rows, bh - y0);
            TexDesc d{};
            d.src = (uint64_t)(uintptr_t)t.src + (uint64_t)y0 * 4 * t.pitch;
            d.dst = (uint64_t)(uintptr_t)t.dst + (uint64_t)y0 * bw * block_bytes(t.format);
            d.pitch = t.pitch;
            d.bw = bw;
            d.nblocks = rows * bw;
            d.magic = div_magic(bw);
            d.fmt = (uint32_t)t.format;
            d.tile_begin = (uint32_t)tiles;
            tiles += (d.nblocks + tile - 1) / tile;
            if (tiles > 0xFFFFFFFFull / tile) return fail(GOOFY_ERR_TOO_LARGE, "batch has too many tiles");
            descs.push_back(d);
            y0 += rows;
        }
    }
    const size_t ntex = descs.size();
    std::vector<uint8_t> host(worklist_bytes(ntex));
    if (ntex) std::memcpy(host.data(), descs.data(), ntex * sizeof(TexDesc));
    uint32_t* tb = worklist_tile_begin(reinterpret_cast<TexDesc*>(host.data()), ntex);
    for (size_t i = 0; i < ntex; ++i) tb[i] = descs[i].tile_begin;
    tb[ntex] = (uint32_t)tiles;
    TexDesc* d = nullptr;
    hipError_t e = hipMalloc((void**)&d, host.size());
    if (e != hipSuccess) return fail_hip(e, "hipMalloc(descriptors)");
    e = hipMemcpy(d, host.data(), host.size(), hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        (void)hipFree(d);
        return fail_hip(e, "hipMemcpy(work-list)");
    }
    *out = Worklist{d, (uint32_t)ntex, (uint32_t)tiles};
    return GOOFY_OK;
}

// Gives the plan the shape c and the work-list of its tile size; on an error
// the plan keeps the shape it has.
int set_shape(goofy_batch* b, const LaunchCfg& c)
{
    Worklist& l = b->lists[__builtin_ctz((unsigned)c.blocks_per_lane)];
    if (!l.d) {
        const int rc = make_worklist(b, (uint64_t)tile_blocks(c), &l);
        if (rc != GOOFY_OK) return rc;
    }
    b->cfg = c;
    b->list = &l;
    return GOOFY_OK;
}

hipError_t launch(const goofy_batch* b, hipStream_t s, hipEvent_t done)
{
    return launch_batch(b->cfg, b->list->d, b->list->ntex, b->list->ntiles, b->num_cus, s, b->alpha, done);
}

// ---- tuning cache ---------------------------------------------------------------

using Key = std::tuple<std::string, int, int, int>;  // arch, log2(blocks), log2(blocks/texture), %DXT1 / 10

std::mutex g_tune_mu;
std::map<Key, LaunchCfg>& tune_cache()
{
    static auto* m = new std::map<Key, LaunchCfg>();
    return *m;
}

Key shape_key(const goofy_batch* b)
{
    uint64_t dxt = 0, alpha = 0;
    for (const auto& t : b->textures) {
        dxt += t.format == GOOFY_FORMAT_DXT1;
        alpha += t.format >= GOOFY_FORMAT_DXT5;
    }
    const int n = (int)std::max<size_t>(1, b->textures.size());
    const int lb = (int)std::log2((double)std::max<uint64_t>(1, b->blocks));
    const int lpt = (int)std::log2((double)std::max<uint64_t>(1, b->blocks / (uint64_t)n));
    // share mix: tenths of DXT1 textures, plus 11 x tenths of alpha textures
    return Key{b->arch, lb, lpt, (int)(dxt * 10 / (uint64_t)n + 11 * (alpha * 10 / (uint64_t)n))};
}

// First line of the tuning file.  The number goes up whenever a field of a shape
// comes to mean something else, or the kernels change so that times of earlier
// builds no longer rank the shapes: files of another number (and those of 1,
// which had no such line) are not used, and written anew by the next autotune.
constexpr int kTuneVersion = 2;  // 2: tile_order 1 is runs of tiles per XCD, no longer eighths

void load_file_cache()
{
    static bool loaded = false;
    if (loaded) return;
    loaded = true;
    const char* path = std::getenv("GOOFY_TUNE_CACHE");
    if (!path) return;
    FILE* f = std::fopen(path, "r");
    if (!f) return;
    int version = 0;
    if (std::fscanf(f, "goofy-tune %d", &version) != 1 || version != kTuneVersion) {
        std::fclose(f);
        return;
    }
    char arch[64];
    int lb, lpt, mix, bpl, wg, wpc, nt, order;
    while (std::fscanf(f, "%63s %d %d %d %d %d %d %d %d", arch, &lb, &lpt, &mix, &bpl, &wg, &wpc, &nt, &order) == 9) {
        LaunchCfg c{bpl, wg, wpc, nt, order};
        if (cfg_valid(c)) tune_cache()[Key{arch, lb, lpt, mix}] = c;
    }
    std::fclose(f);
}

void save_file_cache()
{
    const char* path = std::getenv("GOOFY_TUNE_CACHE");
    if (!path) return;
    FILE* f = std::fopen(path, "w");
    if (!f) return;
    std::fprintf(f, "goofy-tune %d\n", kTuneVersion);
    for (const auto& kv : tune_cache()) {
        const LaunchCfg& c = kv.second;
        std::fprintf(f, "%s %d %d %d %d %d %d %d %d\n", std::get<0>(kv.first).c_str(), std::get<1>(kv.first),
                     std::get<2>(kv.first), std::get<3>(kv.first), c.blocks_per_lane, c.wg_waves, c.waves_per_cu,
                     c.nontemporal, c.tile_order);
    }
    std::fclose(f);
}

int check_texture(const goofy_texture_desc& t, size_t i)
{
    char where[64];
    std::snprintf(where, sizeof where, "texture %zu: ", i);
    if (!format_valid(t.format)) return fail(GOOFY_ERR_INVALID, std::string(where) + "unknown format");
    if (t.width % 4 != 0) return fail(GOOFY_ERR_WIDTH, std::string(where) + "width must be a multiple of 4");
    if (t.height % 4 != 0) return fail(GOOFY_ERR_HEIGHT, std::string(where) + "height must be a multiple of 4");
    if (t.width == 0 || t.height == 0) return GOOFY_OK;
    if (!t.src || !t.dst) return fail(GOOFY_ERR_INVALID, std::string(where) + "null buffer");
    if (t.pitch < (size_t)t.width * 4 || t.pitch % 16 != 0)
        return fail(GOOFY_ERR_INVALID, std::string(where) + "pitch must be >= 4*width and a multiple of 16");
    if ((uintptr_t)t.src % 16 != 0 || (uintptr_t)t.dst % block_bytes(t.format) != 0)
        return fail(GOOFY_ERR_INVALID, std::string(where) + "src must be 16-byte and dst block-size aligned");
    if (max_stripe_brows(t.width / 4) == 0)  // larger textures become several work-list entries
        return fail(GOOFY_ERR_TOO_LARGE, std::string(where) + "too wide (4,194,304 pixels or more per row)");
    return GOOFY_OK;
}

}  // namespace

extern "C" {

int goofy_batch_create(const goofy_texture_desc* textures, size_t count, const goofy_launch_config* ucfg,
                       goofy_batch** out)
{
    clear_error();
    if (!out || (count && !textures)) return fail(GOOFY_ERR_INVALID, "null argument");
    *out = nullptr;
    for (size_t i = 0; i < count; ++i) {
        const int rc = check_texture(textures[i], i);
        if (rc != GOOFY_OK) return rc;
    }
    DeviceInfo di;
    int rc = device_info(&di);
    if (rc != GOOFY_OK) return rc;
    goofy_batch* b = new goofy_batch();
    b->device = di.device;
    b->num_cus = di.num_cus;
    b->arch = di.arch;
    for (size_t i = 0; i < count; ++i) {
        const goofy_texture_desc& t = textures[i];
        if (t.width == 0 || t.height == 0) continue;
        b->textures.push_back(t);
        b->alpha |= t.format >= GOOFY_FORMAT_DXT5;
        b->blocks += (uint64_t)(t.width / 4) * (t.height / 4);
        b->pixels += (uint64_t)t.width * t.height;
    }
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        load_file_cache();
        auto it = tune_cache().find(shape_key(b));
        b->cfg = it != tune_cache().end() ? it->second : wide_cfg(b->blocks, b->num_cus);
    }
    if (ucfg) {
        LaunchCfg c = to_cfg(*ucfg);
        if (!cfg_valid(c)) {
            delete b;
            return fail(GOOFY_ERR_INVALID, "invalid launch config");
        }
        b->cfg = c;
    }
    rc = set_shape(b, b->cfg);
    if (rc != GOOFY_OK) {
        goofy_batch_destroy(b);
        return rc;
    }
    *out = b;
    return GOOFY_OK;
}

int goofy_batch_launch(goofy_batch* b, void* stream)
{
    clear_error();
    if (!b) return fail(GOOFY_ERR_INVALID, "null batch");
    if (b->list->ntiles == 0) return GOOFY_OK;
    const hipStream_t s = (hipStream_t)stream;
    // One kernel: a plain launch.  A hipGraph of this one node cost the host
    // 15-17 us a launch on MI355X (4 ms the first time), the kernel launch
    // 2.8 us, and an event recorded behind it 5 us more than one that the
    // kernel's own dispatch records.  A stream that is being captured takes
    // the launch as a node, without the event.
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess) (void)hipGetLastError();  // the launch says why
    hipError_t e;
    if (cap != hipStreamCaptureStatusNone) {
        e = launch(b, s, nullptr);
    } else {
        std::lock_guard<std::mutex> lock(b->launch_mu);
        goofy_batch::Launched* l = nullptr;
        if ((e = launch_entry(b, s, &l)) != hipSuccess) return fail_hip(e, "hipEventCreate");
        e = launch(b, s, l->ended);
        if (e == hipSuccess) l->pending = true;
    }
    return e == hipSuccess ? GOOFY_OK : fail_hip(e, "batch kernel launch");
}

int goofy_batch_launch_per_texture(goofy_batch* b, void* stream)
{
    clear_error();
    if (!b) return fail(GOOFY_ERR_INVALID, "null batch");
    for (const goofy_texture_desc& t : b->textures) {
        // horizontal stripes of at most max_stripe_brows block rows, as in
        // the work-list: beyond that a launch's block index or its division
        // magic would be out of range
        const uint32_t bw = t.width / 4, bh = t.height / 4, max_rows = max_stripe_brows(bw);
        for (uint32_t y0 = 0; y0 < bh;) {
            const uint32_t rows = std::min(max_rows, bh - y0);
            const uint32_t nb = rows * bw;
            const LaunchCfg c = wide_cfg(nb, b->num_cus);
            hipError_t e = launch_plain(t.format, c, static_cast<const uint8_t*>(t.src) + (size_t)y0 * 4 * t.pitch,
                                        t.pitch, static_cast<uint8_t*>(t.dst) + (size_t)y0 * bw * block_bytes(t.format),
                                        bw, nb, (hipStream_t)stream);
            if (e != hipSuccess) return fail_hip(e, "per-texture launch");
            y0 += rows;
        }
    }
    return GOOFY_OK;
}

int goofy_batch_get_config(const goofy_batch* b, goofy_launch_config* cfg)
{
    clear_error();
    if (!b || !cfg) return fail(GOOFY_ERR_INVALID, "null argument");
    *cfg = to_public(b->cfg);
    return GOOFY_OK;
}

int goofy_batch_set_config(goofy_batch* b, const goofy_launch_config* cfg)
{
    clear_error();
    if (!b || !cfg) return fail(GOOFY_ERR_INVALID, "null argument");
    LaunchCfg c = to_cfg(*cfg);
    if (!cfg_valid(c)) return fail(GOOFY_ERR_INVALID, "invalid launch config");
    const int rc = wait_launched(b);
    return rc != GOOFY_OK ? rc : set_shape(b, c);
}

int goofy_batch_autotune(goofy_batch* b, void* stream, int reps, goofy_launch_config* chosen, float* best_ms)
{
    clear_error();
    if (!b) return fail(GOOFY_ERR_INVALID, "null batch");
    int rc = wait_launched(b);
    if (rc != GOOFY_OK) return rc;
    if (reps < 1) reps = 1;
    hipStream_t s = (hipStream_t)stream;
    hipEvent_t e0, e1;
    hipError_t e = hipEventCreate(&e0);
    if (e != hipSuccess) return fail_hip(e, "hipEventCreate");
    e = hipEventCreate(&e1);
    if (e != hipSuccess) {
        (void)hipEventDestroy(e0);
        return fail_hip(e, "hipEventCreate");
    }
    const LaunchCfg start = b->cfg;
    LaunchCfg best = b->cfg;
    float best_t = 1e30f;
    const int bpls[] = {1, 2, 4}, wgs[] = {2, 4, 8}, wpcs[] = {0, 8, 16, 32}, nts[] = {0, 1}, orders[] = {0, 1};
    for (int bpl : bpls)
        for (int wg : wgs)
            for (int wpc : wpcs)
                for (int nt : nts)
                    for (int order : orders) {
                        if ((rc = set_shape(b, LaunchCfg{bpl, wg, wpc, nt, order})) != GOOFY_OK) goto done;
                        // one warm-up launch, then the median of `reps` timed ones
                        e = launch(b, s, nullptr);
                        if (e != hipSuccess) { rc = fail_hip(e, "autotune launch"); goto done; }
                        std::vector<float> ts;
                        for (int r = 0; r < reps; ++r) {
                            (void)hipEventRecord(e0, s);
                            e = launch(b, s, nullptr);
                            (void)hipEventRecord(e1, s);
                            if (e != hipSuccess) { rc = fail_hip(e, "autotune launch"); goto done; }
                            e = hipEventSynchronize(e1);
                            if (e != hipSuccess) { rc = fail_hip(e, "hipEventSynchronize"); goto done; }
                            float ms = 0;
                            (void)hipEventElapsedTime(&ms, e0, e1);
                            ts.push_back(ms);
                        }
                        std::sort(ts.begin(), ts.end());
                        const float med = ts[ts.size() / 2];
                        if (med < best_t) {
                            best_t = med;
                            best = b->cfg;
                        }
                    }
done:
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)set_shape(b, rc == GOOFY_OK ? best : start);  // both have their lists
    if (rc != GOOFY_OK) return rc;
    {
        std::lock_guard<std::mutex> lock(g_tune_mu);
        tune_cache()[shape_key(b)] = best;
        save_file_cache();
    }
    if (chosen) *chosen = to_public(best);
    if (best_ms) *best_ms = best_t;
    return GOOFY_OK;
}

int goofy_batch_info(const goofy_batch* b, uint64_t* textures, uint64_t* blocks, uint64_t* tiles, uint64_t* pixels)
{
    clear_error();
    if (!b) return fail(GOOFY_ERR_INVALID, "null batch");
    if (textures) *textures = b->textures.size();
    if (blocks) *blocks = b->blocks;
    if (tiles) *tiles = b->list->ntiles;
    if (pixels) *pixels = b->pixels;
    return GOOFY_OK;
}

int goofy_batch_destroy(goofy_batch* b)
{
    clear_error();
    if (!b) return GOOFY_OK;
    (void)wait_launched(b);
    for (const goofy_batch::Launched& l : b->launched) (void)hipEventDestroy(l.ended);
    for (const Worklist& l : b->lists)
        if (l.d) (void)hipFree(l.d);
    delete b;
    return GOOFY_OK;
}

}  // extern "C"
