// internal.h -- declarations shared by the host-side translation units of
// libgoofy_hip.so (not installed; the public C-ABI is include/goofy_hip.h).
#pragma once

#include <hip/hip_runtime_api.h>
#include <stddef.h>
#include <stdint.h>

#include <string>

#include "goofy_hip.h"

namespace goofy_impl {

// Device-side texture descriptor of the flattened work-list (64 bytes).
// Texture t owns wave tiles [tile_begin, tile_begin + ceil(nblocks / tile)).
struct TexDesc {
    uint64_t src;      // device address of pixel (0,0)
    uint64_t dst;      // device address of block 0 (8 bytes per block, row-major)
    uint64_t pitch;    // bytes between pixel rows
    uint64_t magic;    // ceil(2^40 / bw): block row = (i * magic) >> 40
    uint32_t bw;       // blocks per row
    uint32_t nblocks;  // bw * bh
    uint32_t tile_begin;  // also in the work-list's prefix-sum array
    uint32_t fmt;         // GOOFY_FORMAT_DXT1 / GOOFY_FORMAT_ETC1
    uint32_t pad[4];
};
static_assert(sizeof(TexDesc) == 64, "TexDesc layout");

// Kernel launch configuration (what the autotuner searches).
struct LaunchCfg {
    int blocks_per_lane;  // 1, 2 or 4 blocks per lane (tile = 64 * bpl blocks per wave)
    int wg_waves;         // waves per workgroup: 1, 2, 4 or 8
    int waves_per_cu;     // persistent grid size (0 = one wave per tile, no persistence)
    int nontemporal;      // 1 = streaming (non-temporal) loads and stores
    int tile_order;       // 0 = linear, 1 = runs of kXcdRunTiles tiles per XCD
};

// The dispatcher hands workgroup b to XCD b % 8.  With tile_order 1, kernels
// renumber workgroups so that each XCD takes runs of 128 waves' work (a run is
// 512 KiB of pixels with one block per lane; xcd_workgroup in tile_io.h).
// Runs of 64 to 512 waves measured alike on batches of 128 to 4096 textures;
// one run per XCD (a contiguous eighth each) was 3-4% slower than them on 4096
// textures and 12% on 512, whose XCDs then end at different times.
constexpr uint32_t kXcdCount = 8;
constexpr uint32_t kXcdRunTiles = 128;
// The kernels' order argument: 0, or 1 + log2 of the run in workgroups.
inline uint32_t order_arg(const LaunchCfg& c)
{
    return c.tile_order ? 1u + (uint32_t)__builtin_ctz(kXcdRunTiles / (uint32_t)c.wg_waves) : 0u;
}

// The one-image kernels' shape argument: that, and the waves per workgroup from bit 8 up.
inline uint32_t shape_arg(const LaunchCfg& c) { return order_arg(c) | (uint32_t)c.wg_waves << 8; }

inline LaunchCfg to_cfg(const goofy_launch_config& u)
{
    return LaunchCfg{u.blocks_per_lane, u.wg_waves, u.waves_per_cu, u.nontemporal, u.tile_order};
}
inline goofy_launch_config to_public(const LaunchCfg& c)
{
    return goofy_launch_config{c.blocks_per_lane, c.wg_waves, c.waves_per_cu, c.nontemporal, c.tile_order};
}

// A small work-list passed by value in the kernel arguments (no copy to the
// device before the launch): up to kInlineTextures descriptors and their
// ntex+1 tile prefix sums.
constexpr int kInlineTextures = 16;
struct InlineWorklist {
    TexDesc d[kInlineTextures];
    uint32_t tile_begin[kInlineTextures + 1];
};

// A batch work-list in device memory: ntex descriptors followed by the
// ntex+1 prefix sums of their tile counts (uint32, last = total tiles).
inline size_t worklist_bytes(size_t ntex) { return ntex * sizeof(TexDesc) + (ntex + 1) * sizeof(uint32_t); }
inline uint32_t* worklist_tile_begin(TexDesc* descs, size_t ntex) { return reinterpret_cast<uint32_t*>(descs + ntex); }
inline const uint32_t* worklist_tile_begin(const TexDesc* descs, size_t ntex)
{
    return reinterpret_cast<const uint32_t*>(descs + ntex);
}

inline bool format_valid(int f) { return f >= GOOFY_FORMAT_DXT1 && f <= GOOFY_FORMAT_ETC2; }
// Bytes per block: 8 (DXT1, ETC1S) or 16 (DXT5, ETC2 RGBA8).
inline size_t block_bytes(int f) { return f >= GOOFY_FORMAT_DXT5 ? 16u : 8u; }

inline uint64_t div_magic(uint32_t bw) { return ((1ull << 40) + bw - 1) / bw; }

// True when (i * magic) >> 40 == i / bw for every i < nblocks.
inline bool magic_ok(uint64_t bw, uint64_t nblocks) { return bw > 0 && nblocks * bw < (1ull << 40) && nblocks / bw < (1ull << 24); }

// Most block rows one launch (or one work-list entry) may cover for an image
// bw blocks wide: block indices below 2^32 and an exact division magic
// (magic_ok).  Larger images are encoded as horizontal stripes of at most
// this many block rows; blocks are independent, so stripes change nothing in
// the output.  0 when a single block row is already beyond the range
// (bw >= 2^20, i.e. 4,194,304 pixels or more per row).
inline uint32_t max_stripe_brows(uint64_t bw)
{
    if (bw == 0 || bw >= (1ull << 20)) return 0;
    uint64_t r = ((1ull << 40) - 1) / (bw * bw);
    if (r > 0xFFFFFFFFull / bw) r = 0xFFFFFFFFull / bw;
    if (r > (1ull << 24) - 1) r = (1ull << 24) - 1;
    return (uint32_t)r;
}

// Kernel launchers (kernels.hip).
hipError_t launch_plain(int fmt, const LaunchCfg& cfg, const void* src, size_t pitch, void* dst, uint32_t bw,
                        uint32_t nblocks, hipStream_t stream, hipEvent_t start = nullptr, hipEvent_t stop = nullptr);
// cfg: workgroup size and tile order (one block per lane, streaming).
hipError_t launch_dual(const LaunchCfg& cfg, const void* src, size_t pitch, void* dst_dxt1, void* dst_etc1, uint32_t bw,
                       uint32_t nblocks, hipStream_t stream, hipEvent_t start = nullptr, hipEvent_t stop = nullptr);
hipError_t launch_dual_alpha(const LaunchCfg& cfg, const void* src, size_t pitch, void* dst_dxt5, void* dst_etc2,
                             uint32_t bw, uint32_t nblocks, hipStream_t stream, hipEvent_t start = nullptr,
                             hipEvent_t stop = nullptr);
// The drop-in's kernel, which encodes an image in pinned host memory while
// the host is still staging it there.  HostFeed (pinned, coherent): the word
// of a part holds the number of the call whose rows are staged in it, written
// after them; gave_up the number of a call whose kernel stopped waiting; done,
// of each group of kFeedBlocks blocks up to kFeedMarks (8 MiB of pixels), the
// number of the last call whose blocks of it are in host memory.
constexpr uint32_t kFeedParts = 32;
constexpr uint32_t kFeedGroups = 24;
constexpr uint32_t kFeedBlocks = 512;
constexpr uint32_t kFeedMarks = 256;
inline uint32_t feed_groups(uint32_t nblocks) { return nblocks / kFeedBlocks + (nblocks % kFeedBlocks != 0); }
struct HostFeed {
    struct alignas(64) Part {
        uint64_t staged;
    } part[kFeedParts];
    alignas(64) uint64_t gave_up;
    alignas(64) uint64_t done[kFeedMarks];
};
// Pseudo-formats: both 8-byte formats / both 16-byte formats, the second into
// dst2.
constexpr int kFeedDual = 1 << 16, kFeedDualAlpha = (1 << 16) + 1;
// part_blocks: blocks per part (at most kFeedParts parts), or 0 where all rows
// are staged before the launch; call: a number that
// no word holds yet; patience: how long a wait may last, in 10 ns ticks.
hipError_t launch_fed(int fmt, const void* src, size_t pitch, void* dst, void* dst2, uint32_t bw, uint32_t nblocks,
                      HostFeed* feed, uint64_t call, uint32_t part_blocks, uint64_t patience, hipStream_t stream);
// alpha: the work-list holds DXT5 / ETC2 RGBA8 textures too (the kernel
// instance with all four formats; without, DXT1 / ETC1S only).
hipError_t launch_batch(const LaunchCfg& cfg, const TexDesc* d_descs, uint32_t ntex, uint32_t ntiles, int num_cus,
                        hipStream_t stream, bool alpha = false);
// The same with an event that the kernel's own dispatch records (or null).
hipError_t launch_batch(const LaunchCfg& cfg, const TexDesc* d_descs, uint32_t ntex, uint32_t ntiles, int num_cus,
                        hipStream_t stream, bool alpha, hipEvent_t done);
hipError_t launch_batch_inline(const LaunchCfg& cfg, const InlineWorklist& wl, uint32_t ntex, uint32_t ntiles,
                               int num_cus, hipStream_t stream, bool alpha = false);
hipError_t launch_synth(const void* params, void* dst, uint32_t width, uint32_t height, size_t pitch,
                        hipStream_t stream);
hipError_t launch_decode(int fmt, const void* blocks, void* dst, uint32_t width, uint32_t height, size_t pitch,
                         hipStream_t stream);
// Cache policies of the decoders' stores: streaming, streaming written through
// (sc0 sc1 nt), and cached.
constexpr int kStream = 2, kStreamThrough = 19, kCached = 0;

// How a decode stores depends on how what its waves write (the pixels of 64
// blocks in order) lies on the 64-byte sectors.
//   Rows on sectors, of whole groups of 4 blocks: every wave begins and ends on a
// sector, every store fills whole ones, and writing them through is fastest.
// Otherwise neighbouring waves share a sector at their ends, which their XCD's
// L2 has to bring together, so runs of workgroups per XCD and no writing
// through; cached stores keep more of them together, but only images too large
// to lie in the last-level cache gain by that.  Measured in us
// (BC1 / ETC2 RGBA8), streaming in linear order -> as chosen here: 2048^2
// 5.2 / 5.7 -> 4.2 / 4.5, 4096^2 13.8 / 15.7 -> 12.2 / 14.9, 8192^2 47.2 / 53.9
// -> 45.8 / 52.9, with a pitch of 32896 55.3 / 59.7 -> 46.6 / 53.2; rows off the
// sectors 3076^2 10.3 / 11.3 -> 9.8 / 10.9, 6004^2 36.9 / 35.9 -> 31.9 / 34.4,
// 8196x8192 64.9 / 62.2 -> 54.4 / 57.8.  Cached against streaming there, both in
// runs: 3076^2 10.1 / 11.7 and 9.8 / 10.9, 4100^2 14.6 / 17.2 and 15.3 / 17.1,
// 6004^2 31.9 / 34.6 and 34.6 / 34.4, 7004^2 42.5 / 43.9 and 47.7 / 45.5; written
// through at 8196x8192 61.4 / 67.6.  Rows on sectors with a width that is no
// multiple of 16 pixels, streaming in linear order / written through / as chosen
// here: 2052^2 5.5 5.9 / 5.9 6.3 / 5.0 5.5, 3076^2 10.2 11.3 / 11.2 11.4 / 9.6
// 10.6, 4100^2 16.6 18.1 / 17.3 18.1 / 14.3 16.7, 6004^2 36.7 36.0 / 35.2 37.5 /
// 33.0 33.9, 8196x8192 64.5 62.3 / 60.7 66.2 / 56.2 58.9.
inline int decode_store(int fmt, uint32_t bw, const void* dst, size_t pitch, uint32_t height)
{
    if (pitch % 64 == 0 && (uintptr_t)dst % 64 == 0 && bw % 4 == 0) return kStreamThrough;
    const size_t large = fmt < 2 ? (size_t)64 << 20 : (size_t)160 << 20;
    return pitch * height >= large ? kCached : kStream;
}

// Quality sums: squared errors of bytes 0..3, then the sum of squared luma
// differences times 10^4 (an exact integer with the harness's weights).
struct QualitySums {
    unsigned long long sum[5];
};
// The same sums as a pooled call's kernel passes them on: six words, the luma
// sum in two (its low and high 32 bits, each summed by itself), every word
// with a count of its contributions above kQualityCountBit.  A launch's sums
// stay below that bit: at most 2^33.6 pixels (kQualityMaxLaunchUnits blocks)
// of 255^2 < 2^16, and 1536 low words below 2^32.
constexpr uint32_t kQualityWords = 6;
constexpr uint32_t kQualityCountBit = 52;
// Device work area of a pooled call, all zero between launches: the
// workgroups' words spread over the slots (a line each), and their total.
constexpr uint32_t kQualitySlots = 64;
struct QualityAccum {
    struct alignas(64) Line {
        unsigned long long word[kQualityWords];
    } slot[kQualitySlots], total;
};
// Pinned host memory: the words of one launch, without counts.
struct QualityHost {
    uint64_t word[kQualityWords];
};
// A word that no launch has written yet (counts and sums stay below it).
constexpr uint64_t kQualityNone = ~0ull;
// A pooled call waits after this many stripes, each with a QualityHost.
constexpr uint32_t kQualityStripes = 16;
// Where a quality launch leaves its sums.  Pooled: the zeroed accum on the way
// and *host (pinned) in the end.  Allocation-free (host null): work has the
// final sums at offset 0 and one partial per workgroup from
// kQualityPartialsOffset on; every partial the final kernel reads is written
// by the launch before it, and the first stripe replaces the sums, so that
// area needs no clearing between calls.
struct QualityDest {
    QualityAccum* accum;
    QualityHost* host;
    void* work;
};
constexpr size_t kQualityPartialsOffset = 64;
constexpr uint32_t kQualityMaxGroups = 1536;
inline uint32_t quality_grid(uint64_t units)
{
    const uint64_t g = (units + 255u) / 256u;
    return (uint32_t)(g < 1 ? 1 : (g > kQualityMaxGroups ? kQualityMaxGroups : g));
}
inline size_t quality_scratch_bytes(uint64_t units)
{
    return kQualityPartialsOffset + (size_t)quality_grid(units) * sizeof(QualitySums);
}
// A quality lane adds at most kQualityLaneUnits blocks (or 4-pixel quads) in
// 32-bit sums, so one launch covers at most this many units; the callers
// launch larger images as stripes of quality_stripe_rows(units per row) rows.
constexpr uint64_t kQualityLaneUnits = 2048;
constexpr uint64_t kQualityMaxLaunchUnits = kQualityLaneUnits * kQualityMaxGroups * 256u;
inline uint32_t quality_stripe_rows(uint64_t units_per_row)
{
    const uint64_t r = max_stripe_brows(units_per_row), cap = kQualityMaxLaunchUnits / (units_per_row ? units_per_row : 1);
    return (uint32_t)(r < cap ? r : cap);
}
// accumulate (allocation-free): add onto the sums already at offset 0 of the
// work area (later stripes of one image on the same stream).
hipError_t launch_sqerr(int fmt, const void* blocks, const void* src, size_t pitch, uint32_t width, uint32_t height,
                        const QualityDest& dest, bool accumulate, hipStream_t stream);
hipError_t launch_sqerr_images(const void* a, size_t pitch_a, const void* b, size_t pitch_b, uint32_t width,
                               uint32_t height, const QualityDest& dest, hipStream_t stream);
// Size of the allocation-free call's fixed device array (kQualityMaxGroups
// partials).
constexpr size_t kQualityNoAllocBytes = kQualityPartialsOffset + (size_t)kQualityMaxGroups * sizeof(QualitySums);
// Device address of `device`'s copy of that array (the current device of the
// calling thread), looked up once per device and kept.
hipError_t noalloc_scratch_address(int device, void** addr);
// getMsePsnr's figures (Src/main.cpp:403-469) from the integer sums.
void quality_figures(const QualitySums& sums, uint64_t pixels, goofy_quality* out);
hipError_t launch_rgb565_baseline(const void* src, size_t src_pitch, void* dst, size_t dst_pitch, uint32_t width,
                                  uint32_t height, hipStream_t stream, hipEvent_t start = nullptr,
                                  hipEvent_t stop = nullptr);

// Error reporting: every C-ABI function stores a message for its thread.
int fail(int code, const std::string& msg);
int fail_hip(hipError_t e, const char* what);
void clear_error();

// Device properties cached per device.
struct DeviceInfo {
    int device = -1;
    int num_cus = 0;
    size_t total_mem = 0;
    char arch[64] = {0};
};
int device_info(DeviceInfo* out);  // current device; returns GOOFY_OK or an error code

inline int tile_blocks(const LaunchCfg& c) { return 64 * c.blocks_per_lane; }
// Default launch shape for a launch of `blocks` 4x4 blocks on a device with
// num_cus compute units (used wherever the caller gives no shape).
LaunchCfg auto_cfg(uint64_t blocks, int num_cus);
// The default of every encode launch on device memory.  Above 32 MiB of
// pixels (8192 tiles), where loads bound the kernel, tiles go to the XCDs in
// runs, in workgroups of 4 waves, or 8 from 1 GiB on; smaller launches keep
// auto_cfg's shape.  Measured in us per launch, linear order in 8-wave
// workgroups -> runs in 4-wave ones, per format (DXT1, ETC1S, DXT5, ETC2) and
// pair (DXT1 + ETC1S, DXT5 + ETC2):
//   3400^2        9.4   9.5  10.7  11.5  10.3  15.0 ->   8.8   8.8  10.3  11.2  10.1  14.3
//   4096^2       12.9  13.1  14.2  15.0  14.8  19.1 ->  12.3  12.4  14.1  14.9  14.2  18.9
//   8192^2       48.9  49.1  53.4  54.2  54.7  65.8 ->  46.0  46.0  51.5  54.1  52.3  65.5
//   12004x9000   80.0  80.3  86.4  90.2   -   108.2 ->  75.5  74.8  82.6  87.5  85.4 105.2
//   16384^2     192.3 192.2 209.8 209.4   -   246.1 -> 187.2 184.9 206.5 212.2 208.0 245.9
// and batches: 16 textures of 8.7k tiles 9.8 -> 8.9, 256 of 11.5k 10.8 -> 10.2,
// 1024 282 -> 262, 4096 1090 -> 1006.  Below, 3000x2052 (6011 tiles) loses 2%.
// From 262144 tiles 4 and 8 waves are alike on images; a 2048-texture batch of
// 660k tiles took 478 us in 8-wave workgroups and 490 in 4-wave ones.
inline LaunchCfg wide_cfg(uint64_t blocks, int num_cus)
{
    LaunchCfg c = auto_cfg(blocks, num_cus);
    const uint64_t tiles = (blocks + 63u) / 64u;
    if (tiles > 8192u) {
        c.wg_waves = tiles < 262144u ? 4 : 8;
        c.tile_order = 1;
    }
    return c;
}
bool cfg_valid(const LaunchCfg& c);

}  // namespace goofy_impl
