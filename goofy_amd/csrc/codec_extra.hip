// codec_extra.hip -- the other side of the encoder: the decode kernel of the
// four formats (per-block decoders in block_decode.h, with the semantics of
// the reference harness's decoders) and a fused decode-and-compare kernel
// that gives the round-trip quality (per-channel squared error, luma error,
// PSNR) of encoded blocks against their source image.  The quality figures
// mirror getMsePsnr (Src/main.cpp:403-469).
//
// Layout as in kernels.hip: one lane per 4x4 block, a wave covers 64
// consecutive blocks; 8- or 16-byte block loads and 16-byte pixel-row
// accesses are coalesced per wave.
//
// Also here: the harness's quality floor, a 2x-downsampled RGB565 copy of the
// source (generateDownsamlpedRgb565Test, Src/main.cpp:501-555), and the
// image-against-image form of the quality sums, so that a caller gets the
// floor's PSNR and the encoder's PSNR over it, as the harness prints them.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include "block_decode.h"
#include "internal.h"
#include "tile_io.h"

#include <mutex>

namespace goofy_impl {

using goofy_dev::decode_block;
using goofy_dev::decode_block_rows;

// The allocation-free quality call's work area (final sums at offset 0, one
// partial per workgroup from kQualityPartialsOffset on), one copy per GPU for
// the life of the process.  Host code never uses this name as an address: the
// device address of each GPU's copy comes from hipGetSymbolAddress below.
static __device__ __align__(256) uint8_t scratch[kQualityNoAllocBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_addr[kMaxDevices] = {};
}  // namespace

hipError_t noalloc_scratch_address(int device, void** addr)
{
    if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch_addr[device]) {
        // `device` is the calling thread's current device: the address is
        // that GPU's copy of the array
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        g_scratch_addr[device] = p;
    }
    *addr = g_scratch_addr[device];
    return hipSuccess;
}

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint2 load_block(const uint2* p)
{
    const u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
    return make_uint2(v.x, v.y);
}

// A block of format FMT: 8 bytes (words x, y; z, w unused) or 16 bytes
// (DXT5 / ETC2 RGBA8: alpha block in x, y, colour block in z, w).
template <int FMT>
__device__ __forceinline__ uint4 load_block_fmt(const uint8_t* blocks, uint64_t i)
{
    if constexpr (FMT >= 2) {
        const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(blocks + i * 16u));
        return make_uint4(v.x, v.y, v.z, v.w);
    } else {
        const uint2 b = load_block(reinterpret_cast<const uint2*>(blocks) + i);
        return make_uint4(b.x, b.y, 0u, 0u);
    }
}

template <int FMT, int STORE>
__global__ __launch_bounds__(256) void k_decode(const uint8_t* __restrict__ blocks, uint8_t* __restrict__ dst,
                                                uint64_t pitch, uint32_t bw, uint32_t nblocks, uint64_t magic,
                                                uint32_t order)
{
    // a wave's 64 consecutive blocks start at `first` (wave-uniform)
    const uint32_t first = __builtin_amdgcn_readfirstlane(xcd_workgroup(order) * 256u + (threadIdx.x & ~63u));
    const uint32_t lane = threadIdx.x & 63u, i = first + lane;
    if (i >= nblocks) return;
    // the four rows are stored together after the block is decoded: storing
    // each row as it comes made the decoders 2-7% slower
    uint32_t px[16];
    decode_block<FMT>(load_block_fmt<FMT>(blocks, i), px);
    if (tile_near(bw, 64u, pitch)) {
        const BlockRows t = block_rows(dst, pitch, bw, magic, first);
        const uint32_t off = block_offset(t, bw, lane);
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const u32x4 v = {px[4 * y], px[4 * y + 1], px[4 * y + 2], px[4 * y + 3]};
            __builtin_amdgcn_raw_buffer_store_b128(v, t.rows, off, (uint32_t)pitch * y, STORE);
        }
    } else {
        const uint32_t by = (uint32_t)(((uint64_t)i * magic) >> 40), bx = i - by * bw;
        uint8_t* out = dst + (uint64_t)by * 4u * pitch + (uint64_t)bx * 16u;
#pragma unroll
        for (int y = 0; y < 4; ++y) {
            const u32x4 v = {px[4 * y], px[4 * y + 1], px[4 * y + 2], px[4 * y + 3]};
            __builtin_nontemporal_store(v, reinterpret_cast<u32x4*>(out + (uint64_t)y * pitch));
        }
    }
}

// Squared errors, summed exactly in integers.  The harness's luma weights are
// 0.21 / 0.72 / 0.07 on bytes 2 / 1 / 0, so 100 x the luma difference is the
// integer 21 dr + 72 dg + 7 db, whose square is
//   441 dr^2 + 5184 dg^2 + 49 db^2 + 3024 dr dg + 294 dr db + 1008 dg db.
// Beyond the channel squares the luma sum needs only the three cross products.
// lane_totals() forms the weighted total once per lane.  The host divides it by
// 10^4 once: the exact value of the harness's sum, which its own double
// arithmetic rounds per pixel (relative differences of order 1e-15 per term).
//   The differences themselves are never formed.  With a row of each image as
// channel planes, four pixels' bytes to a word, products of bytes sum by
// v_dot4_u32_u8, and
//   (a - d)^2         = (a a + d d) - 2 a d
//   (ai - di)(aj - dj) = (ai aj + di dj) - (ai dj + di aj),
// each bracket and product a sum of its own, subtracted once per lane.  24 dot
// products a row of four pixels and 8 v_perm_b32 to split the source's words
// into planes, where forming 16-bit differences and 7 products of them took 38
// instructions and the decoders 6 to 8 more to interleave their planes.  Whole
// calls went from 27.7 to 26.9 us at 4100x3076 and 65.6 to 65.4 at 8192^2
// (ETC1; ETC2 RGBA8 30.6 to 30.1 and 73.3 to 71.8): the kernel then moves 6.0
// TB/s.
//   A lane sums over at most kQualityLaneUnits blocks (or 4-pixel quads): each
// sum is at most 2048 * 16 * 2 * 255^2 = 4,261,478,400 < 2^32.
struct ErrSums {
    uint32_t sq[4], ad[4];       // per byte: a a + d d, and a d
    uint32_t same[3], mixed[3];  // per pair of bytes (2, 1), (2, 0), (1, 0)
};

__device__ __forceinline__ uint32_t dot4(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_udot4(a, b, c, false);
}

// The four pixels of a row as channel planes.
__device__ __forceinline__ void split_row(u32x4 v, uint32_t (&plane)[4])
{
    const uint32_t rg01 = __builtin_amdgcn_perm(v.y, v.x, 0x05010400u), ba01 = __builtin_amdgcn_perm(v.y, v.x, 0x07030602u);
    const uint32_t rg23 = __builtin_amdgcn_perm(v.w, v.z, 0x05010400u), ba23 = __builtin_amdgcn_perm(v.w, v.z, 0x07030602u);
    plane[0] = __builtin_amdgcn_perm(rg23, rg01, 0x05040100u);
    plane[1] = __builtin_amdgcn_perm(rg23, rg01, 0x07060302u);
    plane[2] = __builtin_amdgcn_perm(ba23, ba01, 0x05040100u);
    plane[3] = __builtin_amdgcn_perm(ba23, ba01, 0x07060302u);
}

// Four pixels: source words against decoded planes.  OPAQUE: decoded alpha is
// 255 everywhere, and its error the square of the source's complement.
template <bool OPAQUE>
__device__ __forceinline__ void accum_row(u32x4 src, const uint32_t (&d)[4], ErrSums& s)
{
    uint32_t a[4];
    split_row(src, a);
#pragma unroll
    for (int c = 0; c < (OPAQUE ? 3 : 4); ++c) {
        s.sq[c] = dot4(a[c], a[c], dot4(d[c], d[c], s.sq[c]));
        s.ad[c] = dot4(a[c], d[c], s.ad[c]);
    }
    if constexpr (OPAQUE) s.sq[3] = dot4(~a[3], ~a[3], s.sq[3]);
    constexpr int first[3] = {2, 2, 1}, second[3] = {1, 0, 0};
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const int i = first[k], j = second[k];
        s.same[k] = dot4(a[i], a[j], dot4(d[i], d[j], s.same[k]));
        s.mixed[k] = dot4(a[i], d[j], dot4(d[i], a[j], s.mixed[k]));
    }
}
// The lane's channel sums and its sum of squared luma differences (x 10^4),
// in 64 bits; the luma total is exact and non-negative.
__device__ __forceinline__ void lane_totals(const ErrSums& s, unsigned long long (&e)[4], unsigned long long& ey)
{
    long long x[3];
#pragma unroll
    for (int ch = 0; ch < 4; ++ch) e[ch] = s.sq[ch] - 2ull * s.ad[ch];
#pragma unroll
    for (int k = 0; k < 3; ++k) x[k] = (long long)s.same[k] - (long long)s.mixed[k];
    ey = 441ull * e[2] + 5184ull * e[1] + 49ull * e[0] + (unsigned long long)(3024ll * x[0] + 294ll * x[1] + 1008ll * x[2]);
}

// Sums of one workgroup (256 lanes = 4 waves): wave reduction by lane
// exchange, then the four wave sums.  Lane k of the first wave returns sum k
// (the four channels, then luma, which later lanes return too).
// Every lane of the workgroup must reach this.
__device__ __forceinline__ unsigned long long block_sums(unsigned long long (&e)[4], unsigned long long ey)
{
    __shared__ unsigned long long s_sum[5][4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) e[ch] += __shfl_xor(e[ch], off, 64);
        ey += __shfl_xor(ey, off, 64);
    }
    const uint32_t wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63u) == 0) {
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) s_sum[ch][wave] = e[ch];
        s_sum[4][wave] = ey;
    }
    __syncthreads();
    const uint32_t k = min(threadIdx.x, 4u);
    return s_sum[k][0] + s_sum[k][1] + s_sum[k][2] + s_sum[k][3];
}

// End of a quality kernel.  With a host result (d.host) the launch finishes
// the sums itself, one lane per word (QualityAccum): a lane adds its word and a
// count of one with a device-scope atomic, and the lane whose returned count
// completes the word takes its total in exchange for the zero that the next
// launch starts from, and writes it to pinned host memory, where the host waits
// for it.  The total depends on the exchange's return, so the zero is in place
// before the host can see the word and give the work area to another stream.
// The words need no order among each other and there is no fence (one per
// workgroup is a write-back of the whole L2: the BC1 round trip of an 8192^2
// image took 124 us instead of 51 with it).
//   Atomics on one line run one after another, about 8 ns each: 1536
// workgroups counting on one word took 12 us.  Grids of more workgroups than
// slots therefore add into one of 64 slots first, and the completed slots into
// the total: 24 + 64 at most on a line.
//   A second launch that adds the workgroups' partials (4 us and the gap before
// it) was slower: whole calls from Python, second launch -> this, both with a
// stream synchronisation behind, 512x512 DXT1 21.0 -> 18.9 us, 8192^2 ETC1 69.1
// -> 66.7, floor and image-against-image figures of 4100x3076 57.5 -> 54.7.
// Integer sums: the order of the adds does not show.
// Without d.host the workgroup leaves its partial for k_sums_final.
__device__ __forceinline__ void finish_sums(unsigned long long (&e)[4], unsigned long long ey, const QualityDest& d)
{
    const uint32_t lane = threadIdx.x;
    unsigned long long v = block_sums(e, ey);
    if (!d.host) {
        unsigned long long* part = reinterpret_cast<unsigned long long*>((uint8_t*)d.work + kQualityPartialsOffset);
        if (lane < 5u) part[(size_t)blockIdx.x * 5u + lane] = v;
        return;
    }
    if (lane >= kQualityWords) return;
    if (lane == 4u) v &= 0xFFFFFFFFull;
    if (lane == 5u) v >>= 32;
    constexpr unsigned long long one = 1ull << kQualityCountBit;
    uint32_t parts = gridDim.x;
    if (parts > kQualitySlots) {
        const uint32_t s = blockIdx.x % kQualitySlots;
        const uint32_t in_slot = (parts - s + kQualitySlots - 1u) / kQualitySlots;  // workgroups s, s + 64, ...
        unsigned long long* w = &d.accum->slot[s].word[lane];
        const unsigned long long before = __hip_atomic_fetch_add(w, v + one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((before >> kQualityCountBit) != in_slot - 1u) return;
        v = __hip_atomic_exchange(w, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & (one - 1u);
        parts = kQualitySlots;
    }
    unsigned long long* w = &d.accum->total.word[lane];
    const unsigned long long before = __hip_atomic_fetch_add(w, v + one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((before >> kQualityCountBit) != parts - 1u) return;
    v = __hip_atomic_exchange(w, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & (one - 1u);
    __hip_atomic_store(&d.host->word[lane], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One wave's tile of the round trip: 64 consecutive blocks from `first`,
// each lane's block and its four source rows.  Lanes past the last block
// load the last block again and skip its sums, so every load is issued
// unconditionally.
struct QTile {
    uint4 b;
    u32x4 v[4];
};

template <int FMT, bool NEAR>
__device__ __forceinline__ void load_qtile(const uint8_t* __restrict__ blocks, const uint8_t* __restrict__ src,
                                           uint64_t pitch, uint32_t bw, uint32_t nblocks, uint64_t magic,
                                           uint32_t first, uint32_t lane, QTile& t)
{
    const uint32_t k = min(lane, nblocks - 1u - first), i = first + k;
    t.b = load_block_fmt<FMT>(blocks, i);
    if constexpr (NEAR) {
        const BlockRows r = block_rows(src, pitch, bw, magic, first);
        const uint32_t off = block_offset(r, bw, k);
#pragma unroll
        for (int y = 0; y < 4; ++y)
            t.v[y] = __builtin_amdgcn_raw_buffer_load_b128(r.rows, off, (uint32_t)pitch * y, kBufAux<true>);
    } else {
        const uint32_t by = (uint32_t)(((uint64_t)i * magic) >> 40), bx = i - by * bw;
        const uint8_t* row = src + (uint64_t)by * 4u * pitch + (uint64_t)bx * 16u;
#pragma unroll
        for (int y = 0; y < 4; ++y)
            t.v[y] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(row + (uint64_t)y * pitch));
    }
}

// Decode the lane's block and add its errors against the source rows, each
// decoded row compared as it comes (4 decoded pixels live).
template <int FMT>
__device__ __forceinline__ void sqerr_tile(const QTile& t, bool valid, ErrSums& acc)
{
    if (valid)
        decode_block_rows<FMT>(t.b, [&](int y, const uint32_t (&plane)[4]) {
            accum_row<goofy_dev::kOpaque<FMT>>(t.v[y], plane, acc);
        });
}

// Runs of 32 workgroups per XCD (xcd_workgroup), as the grid-stride loops of
// the quality kernels walk the image: BC1 at 8192^2 64.7 -> 63.9 us, ETC2 RGBA8
// 72.3 -> 70.9, at 12004x9000 106.5 -> 103.4, image sums 94.5 -> 93.5.
constexpr uint32_t kQualityOrder = 6;

// A wave's tiles first, first + step, ... in a grid-stride loop, one tile at a
// time (48-65 VGPRs, so that all of the grid's 6 waves per SIMD fit).  Loading
// the next tile into a second register set before comparing this one needs
// 89-100 VGPRs with the plane sums and was no faster (whole calls at 8192^2,
// two sets / one: BC1 65.7 / 64.8 us, ETC1 65.4 / 65.4, BC3 71.6 / 70.5).
template <int FMT, bool NEAR>
__device__ __forceinline__ void sqerr_loop(const uint8_t* __restrict__ blocks, const uint8_t* __restrict__ src,
                                           uint64_t pitch, uint32_t bw, uint32_t nblocks, uint64_t magic,
                                           ErrSums& acc)
{
    const uint32_t step = gridDim.x * 256u;  // nblocks <= kQualityMaxLaunchUnits < 2^30: no overflow below
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t t = __builtin_amdgcn_readfirstlane(xcd_workgroup(kQualityOrder) * 256u + (threadIdx.x & ~63u));
    for (; t < nblocks; t += step) {
        QTile a;
        load_qtile<FMT, NEAR>(blocks, src, pitch, bw, nblocks, magic, t, lane, a);
        sqerr_tile<FMT>(a, t + lane < nblocks, acc);
    }
}

// Round-trip error: decode each block in registers and compare it with the
// source pixels.  Per workgroup: e[0..3] = squared error of bytes 0..3 of the
// pixels, ey = sum of squared luma differences x 10^4 with the harness's
// weights (0.21, 0.72, 0.07 on bytes 2, 1, 0 -- getMsePsnr reads a pixel as a
// little-endian word and takes bits 16..23 as "red").  Grid-stride over the
// blocks (at most 1536 workgroups); finish_sums brings the workgroups' sums
// together, or, for the allocation-free call, leaves them for k_sums_final.
template <int FMT>
__global__ __launch_bounds__(256) void k_sqerr(const uint8_t* __restrict__ blocks, const uint8_t* __restrict__ src,
                                               uint64_t pitch, uint32_t bw, uint32_t nblocks, uint64_t magic,
                                               const QualityDest dest)
{
    ErrSums acc = {};
    if (tile_near(bw, 64u, pitch)) sqerr_loop<FMT, true>(blocks, src, pitch, bw, nblocks, magic, acc);
    else sqerr_loop<FMT, false>(blocks, src, pitch, bw, nblocks, magic, acc);
    unsigned long long e[4], ey;
    lane_totals(acc, e, ey);
    finish_sums(e, ey, dest);
}

// Squared errors of two whole RGBA8 images (getMsePsnr over a source and any
// other image of its size).  One lane-step per 4 pixels of one row.
__global__ __launch_bounds__(256) void k_sqerr_images(const uint8_t* __restrict__ a, uint64_t pitch_a,
                                                      const uint8_t* __restrict__ b, uint64_t pitch_b, uint32_t qw,
                                                      uint32_t nquads, uint64_t magic, const QualityDest dest)
{
    ErrSums acc = {};
    for (uint64_t i = (uint64_t)xcd_workgroup(kQualityOrder) * 256u + threadIdx.x; i < nquads; i += (uint64_t)gridDim.x * 256u) {
        const uint32_t y = (uint32_t)((i * magic) >> 40), x = (uint32_t)i - y * qw;
        const u32x4 va =
            __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(a + (uint64_t)y * pitch_a + (uint64_t)x * 16u));
        const u32x4 vb =
            __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(b + (uint64_t)y * pitch_b + (uint64_t)x * 16u));
        uint32_t d[4];
        split_row(vb, d);
        accum_row<false>(va, d, acc);
    }
    unsigned long long e[4], ey;
    lane_totals(acc, e, ey);
    finish_sums(e, ey, dest);
}

// One workgroup adds the g <= kQualityMaxGroups partials of the
// allocation-free call in a fixed order into *out -- with accumulate, onto the
// sums already in *out (the stripes of a large image, launched one after
// another on one stream).  A lane issues the loads of all its partials before
// it adds any.
__global__ __launch_bounds__(256) void k_sums_final(const QualitySums* __restrict__ part, uint32_t g,
                                                    QualitySums* __restrict__ out, uint32_t accumulate)
{
    constexpr uint32_t kPer = kQualityMaxGroups / 256u;
    static_assert(kQualityMaxGroups % 256u == 0, "partials per lane");
    QualitySums p[kPer];
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        const uint32_t k = threadIdx.x + 256u * j;
        p[j] = k < g ? part[k] : QualitySums{{0, 0, 0, 0, 0}};
    }
    unsigned long long acc[4] = {0, 0, 0, 0};
    unsigned long long ey = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
#pragma unroll
        for (int ch = 0; ch < 4; ++ch) acc[ch] += p[j].sum[ch];
        ey += p[j].sum[4];
    }
    const unsigned long long v = block_sums(acc, ey);
    if (threadIdx.x < 5u) out->sum[threadIdx.x] = v + (accumulate ? out->sum[threadIdx.x] : 0ull);
}

// One 2x2 cell of the quality floor (Src/main.cpp:507-553).  p and q are the
// cell's two pixels of its upper row, u and v those of its lower row, each
// read as a little-endian word (byte 0 = "b", 1 = "g", 2 = "r").  Each
// channel is averaged with rounding, (sum + 2) >> 2, cut to 5 ("r") or 6 bits
// ("g", "b") and widened back to 8 bits as the harness does it: r5 << 3 | r5 >> 2,
// g6 << 2 | g6 >> 4, and for "b" b6 << 2 | (b6 >> 2) & 7, three bits ORed into
// a two-bit gap (so "b" is not a plain 6-bit replication).  Alpha is 255.
__device__ __forceinline__ uint32_t rgb565_cell(uint32_t p, uint32_t q, uint32_t u, uint32_t v)
{
    const uint32_t m = 0x00FF00FFu;
    const uint32_t s02 = (p & m) + (q & m) + (u & m) + (v & m) + 0x00020002u;  // bytes 0 and 2, 16-bit lanes
    const uint32_t s1 = ((p >> 8) & 0xFFu) + ((q >> 8) & 0xFFu) + ((u >> 8) & 0xFFu) + ((v >> 8) & 0xFFu) + 2u;
    const uint32_t b6 = ((s02 >> 2) & 0xFFu) >> 2;
    const uint32_t r5 = ((s02 >> 18) & 0xFFu) >> 3;
    const uint32_t g6 = ((s1 >> 2) & 0xFFu) >> 2;
    const uint32_t r = (r5 << 3) | ((r5 >> 2) & 7u);
    const uint32_t g = (g6 << 2) | ((g6 >> 4) & 3u);
    const uint32_t b = (b6 << 2) | ((b6 >> 2) & 7u);
    return (r << 16) | (g << 8) | b | 0xFF000000u;
}

// One lane per 4 pixels x 2 rows (two cells): 32 bytes in, 32 bytes out.
__global__ __launch_bounds__(256) void k_rgb565_baseline(const uint8_t* __restrict__ src, uint64_t src_pitch,
                                                         uint8_t* __restrict__ dst, uint64_t dst_pitch, uint32_t qw,
                                                         uint32_t nunits, uint64_t magic, uint32_t order)
{
    const uint32_t i = xcd_workgroup(order) * 256u + threadIdx.x;
    if (i >= nunits) return;
    const uint32_t ry = (uint32_t)(((uint64_t)i * magic) >> 40), x = i - ry * qw;
    const uint8_t* s0 = src + (uint64_t)(2u * ry) * src_pitch + (uint64_t)x * 16u;
    const u32x4 t = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(s0));
    const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(s0 + src_pitch));
    const uint32_t c0 = rgb565_cell(t.x, t.y, w.x, w.y);
    const uint32_t c1 = rgb565_cell(t.z, t.w, w.z, w.w);
    const u32x4 o = {c0, c0, c1, c1};
    uint8_t* d0 = dst + (uint64_t)(2u * ry) * dst_pitch + (uint64_t)x * 16u;
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(d0));
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4*>(d0 + dst_pitch));
}

}  // namespace

template <int FMT>
static void decode_go(int store, dim3 grid, hipStream_t stream, const uint8_t* blocks, uint8_t* dst, uint64_t pitch,
                      uint32_t bw, uint32_t nblocks, uint64_t magic)
{
    const auto go = [&](auto kernel) {  // runs of 64 workgroups per XCD
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, blocks, dst, pitch, bw, nblocks, magic, 7u);
    };
    if (store == kStreamThrough) go(k_decode<FMT, kStreamThrough>);
    else if (store == kCached) go(k_decode<FMT, kCached>);
    else go(k_decode<FMT, kStream>);
}

hipError_t launch_decode(int fmt, const void* blocks, void* dst, uint32_t width, uint32_t height, size_t pitch,
                         hipStream_t stream)
{
    const uint32_t bw = width / 4, nblocks = bw * (height / 4);
    if (nblocks == 0) return hipSuccess;
    const dim3 grid((nblocks + 255u) / 256u);
    const uint64_t magic = div_magic(bw);
    const uint8_t* b = static_cast<const uint8_t*>(blocks);
    uint8_t* d = static_cast<uint8_t*>(dst);
    const int store = decode_store(fmt, bw, dst, pitch, height);
    switch (fmt) {
    case 0: decode_go<0>(store, grid, stream, b, d, pitch, bw, nblocks, magic); break;
    case 1: decode_go<1>(store, grid, stream, b, d, pitch, bw, nblocks, magic); break;
    case 2: decode_go<2>(store, grid, stream, b, d, pitch, bw, nblocks, magic); break;
    default: decode_go<3>(store, grid, stream, b, d, pitch, bw, nblocks, magic);
    }
    return hipGetLastError();
}

// The allocation-free call's second kernel.
static hipError_t quality_final(const QualityDest& d, uint32_t grid, bool accumulate, hipStream_t stream)
{
    if (!d.host)
        hipLaunchKernelGGL(k_sums_final, dim3(1), dim3(256), 0, stream,
                           reinterpret_cast<const QualitySums*>(static_cast<uint8_t*>(d.work) + kQualityPartialsOffset),
                           grid, static_cast<QualitySums*>(d.work), accumulate ? 1u : 0u);
    return hipGetLastError();
}

hipError_t launch_sqerr(int fmt, const void* blocks, const void* src, size_t pitch, uint32_t width, uint32_t height,
                        const QualityDest& dest, bool accumulate, hipStream_t stream)
{
    const uint32_t bw = width / 4, nblocks = bw * (height / 4);
    if (nblocks == 0 || nblocks > kQualityMaxLaunchUnits) return hipErrorInvalidValue;  // 32-bit lane sums
    const uint32_t g = quality_grid(nblocks);
    const uint64_t magic = div_magic(bw);
    const uint8_t* b = static_cast<const uint8_t*>(blocks);
    const uint8_t* s = static_cast<const uint8_t*>(src);
    switch (fmt) {
    case 0: hipLaunchKernelGGL(k_sqerr<0>, dim3(g), dim3(256), 0, stream, b, s, (uint64_t)pitch, bw, nblocks, magic, dest); break;
    case 1: hipLaunchKernelGGL(k_sqerr<1>, dim3(g), dim3(256), 0, stream, b, s, (uint64_t)pitch, bw, nblocks, magic, dest); break;
    case 2: hipLaunchKernelGGL(k_sqerr<2>, dim3(g), dim3(256), 0, stream, b, s, (uint64_t)pitch, bw, nblocks, magic, dest); break;
    default: hipLaunchKernelGGL(k_sqerr<3>, dim3(g), dim3(256), 0, stream, b, s, (uint64_t)pitch, bw, nblocks, magic, dest);
    }
    return quality_final(dest, g, accumulate, stream);
}

hipError_t launch_sqerr_images(const void* a, size_t pitch_a, const void* b, size_t pitch_b, uint32_t width,
                               uint32_t height, const QualityDest& dest, hipStream_t stream)
{
    const uint32_t qw = width / 4, n = qw * height;
    if (n == 0 || n > kQualityMaxLaunchUnits) return hipErrorInvalidValue;  // 32-bit lane sums
    hipLaunchKernelGGL(k_sqerr_images, dim3(quality_grid(n)), dim3(256), 0, stream, (const uint8_t*)a,
                       (uint64_t)pitch_a, (const uint8_t*)b, (uint64_t)pitch_b, qw, n, div_magic(qw), dest);
    return hipGetLastError();
}

hipError_t launch_rgb565_baseline(const void* src, size_t src_pitch, void* dst, size_t dst_pitch, uint32_t width,
                                  uint32_t height, hipStream_t stream, hipEvent_t start, hipEvent_t stop)
{
    const uint32_t qw = width / 4, n = qw * (height / 2);
    if (n == 0) return hipSuccess;
    const dim3 grid((n + 255u) / 256u), block(256);
    // Rows off the 128-byte lines in runs of 32 workgroups per XCD: 4100x3076
    // 19.0 -> 18.5 us, 8196x8192 88.9 -> 88.2; rows on them were up to 2% slower so
    // (8192^2 81.4 -> 83.3).
    const uint32_t order = src_pitch % 128 != 0 || dst_pitch % 128 != 0 ? 6u : 0u;
    if (start || stop)
        hipExtLaunchKernelGGL(k_rgb565_baseline, grid, block, 0, stream, start, stop, 0, (const uint8_t*)src,
                              (uint64_t)src_pitch, (uint8_t*)dst, (uint64_t)dst_pitch, qw, n, div_magic(qw), order);
    else
        hipLaunchKernelGGL(k_rgb565_baseline, grid, block, 0, stream, (const uint8_t*)src, (uint64_t)src_pitch,
                           (uint8_t*)dst, (uint64_t)dst_pitch, qw, n, div_magic(qw), order);
    return hipGetLastError();
}

}  // namespace goofy_impl
