// block_codec.h -- the per-4x4-block DXT1 / ETC1S encoder for gfx950.
//
// One lane owns one block: its 16 RGBA8 pixels sit in 16 VGPRs (dword p =
// pixel 4*row+col, R in bits 0..7) and every step below is lane-local byte
// arithmetic.  This replaces the 16-byte SSE2 lanes of goofySimdEncode
// (GoofyTC/goofy_tc.h:1069-1494), which encode 4 blocks per call and spend
// most of their instructions on transposes (transposeAs4x4 :263-276,
// deinterleaveRGB :278-299, transposeAs4x4x4 :327-358); here there is no
// transpose at all: v_perm_b32 gathers bytes, v_lerp_u8 is the per-byte
// rounding average (_mm_avg_epu8), packed 16-bit min/max (three-input ones
// where the lanes hold bytes) give the bounding box, and per-byte comparisons
// come out of the same rounding average.
//
// Integer semantics (all values u8, avg(a,b) = (a+b+1)>>1):
//   Y(r,g,b) = avg(avg(r,b),g)                       goofy_tc.h:1166,1205
//   range = max(Y(max)-Y(min), 8), mid = avg(Y(min),Y(max))   :1176-1179
//   qt = avg(avg(range,0),0) + avg(avg(avg(range,0),0),0)     :1184-1190
//   gez(p) = Y(p) >= mid ; near(p) = |Y(p)-mid| < qt          :1212-1224
//     (the header clamps |Y-mid| to 127 before a signed compare; qt <= 96,
//      so the clamp never changes the outcome)
//   q5(c) = avg(avg(avg(subsat(c,8),0),0),0) = c ? (c-1)>>3 : 0   :1309
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace goofy_dev {

// DXT5 (BC3) and ETC2 RGBA8 are 16-byte blocks: an alpha block, then the
// DXT1 / ETC1S block of the same pixels.
enum : int { kDXT1 = 0, kETC1 = 1, kDXT5 = 2, kETC2 = 3 };

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));

// Per-byte rounding average of two packed words: v_lerp_u8 with a carry-in
// of one in every byte, i.e. (a+b+1)>>1 per byte.
__device__ __forceinline__ uint32_t avg4(uint32_t a, uint32_t b) { return __builtin_amdgcn_lerp(a, b, 0x01010101u); }
// a ^ b ^ c as one v_bitop3_b32 (truth table 0x96, the same for every operand order).
__device__ __forceinline__ uint32_t xor3(uint32_t a, uint32_t b, uint32_t c)
{
    return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96u);
}

// Bits of m where `sel` is set, bits of o elsewhere: one v_bitop3_b32
// (truth table indexed by sel*4 + m*2 + o).  Written as the builtin so that
// the compiler keeps the single select instead of re-deriving masks from
// the known-zero bits of shifted operands.
__device__ __forceinline__ uint32_t bsel(uint32_t sel, uint32_t m, uint32_t o)
{
    return __builtin_amdgcn_bitop3_b32(sel, m, o, 0xCAu);
}

// v_perm_b32: byte i of the result is byte sel[i] of {hi:lo} (0..3 = lo,
// 4..7 = hi, 0x0c = zero).
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel)
{
    return __builtin_amdgcn_perm(hi, lo, sel);
}

__device__ __forceinline__ uint32_t pk_min16(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
__device__ __forceinline__ uint32_t pk_max16(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// Three-input min / max of 16-bit lanes that hold 0..255, as one
// v_pk_minimum3_f16 / v_pk_maximum3_f16: read as half-precision numbers such
// lanes are +0 and positive subnormals, whose order is that of the integers,
// and the kernels keep half-precision subnormals (denorm mode 16/64 = 3), so
// the selected lane comes out bit for bit.  One instruction takes two new
// pairs of lanes where v_pk_min_u16 takes one.
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t min3_b16(uint32_t a, uint32_t b, uint32_t c)
{
    const h16x2 r = __builtin_elementwise_minimum(
        __builtin_elementwise_minimum(__builtin_bit_cast(h16x2, a), __builtin_bit_cast(h16x2, b)),
        __builtin_bit_cast(h16x2, c));
    return __builtin_bit_cast(uint32_t, r);
}
__device__ __forceinline__ uint32_t max3_b16(uint32_t a, uint32_t b, uint32_t c)
{
    const h16x2 r = __builtin_elementwise_maximum(
        __builtin_elementwise_maximum(__builtin_bit_cast(h16x2, a), __builtin_bit_cast(h16x2, b)),
        __builtin_bit_cast(h16x2, c));
    return __builtin_bit_cast(uint32_t, r);
}

// Luma of the colour in bytes 0..2 of c (byte 3 ignored), in byte 1 of the
// result; bytes 2 and 3 are zero, byte 0 is don't-care.  The two nested
// rounding averages come to (R + 2G + B + 3) >> 2, a dot product: with the
// weights and the 3 times 64 the shift by 2 ends on a byte boundary (64 x 1023
// < 2^16).  One v_dot4_u32_u8 per pixel.
__device__ __forceinline__ uint32_t luma_b1(uint32_t c)
{
    return __builtin_amdgcn_udot4(c, 0x00408040u, 192u, false);
}

// Luma of four pixels, packed: byte i = Y(p_i).  Seven instructions (nine with
// byte averages).
__device__ __forceinline__ uint32_t luma4(uint32_t p0, uint32_t p1, uint32_t p2, uint32_t p3)
{
    return perm(luma_b1(p1), luma_b1(p0), 0x0c0c0501u) | perm(luma_b1(p3), luma_b1(p2), 0x05010c0cu);
}

// Byte 0 of x copied into all four bytes (v_perm_b32 broadcast; avoids the
// quarter-rate v_mul_lo_u32 of x * 0x01010101).
__device__ __forceinline__ uint32_t rep4(uint32_t x) { return perm(0u, x, 0x00000000u); }

// 8-bit channel -> 5-bit, closed form of the header's three-halvings cascade.
__device__ __forceinline__ uint32_t q5(uint32_t c) { return (c - (c != 0u ? 1u : 0u)) >> 3; }

struct BlockStats {
    uint32_t range, mid, qt;
    uint32_t mn, mx;  // corners of the bounding box: bytes R, G, B, 0
};

// The rest of the statistics from the bounding-box corners.  The roundings
// (x + 1) >> 1 of mid and qt are byte averages (range <= 255).
__device__ __forceinline__ BlockStats corner_stats(uint32_t mn, uint32_t mx)
{
    BlockStats s;
    s.mn = mn;
    s.mx = mx;
    const uint32_t ymn = luma_b1(mn), ymx = luma_b1(mx);
    const uint32_t d = (ymx >> 8) - (ymn >> 8);  // >= 0: luma is monotone per channel
    s.range = d > 8u ? d : 8u;
    s.mid = (avg4(ymn, ymx) >> 8) & 0xFFu;
    const uint32_t half = avg4(s.range, 0u);
    const uint32_t quarter = avg4(half, 0u);
    const uint32_t eighth = avg4(quarter, 0u);
    s.qt = quarter + eighth;  // <= 96
    return s;
}

// R, B bounding box in the two 16-bit halves of p & 0x00ff00ff: the 16
// masked words through a chain of three-input min / max (8 + 8 instructions
// instead of 15 + 15).
__device__ __forceinline__ void rb_box(const uint32_t (&p)[16], uint32_t& mnrb, uint32_t& mxrb)
{
    uint32_t rb[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) rb[i] = p[i] & 0x00FF00FFu;
    mnrb = min3_b16(rb[0], rb[1], rb[2]);
    mxrb = max3_b16(rb[0], rb[1], rb[2]);
#pragma unroll
    for (int i = 3; i < 15; i += 2) {
        mnrb = min3_b16(mnrb, rb[i], rb[i + 1]);
        mxrb = max3_b16(mxrb, rb[i], rb[i + 1]);
    }
    mnrb = pk_min16(mnrb, rb[15]);
    mxrb = pk_max16(mxrb, rb[15]);
}

__device__ __forceinline__ BlockStats block_stats(const uint32_t (&p)[16])
{
    uint32_t mnrb, mxrb;
    rb_box(p, mnrb, mxrb);
    // G of two pixels packed into one word with v_perm ([G_a 0 G_b 0]),
    // then the three-input min / max over the eight words
    uint32_t g[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) g[i] = perm(p[2 * i + 1], p[2 * i], 0x0c050c01u);
    uint32_t mng = min3_b16(g[0], g[1], g[2]), mxg = max3_b16(g[0], g[1], g[2]);
    mng = min3_b16(mng, g[3], g[4]);
    mxg = max3_b16(mxg, g[3], g[4]);
    mng = min3_b16(mng, g[5], g[6]);
    mxg = max3_b16(mxg, g[5], g[6]);
    mng = pk_min16(mng, g[7]);
    mxg = pk_max16(mxg, g[7]);
    mng = pk_min16(mng, mng >> 16);
    mxg = pk_max16(mxg, mxg >> 16);
    return corner_stats(perm(mng, mnrb, 0x0c020400u), perm(mxg, mxrb, 0x0c020400u));
}

// The same for a block whose alpha range is needed too: v_pk_min_u16 /
// v_pk_max_u16 over the raw pixel words order each 16-bit lane by its high
// byte first, so the lanes' high bytes come out as the G range (byte 1) and
// the alpha range (byte 3) together, in the 30 instructions that the G
// pairs and a separate alpha pass would take 44.
__device__ __forceinline__ BlockStats block_stats_alpha(const uint32_t (&p)[16], uint32_t& amn, uint32_t& amx)
{
    uint32_t mnrb, mxrb;
    rb_box(p, mnrb, mxrb);
    uint32_t lo = p[0], hi = p[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) {
        lo = pk_min16(lo, p[i]);
        hi = pk_max16(hi, p[i]);
    }
    amn = lo >> 24;
    amx = hi >> 24;
    return corner_stats(perm(lo, mnrb, 0x0c020500u), perm(hi, mxrb, 0x0c020500u));
}

// Per-byte comparison masks for four packed lumas y4 against the block's mid
// and threshold: bit 7 of each byte of *gez = (y >= mid), other bits
// don't-care; of *near = (|y - mid| < qt) = (lo <= y <= hi), other bits zero.  Uses avg(~a, b) >= 128  <=>  b >= a
// for bytes a, b, and for the upper bound the floor average:
// (~hi + y) >> 1 >= 128  <=>  y > hi, which also holds for hi = 255 (never).
// nhi4 = ~hi in all four bytes.
__device__ __forceinline__ void compare4(uint32_t y4, uint32_t nmid4, uint32_t nlo4, uint32_t nhi4, uint32_t* gez,
                                         uint32_t* near)
{
    *gez = avg4(nmid4, y4);
    // a & ~b & c (truth table 0x20)
    *near = __builtin_amdgcn_bitop3_b32(avg4(nlo4, y4), __builtin_amdgcn_lerp(nhi4, y4, 0u), 0x80808080u, 0x20u);
}

// q5 of the two 16-bit lanes of x: subsat(c, 1) >> 3 per lane.
__device__ __forceinline__ uint32_t q5x2(uint32_t x)
{
    const u16x2 one = {1, 1}, three = {3, 3};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_sub_sat(__builtin_bit_cast(u16x2, x), one) >> three);
}

// The DXT1 endpoint word c0 | c1 << 16: c0 = RGB565 of the box maximum with
// the green LSB forced to 1 (so c0 > c1, 4-colour mode), c1 = RGB565 of the
// minimum.  A v_perm_b32 per channel pairs it of both corners, maximum in the
// low 16-bit lane, and all six channels go through q5 in 16-bit lanes.
__device__ __forceinline__ uint32_t dxt1_endpoints(const BlockStats& s)
{
    const uint32_t r = q5x2(perm(s.mn, s.mx, 0x0c040c00u));
    const uint32_t g = q5x2(perm(s.mn, s.mx, 0x0c050c01u));
    const uint32_t b = q5x2(perm(s.mn, s.mx, 0x0c060c02u));
    return (r << 11) | (g << 6) | b | 0x20u;
}

// The DXT1 index word from the per-row compare masks (bit 7 of byte c of
// gez[r] / near[r] for pixel (r, c)): pixel (r, c)'s 2-bit code, bit 0 =
// y < mid and bit 1 = near, at bits 8r + 2c.  A row's flags, 0 or 128 each,
// weighted by 4^c and 2 x 4^c, are 128 times the row's index byte: two dot
// products a row.  Rows are joined in pairs below 2^23 before the 128 goes.
__device__ __forceinline__ uint32_t dxt1_index_word(const uint32_t (&gez)[4], const uint32_t (&near)[4])
{
    uint32_t row[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        row[r] = __builtin_amdgcn_udot4(
            near[r], 0x80200802u, __builtin_amdgcn_udot4(~gez[r] & 0x80808080u, 0x40100401u, 0u, false), false);
    return ((row[0] + (row[1] << 8)) >> 7) | ((row[2] + (row[3] << 8)) << 9);
}

// The ETC1S selector word (goofy_tc.h:1375-1395: word bit j <-> column
// {2,3,0,1}[j>>2], row j&3; the MSB plane N in bits 16..31, then inverted)
// from the same masks.  Each plane gathers row r's flags into bit 4 + r of
// byte c (row 3's stay in bit 7), then a bit select folds the column nibbles
// into bytes 1 (columns 0, 1) and 3 (columns 2, 3).
__device__ __forceinline__ uint32_t etc1_selector_word(const uint32_t (&gez)[4], const uint32_t (&near)[4])
{
    auto plane = [](const uint32_t (&f)[4]) {
        const uint32_t t = bsel(0x10101010u, f[0] >> 3, bsel(0x20202020u, f[1] >> 2, bsel(0x40404040u, f[2] >> 1, f[3])));
        return bsel(0x0F000F00u, t << 4, t);
    };
    return ~perm(plane(near), plane(gez), 0x05070103u);  // G: cols 2|3, 0|1; then N's
}

// DXT1 (BC1) block: returns {c0 | c1<<16, indices} as two little-endian words.
__device__ __forceinline__ uint2 encode_dxt1(const uint32_t (&p)[16], const BlockStats& s)
{
    const uint32_t lo = s.mid + 1u > s.qt ? s.mid + 1u - s.qt : 0u;          // y >= lo
    const uint32_t hi = s.mid + s.qt - 1u < 255u ? s.mid + s.qt - 1u : 255u;  // y <= hi
    const uint32_t nmid4 = rep4(~s.mid);
    const uint32_t nlo4 = rep4(~lo);
    const uint32_t nhi4 = rep4(~hi);

    uint32_t gez[4], near[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        compare4(luma4(p[4 * r], p[4 * r + 1], p[4 * r + 2], p[4 * r + 3]), nmid4, nlo4, nhi4, &gez[r], &near[r]);
    return make_uint2(dxt1_endpoints(s), dxt1_index_word(gez, near));
}

__device__ __forceinline__ uint2 encode_dxt1(const uint32_t (&p)[16]) { return encode_dxt1(p, block_stats(p)); }

// ETC1 base-colour bytes of the block, from its average colour: each
// channel of avgc moved by the luma correction (up: + corr, else - corr) with
// saturation to 0..255 (goofy_tc.h:1431-1449), then cut to 5 bits in place,
// q5(b) << 3 == subsat(b, 1) & 0xf8.  The correction is the signed
// clamp(mid - Y(avgc), -127, 127), so a channel becomes
// clamp(c + clamp(mid - Y, -127, 127), 0, 255); with the subtraction of one
// folded in, clamp(c + clamp(mid - Y, -127, 127) - 1, 0, 254) & 0xf8.  R and
// B run in the two 16-bit lanes of one word, G in another: one signed 16-bit
// add and a v_pk_max_i16 / v_pk_min_i16 clamp per word.
typedef short i16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ uint32_t etc1_base_bytes(uint32_t avgc, uint32_t mid)
{
    const int32_t ya = (int32_t)(luma_b1(avgc) >> 8);
    const int32_t t = (int32_t)mid - ya - 1;
    const int32_t sd = t < -128 ? -128 : (t > 126 ? 126 : t);  // the correction minus one
    const uint32_t sd2 = perm(0u, (uint32_t)sd, 0x01000100u);   // in both lanes
    const i16x2 zero = {0, 0}, top = {254, 254};
    auto base = [&](uint32_t lanes) {  // lanes: two channels in 16-bit lanes, 0..255 each
        const i16x2 v = __builtin_bit_cast(i16x2, lanes) + __builtin_bit_cast(i16x2, sd2);
        const i16x2 c = __builtin_elementwise_min(__builtin_elementwise_max(v, zero), top);
        return __builtin_bit_cast(uint32_t, c) & 0x00F800F8u;
    };
    return base(avgc & 0x00FF00FFu) | ((base((avgc >> 8) & 0x00FF00FFu) & 0xFFu) << 8);
}

// ETC1 codeword-table index for the brightness range: the number of the
// breakpoints 21, 43, 73, 105, 151, 181, 253 of etc1BrighnessRangeTocontrolByte
// (GoofyTC/goofy_tc.h:1040-1056) that the range exceeds.  range <= 255, so
// the seven compares range >= t + 1 run as byte compares, four to a word
// (avg(~t', r) >= 128 <=> r >= t'), and a popcount of their flags counts them.
__device__ __forceinline__ uint32_t etc1_table(uint32_t range)
{
    const uint32_t r4 = rep4(range);
    const uint32_t lo = avg4(~0x6A4A2C16u, r4);  // t + 1 = 22, 44, 74, 106
    const uint32_t hi = avg4(~0x00FEB698u, r4);  // 152, 182, 254 (byte 3 unused)
    return (uint32_t)(__builtin_popcount(lo & 0x80808080u) + __builtin_popcount(hi & 0x00808080u));
}

// ETC1S block: differential mode, zero deltas, one table for both halves,
// flip = 1; returns the 8 bytes as two little-endian words.
__device__ __forceinline__ uint2 encode_etc1(const uint32_t (&p)[16], const BlockStats& s)
{
    const uint32_t lo = s.mid + 1u > s.qt ? s.mid + 1u - s.qt : 0u;
    const uint32_t hi = s.mid + s.qt - 1u < 255u ? s.mid + s.qt - 1u : 255u;
    const uint32_t nmid4 = rep4(~s.mid);
    const uint32_t nlo4 = rep4(~lo);
    const uint32_t nhi4 = rep4(~hi);

    uint32_t gez[4], near[4];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        compare4(luma4(p[4 * r], p[4 * r + 1], p[4 * r + 2], p[4 * r + 3]), nmid4, nlo4, nhi4, &gez[r], &near[r]);
    const uint32_t w1 = etc1_selector_word(gez, near);

    // Average colour: rows first, then columns (goofy_tc.h:1402-1414).
    uint32_t col[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) col[x] = avg4(avg4(p[x], p[4 + x]), avg4(p[8 + x], p[12 + x]));
    const uint32_t avgc = avg4(avg4(col[0], col[1]), avg4(col[2], col[3]));
    // Shift its brightness onto mid (goofy_tc.h:1431-1449).
    uint32_t w0 = etc1_base_bytes(avgc, s.mid);
    const uint32_t cw = etc1_table(s.range);
    w0 |= ((cw << 5) | (cw << 2) | 3u) << 24;
    return make_uint2(w0, w1);
}

__device__ __forceinline__ uint2 encode_etc1(const uint32_t (&p)[16]) { return encode_etc1(p, block_stats(p)); }

// ---- both formats from one classification (the dual-format kernel) --------
// The same arithmetic as encode_dxt1 / encode_etc1 above, split into the part
// both formats share -- statistics and, per row r, the per-byte masks of
// (y >= mid) and (|y - mid| < qt) -- and the packing of each format.  The
// single-format encoders keep their own instruction order.
//
// What both formats need from a block.
struct BlockClass {
    BlockStats s;
    uint32_t gez[4], near[4];
};

__device__ __forceinline__ BlockClass classify(const uint32_t (&p)[16], const BlockStats& s)
{
    BlockClass c;
    c.s = s;
    const uint32_t lo = c.s.mid + 1u > c.s.qt ? c.s.mid + 1u - c.s.qt : 0u;          // y >= lo
    const uint32_t hi = c.s.mid + c.s.qt - 1u < 255u ? c.s.mid + c.s.qt - 1u : 255u;  // y <= hi
    const uint32_t nmid4 = rep4(~c.s.mid);
    const uint32_t nlo4 = rep4(~lo);
    const uint32_t nhi4 = rep4(~hi);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t y4 = luma4(p[4 * r], p[4 * r + 1], p[4 * r + 2], p[4 * r + 3]);
        compare4(y4, nmid4, nlo4, nhi4, &c.gez[r], &c.near[r]);
    }
    return c;
}

__device__ __forceinline__ BlockClass classify(const uint32_t (&p)[16]) { return classify(p, block_stats(p)); }

// DXT1 words from a classified block (as encode_dxt1).
__device__ __forceinline__ uint2 pack_dxt1(const BlockClass& c)
{
    return make_uint2(dxt1_endpoints(c.s), dxt1_index_word(c.gez, c.near));
}

// ETC1S words from a classified block and its pixels (as encode_etc1).
__device__ __forceinline__ uint2 pack_etc1(const uint32_t (&p)[16], const BlockClass& c)
{
    const uint32_t w1 = etc1_selector_word(c.gez, c.near);

    // Average colour: rows first, then columns (goofy_tc.h:1402-1414).
    uint32_t col[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) col[x] = avg4(avg4(p[x], p[4 + x]), avg4(p[8 + x], p[12 + x]));
    const uint32_t avgc = avg4(avg4(col[0], col[1]), avg4(col[2], col[3]));
    // Shift its brightness onto mid (goofy_tc.h:1431-1449).
    uint32_t w0 = etc1_base_bytes(avgc, c.s.mid);
    const uint32_t cw = etc1_table(c.s.range);
    w0 |= ((cw << 5) | (cw << 2) | 3u) << 24;
    return make_uint2(w0, w1);
}

template <int FMT>
__device__ __forceinline__ uint2 encode_block(const uint32_t (&p)[16])
{
    if constexpr (FMT == kDXT1) return encode_dxt1(p);
    else return encode_etc1(p);
}

// ---- alpha blocks (DXT5 / ETC2 RGBA8) ---------------------------------------
// The reference has no alpha encoder; its README names one that works on
// alpha directly instead of brightness as the next step.  This one does that
// with the same byte arithmetic as the colour blocks:
//   * min/max alpha of the block;
//   * the 8 palette levels in ascending order, exactly as a decoder forms
//     them (Src/decoder.cpp:25-42 EAC tables, :874-896 BC3 palette);
//   * per pixel, its rank among the levels = the number of midpoints
//     ceil((lv[k-1] + lv[k]) / 2) it reaches, so every pixel takes the level
//     nearest to it and a pixel exactly between two takes the higher one;
//   * the rank's selector, packed in the format's bit order.
// BC3: a0 = max, a1 = min (8-level mode when they differ), level k =
// min + floor(k*(max-min)/7).  EAC: table 9 ({-10,-8,-5,-2,1,4,7,9} sorted),
// multiplier m = max(1, ceil((max-min)/19)) so that 19m covers the range,
// base min + 10m (lowest level on the minimum) or, when that passes 255,
// max - 9m (highest level on the maximum).

struct AlphaRows {
    uint32_t pair[8];  // the alphas of pixels 2i and 2i + 1 in the 16-bit lanes
    uint32_t w[4];     // word r: byte c = alpha of pixel (row r, column c)
    uint32_t mn, mx;
};

// Alphas of a block whose alpha range [amn, amx] is known.
__device__ __forceinline__ AlphaRows alpha_rows(const uint32_t (&p)[16], uint32_t amn, uint32_t amx)
{
    AlphaRows a;
    a.mn = amn;
    a.mx = amx;
#pragma unroll
    for (int i = 0; i < 8; ++i) a.pair[i] = perm(p[2 * i + 1], p[2 * i], 0x0c070c03u);
#pragma unroll
    for (int r = 0; r < 4; ++r) a.w[r] = perm(a.pair[2 * r + 1], a.pair[2 * r], 0x06040200u);
    return a;
}

// From the inverted ascending levels n_k = 255 - lv[k], each replicated to
// all four bytes: ~thr_k in all four bytes, thr_k = ceil((lv[k-1] + lv[k]) /
// 2).  255 - ceil(y / 2) = floor((510 - y) / 2), the floor average of n_{k-1}
// and n_k, which is v_lerp_u8 with a zero rounding operand.
__device__ __forceinline__ void rep_midpoints(const uint32_t (&r)[8], uint32_t (&nthr4)[7])
{
#pragma unroll
    for (int k = 1; k < 8; ++k) nthr4[k - 1] = __builtin_amdgcn_lerp(r[k - 1], r[k], 0u);
}

// Threshold flags of four alphas: m[k] has bit 7 of byte c set when alpha c
// reaches thr_{k+1} (f_{k+1} below); the other bits are don't-care.  The
// thresholds ascend, so the flags of a byte are a thermometer code f_1 >= f_2
// >= ... >= f_7 and its rank t (0..7) is their count.
__device__ __forceinline__ void rank_flags(uint32_t w, const uint32_t (&nthr4)[7], uint32_t (&m)[7])
{
#pragma unroll
    for (int k = 0; k < 7; ++k) m[k] = avg4(nthr4[k], w);  // avg(~t, v) >= 128 <=> v >= t
}

// Three selector bits at bit 7 of each byte -> the 3-bit selector in bits
// 5..7 of the byte (bit 2 from s2); bits 0..4 are left as don't-care.
__device__ __forceinline__ uint32_t sel3(uint32_t s2, uint32_t s1, uint32_t s0)
{
    return bsel(0x80808080u, s2, bsel(0x40404040u, s1 >> 1, s0 >> 2));
}

// The BC3 ranks of a block by one multiply-add per pixel.  With d = alpha - min
// and range R = max - min, the rank of a pixel among the 8 levels (as above:
// the number of midpoints ceil((lv[k-1] + lv[k]) / 2), lv[k] = floor(k R / 7),
// that d reaches) is the top three bits of the 16-bit number d * mul + add for
// a suitable mul and add of each R: the midpoints lie close enough to a line.
// One entry per R, from the midpoints themselves: for each of them d * mul +
// add has to reach k * 8192 there and not one step before, and 2^16 nowhere.
// lut: the selector of each rank (0 -> 1 (min), 7 -> 0 (max), 8 - t between).
//   R = 2 and R = 4 have other ranks: their few values of d take ranks of
// their own, and the entry's lut has the selectors.  R = 254 misses by little
// (bc3_alpha).
struct Bc3Entry {
    uint32_t mul, add, lut_lo, lut_hi;
};
struct Bc3Table {
    Bc3Entry e[256];
};

constexpr Bc3Table make_bc3_table()
{
    Bc3Table t{};
    for (int range = 0; range < 256; ++range) {
        Bc3Entry& e = t.e[range];
        e.lut_lo = 0x05060701u;
        e.lut_hi = 0x00020304u;
        if (range == 0) {  // one value, the maximum's selector
            e.add = 7u * 8192u;
            continue;
        }
        if (range == 2) {  // ranks 3, 6, 7, the last taken as 9 mod 8
            e.mul = e.add = 3u * 8192u;
            e.lut_lo = 0x05060001u;
            continue;
        }
        if (range == 4) {  // ranks 1, 3, 5, 6, 7, taken as 1 .. 5
            e.mul = e.add = 8192u;
            e.lut_lo = 0x03050701u;
            e.lut_hi = 0x00020002u;
            continue;
        }
        int mid[8] = {};
        for (int k = 1; k < 8; ++k) mid[k] = ((k - 1) * range / 7 + k * range / 7 + 1) / 2;
        for (int mul = range < 7 ? 8192 : 57344 / range - 24; mul < 57344 / range + 24 && !e.mul; ++mul) {
            int lo = 0, hi = 65535 - range * mul;
            for (int k = 1; k < 8; ++k) {
                if (k * 8192 - mid[k] * mul > lo) lo = k * 8192 - mid[k] * mul;
                if (mid[k] > 0 && k * 8192 - 1 - (mid[k] - 1) * mul < hi) hi = k * 8192 - 1 - (mid[k] - 1) * mul;
            }
            if (lo <= hi) {
                e.mul = (uint32_t)mul;
                e.add = (uint32_t)lo;
            }
        }
        if (range == 254) {  // right but for d = 235, 2 above the last step's 57344
            e.mul = 226u;
            e.add = 4236u;
        }
    }
    return t;
}
static __device__ const Bc3Table bc3_table = make_bc3_table();

// BC3 alpha block as two little-endian words, from the block's alphas.  Nine
// instructions a row where seven threshold compares and the selector logic
// take twenty, and one 16-byte table entry instead of eight levels.  The alpha
// encoders are bound by their instructions as much as by memory (84-90% of
// their cycles issued one): with this, the lumas and the index word by dot
// products and EAC's packing in bytes, DXT5 at 8192^2 went from 53.7 to 52.3 us
// (4100x3076: 13.1 to 12.2), ETC2 RGBA8 54.5 to 53.5, both from one read 70.0
// to 65.8.
__device__ __forceinline__ uint2 bc3_alpha(const AlphaRows& a)
{
    const uint32_t range = a.mx - a.mn;
    const Bc3Entry e = bc3_table.e[range];
    const unsigned short mul = (unsigned short)e.mul, add = (unsigned short)(e.add - a.mn * e.mul);
    const u16x2 mul2 = {mul, mul}, add2 = {add, add};
    uint32_t pair[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) pair[i] = a.pair[i];
    if (__builtin_expect(range == 254u, 0)) {
        // d = 235 ranks one too high: take it as 234, which has its rank
        const unsigned short at = (unsigned short)(a.mn + 235u);
        const u16x2 at2 = {at, at}, one = {1, 1};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u16x2 v = __builtin_bit_cast(u16x2, pair[i]);
            pair[i] = __builtin_bit_cast(uint32_t, v - one + __builtin_elementwise_min(v ^ at2, one));
        }
    }
    uint32_t row[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const u16x2 t0 = __builtin_bit_cast(u16x2, pair[2 * r]) * mul2 + add2;
        const u16x2 t1 = __builtin_bit_cast(u16x2, pair[2 * r + 1]) * mul2 + add2;
        // the four ranks in bits 5..7 of the bytes, then bits 0..2: the lookup's selectors
        const uint32_t t = perm(__builtin_bit_cast(uint32_t, t1), __builtin_bit_cast(uint32_t, t0), 0x07050301u);
        const uint32_t s = perm(e.lut_hi, e.lut_lo, (t >> 5) & 0x07070707u);
        // column c at bits 3c
        row[r] = ((s >> 24) << 9) | __builtin_amdgcn_udot4(s, 0x00400801u, 0u, false);
    }
    // row r at bits 12r..12r+11 of the 48 index bits after a0, a1
    const uint32_t lo = row[0] | (row[1] << 12), hi = row[2] | (row[3] << 12);
    return make_uint2((a.mx | (a.mn << 8)) | (lo << 16), perm(hi, lo, 0x06050402u));
}

// EAC (ETC2 RGBA8 alpha) block as two little-endian words, from the block's
// alpha rows.
__device__ __forceinline__ uint2 eac_alpha(const AlphaRows& a)
{
    const uint32_t range = a.mx - a.mn;
    uint32_t m = ((range + 18u) * 3450u) >> 16;  // ceil(range / 19) for range <= 255
    m = m > 1u ? m : 1u;
    int32_t b = (int32_t)(a.mn + 10u * m);
    if (b > 255) b = (int32_t)a.mx - 9 * (int32_t)m;
    // Inverted levels 255 - clamp(b + m*s) = clamp(nb - m*s), nb = 255 - b,
    // two to a word in 16-bit lanes.  0 <= b <= 255 (the second base only
    // occurs for m <= 2 and mx > 235), so for the negative modifiers
    // nb - m*s >= 0 and only 255 bounds it, and for the positive ones
    // nb - m*s <= 255 and only 0 does: a v_pk_mad_u16 and one v_pk_min_u16,
    // or a v_pk_mul_lo_u16 and a saturating v_pk_sub_u16, per pair.
    const unsigned short nb = (unsigned short)(255 - b), ms = (unsigned short)m;
    const u16x2 nb2 = {nb, nb}, m2 = {ms, ms}, top = {255, 255};
    const u16x2 n01 = __builtin_elementwise_min(m2 * u16x2{10, 8} + nb2, top);  // modifiers -10, -8
    const u16x2 n23 = __builtin_elementwise_min(m2 * u16x2{5, 2} + nb2, top);   // -5, -2
    const u16x2 n45 = __builtin_elementwise_sub_sat(nb2, m2 * u16x2{1, 4});      // 1, 4
    const u16x2 n67 = __builtin_elementwise_sub_sat(nb2, m2 * u16x2{7, 9});      // 7, 9
    const uint32_t w[4] = {__builtin_bit_cast(uint32_t, n01), __builtin_bit_cast(uint32_t, n23),
                           __builtin_bit_cast(uint32_t, n45), __builtin_bit_cast(uint32_t, n67)};
    uint32_t nlv4[8];  // level k's byte in all four bytes
#pragma unroll
    for (int k = 0; k < 8; ++k) nlv4[k] = perm(0u, w[k >> 1], (k & 1) ? 0x02020202u : 0u);
    uint32_t nthr4[7];
    rep_midpoints(nlv4, nthr4);
    uint32_t z[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t f[7];
        rank_flags(a.w[r], nthr4, f);
        // rank t -> selector: 0..3 -> 3..0 (negative modifiers), 4..7
        // unchanged: s2 = f4, s1 = ~(f2 ^ f6), s0 = ~(f1 ^ f2 ^ f3 ^ f5 ^ f6 ^ f7)
        const uint32_t s1 = ~(f[1] ^ f[5]);
        const uint32_t s0 = ~(xor3(f[0], f[1], f[2]) ^ xor3(f[4], f[5], f[6]));
        z[r] = sel3(f[3], s1, s0);
    }
    // 48 bits, big-endian: column 0 (x = 0) first, 12 bits per column, row 0
    // in its top three.  Rows 0, 1 and 2, 3 of every column in bits 2..7 of a
    // byte; the two bytes of a column in a 16-bit lane, moved together to bits
    // 4..15; and the lanes of two columns together to bits 8..31.
    const uint32_t r01 = bsel(0xE0E0E0E0u, z[0], z[1] >> 3), r23 = bsel(0xE0E0E0E0u, z[2], z[3] >> 3);
    auto columns = [](uint32_t c) {  // c: bytes r23, r01 of the second column, then of the first
        const uint32_t q = bsel(0xFC00FC00u, c, c << 2);
        return bsel(0xFFF00000u, q, q << 4);
    };
    const uint32_t hi = columns(perm(r01, r23, 0x04000501u)), lo = columns(perm(r01, r23, 0x06020703u));
    const uint32_t head = (uint32_t)b | (((m << 4) | 9u) << 8);
    return make_uint2(perm(hi, head, 0x06070100u), perm(lo, hi, 0x05060701u));
}

// DXT5 / ETC2 RGBA8 block: {alpha words, colour words}.  One pass over the
// pixels gives the colour box and the alpha range (block_stats_alpha).
template <int FMT>
__device__ __forceinline__ uint4 encode_block16(const uint32_t (&p)[16])
{
    uint32_t amn, amx;
    const BlockStats s = block_stats_alpha(p, amn, amx);
    const AlphaRows a = alpha_rows(p, amn, amx);
    if constexpr (FMT == kDXT5) {
        const uint2 al = bc3_alpha(a), c = encode_dxt1(p, s);
        return make_uint4(al.x, al.y, c.x, c.y);
    } else {
        const uint2 al = eac_alpha(a), c = encode_etc1(p, s);
        return make_uint4(al.x, al.y, c.x, c.y);
    }
}

}  // namespace goofy_dev
