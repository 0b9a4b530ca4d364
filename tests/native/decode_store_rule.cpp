// Host check of the rule by which a decode writes its stores through
// (decode_store in internal.h): only where every wave's 64 blocks begin and end
// on 64-byte sectors, so that no two waves write parts of one, and wherever
// they do.  Prints "decode store rule ok" and exits 0.
#include <cstdio>

#include "internal.h"

using namespace goofy_impl;

int main()
{
    int failures = 0;
    for (uint32_t bw = 1; bw <= 600; ++bw)
        for (size_t pad : {0, 16, 32, 48, 64, 96, 128})
            for (uintptr_t base : {4096, 4112, 4128, 4160}) {
                const size_t pitch = (size_t)bw * 16 + pad;
                const uint32_t bh = 40;
                bool whole = true;  // every start of a wave's pixels, and every start and end of a row, on a sector
                for (uint32_t first = 0; first < bw * bh; first += 64) {
                    const uint32_t by = first / bw, bx = first % bw;
                    for (uint32_t y = 0; y < 4; ++y) whole &= (base + (by * 4 + y) * pitch + bx * 16) % 64 == 0;
                }
                for (uint32_t y = 0; y < 4 * bh; ++y)
                    whole &= (base + y * pitch) % 64 == 0 && (base + y * pitch + bw * 16) % 64 == 0;
                for (int fmt = 0; fmt < 4; ++fmt) {
                    const bool through = decode_store(fmt, bw, (const void*)base, pitch, 4 * bh) == kStreamThrough;
                    if (through != whole && failures++ < 10)
                        std::printf("FAIL bw=%u pitch=%zu base=%zu format %d: written through %d, whole sectors %d\n", bw,
                                    pitch, (size_t)base, fmt, through, whole);
                }
            }
    if (!failures) std::printf("decode store rule ok\n");
    return failures != 0;
}
