// Which kernel and tile a matrix product takes, by its sizes: the rules the
// product's translation units share.
#pragma once

#include <algorithm>

#include "common.hpp"

namespace tc {

// The sliced kernel's tile for a product: 64 x 64 where that gives at least
// half the CUs a block, else 32 x 32 where that does, else 16 x 16, and never
// a tile twice the product's smaller side.  More, smaller tiles fill the chip
// but read the operands more often (us a call): f32 768^3, 144 / 576 tiles of
// 64 / 32: 17.7 / 20.0; f32 512^3, 64 / 256: 12.6 / 5.8; f32 256 x 8192 x 256,
// 64 / 256 tiles of 32 / 16: 44 / 27; bf16 64 x 4096 x 4096 with B transposed,
// 64 / 256 / 1024 of 64 / 32 / 16: 32 / 17 / 45.
inline uint32_t sliced_tile(uint32_t m, uint32_t n) {
    const uint64_t cus = static_cast<uint64_t>(compute_units());
    const uint32_t narrow = std::min(m, n);
    for (uint32_t tile = 64; tile > 16; tile /= 2) {
        const uint64_t blocks = static_cast<uint64_t>((m + tile - 1) / tile) * ((n + tile - 1) / tile);
        if (narrow > tile / 2 && blocks * 2 >= cus) return tile;
    }
    return 16;
}

// Whether a product is small enough for the sliced kernel rather than a tiled
// one: at most a 64 x 64 tile a CU.  There a tiled kernel has a tile for one CU
// in four and takes as long as if each had one; past it the sliced kernel's
// CUs get a second tile.  us a call, tiled / sliced: 256 such tiles (1024^3) f32
// 37.4 / 22.7, bf16 10.7 / 8.5; (64 x 2048 x 16384) 67 / 38 and 27 / 15; 324
// (1152 x 1024 x 1152) 38.8 / 48.2 and 10.9 / 14.6; 384 (192 x 2048 x 8192) 67 /
// 89.  An f32 product of at most 32 rows or columns is bound by its 128-wide
// tiles' padding however long it is: 16 x 4096 x 20480 237 / 108, 32 x 2048 x
// 20480 117 / 44, 32768 x 2048 x 16 81 / 56; 16-bit ones are not (45 / 52, 25 /
// 24, 27 / 36).
inline bool small_product(uint32_t m, uint32_t n, bool f32) {
    return (f32 && std::min(m, n) <= 32) ||
           static_cast<uint64_t>((m + 63) / 64) * ((n + 63) / 64) <= static_cast<uint64_t>(compute_units());
}

// The sliced kernel addresses its operands with 32-bit byte offsets.
inline bool sliced_reach(uint64_t m, uint64_t k, uint64_t n, size_t width) {
    const uint64_t limit = uint64_t{1} << 31;
    return m * k * width < limit && k * n * width < limit;
}

// Whether an f32 product takes 128 x 64 tiles rather than 128 x 128: where that
// leaves fewer CUs waiting for the last of them.  A CU's time is its tiles' (two
// at once share its matrix cores), and a narrow tile takes a little over half a
// wide one's: 384 wide tiles are two on some CUs, 768 narrow ones three halves
// (us, wide / narrow: 4096 x 1024 x 1536 120 / 99; 2048 x 2048 x 1024, 128 wide
// tiles, 120 / 71; 4096 x 1024 x 4096 with A transposed, 1024, 236 / 271).
inline bool narrow32(uint32_t m, uint32_t n) {
    const uint64_t cus = static_cast<uint64_t>(compute_units()), rows = (m + 127) / 128;
    const uint64_t wide = rows * ((n + 127) / 128), narrow = rows * ((n + 63) / 64);
    return (narrow + cus - 1) / cus * 21 < (wide + cus - 1) / cus * 40;
}

}  // namespace tc
