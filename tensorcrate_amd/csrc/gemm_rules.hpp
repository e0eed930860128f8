// Which kernel and tile a matrix product takes, by its sizes: the rules, and the
// launches, that the product's translation units share.
#pragma once

#include <algorithm>

#include "common.hpp"
#include "gemm_kernels.hpp"
#include "gemm_sliced.hpp"

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

// The waves that share a 16 x 16 tile's K: eight, or two where four chunks are all
// of K and there are more tiles than blocks of eight waves are resident, which
// then wait for one another (us a call, eight / two: f32 1000000 x 8 x 16 173 /
// 42, 1000000 x 32 x 16 143 / 31, bf16 1000000 x 16 x 10 157 / 41).
inline uint32_t sliced_waves(uint32_t m, uint32_t k, uint32_t n, size_t width) {
    const uint64_t tiles = static_cast<uint64_t>((m + 15) / 16) * ((n + 15) / 16);
    return k * width <= 256 && tiles > static_cast<uint64_t>(compute_units()) * 4 ? 2 : 8;
}

// Whether its grid is one a dispatch can hold, fewer than 2^32 work-items: 16 x 16
// tiles of 512 threads pass that from 2^23 tiles on (16-bit 2^27 x 8 x 3).
inline bool sliced_fits(uint32_t m, uint32_t n) {
    const uint64_t tile = sliced_tile(m, n), threads = tile == 16 ? 512 : 256;
    return ((m + tile - 1) / tile) * ((n + tile - 1) / tile) * threads <= UINT32_MAX;
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

// The 16-bit tiled kernel for products of fewer 256 x 256 tiles than CUs.  A step's
// loads take longer to land (some 0.6 us) than its matrix-core steps (0.2), so
// what bounds it is how many loads a CU keeps in flight: two blocks of two stages
// where there are tiles for that, else one block of more stages, in 128 x 64 tiles
// while those are no more than the CUs.  us a call, two stages / three / 128 x 64
// and four: 1152 x 4096 x 1152, 162 narrow tiles, 46.3 / 36.3 / 26.4 (B transposed
// 44.4 / 31.8 / 24.9); 1280 x 1024 x 1280, 200, 11.7 / 10.9 / 9.5; (B transposed) 2048^3,
// 512, 27.3 / 20.9 / 27.7; 4096 x 1024 x 2048, 1024, 21.1 / 22.5 / 29.3.  The order of
// the sums is the same in all.  A program's epilogue keeps the one shape it is
// compiled for.
template <typename S, typename O, bool A_KC, bool B_KC, class EPI = PlainStore>
void launch_direct16(const S* a, const S* b, O* c, uint32_t m, uint32_t k, uint32_t n, bool accumulate, hipStream_t s,
                     const EPI& epi = EPI{}) {
    const uint32_t cus = static_cast<uint32_t>(compute_units()), rows = (m + 127) / 128;
    const uint32_t wide = rows * ((n + 127) / 128), narrow = rows * ((n + 63) / 64);
    if constexpr (!EPI::kProgram) {
        if (narrow <= cus) {
            direct16_kernel<S, O, A_KC, B_KC, 128, 64, 2, 2, 64, 4, EPI><<<narrow, 256, 0, s>>>(a, b, c, m, n, k,
                                                                                             accumulate, epi);
            return;
        }
        if (wide <= cus) {
            direct16_kernel<S, O, A_KC, B_KC, 128, 128, 2, 2, 64, 3, EPI><<<wide, 256, 0, s>>>(a, b, c, m, n, k,
                                                                                            accumulate, epi);
            return;
        }
    }
    direct16_kernel<S, O, A_KC, B_KC, 128, 128, 2, 2, 64, 2, EPI><<<wide, 256, 0, s>>>(a, b, c, m, n, k, accumulate,
                                                                                    epi);
}

// Whether operands that the tiled kernels cannot read in place are worth
// copying for one.  us a call, register-fed kernel / copies and tiled kernel:
//  - 16-bit, an operand along K: the register-fed kernel's odd loads along K are
//    slow, and the copies' few microseconds are made up from about 2^28
//    multiplications: (A along K) 1153 x 33 x 1153 4.9 / 8.1, 2047 x 17 x 2047 9.1 /
//    10.1, 1153 x 255 x 1153 13.3 / 10.8, 2047 x 1001 x 1531 38 / 23, 4097^3 1041 /
//    206; (both) 5.6 / 8.0, 9.9 / 9.9, 19.8 / 10.5, 54 / 23, 1653 / 205.
//  - 16-bit, neither: from about 2^32: 1153 x 1025 x 1153 16.8 / 16.5, 2047 x 1001
//    x 1531 24.0 / 24.6, 1025 x 4095 x 2047 72 / 61, 4097^3 413 / 207.
//  - f32, whose matrix cores hide those loads better: where the tiles' last
//    rounds and edges leave the CUs four sevenths of a whole product's work
//    (65 x 2049 x 20481, a third: 130 / 173; 1025 x 4095 x 2047, half: 246 / 252;
//    1153 x 1025 x 1153, 0.6: 49 / 48; 2047 x 1001 x 1531, 0.75: 84 / 76; 4097^3
//    1433 / 1093), from 2^30 (1153 x 255 x 1153 16.4 / 17.5).
inline bool worth_tiled_copies(uint32_t m, uint32_t k, uint32_t n, bool f32, bool along_k) {
    const uint64_t work = static_cast<uint64_t>(m) * n * k;
    if (!f32) return work >= (along_k ? uint64_t{1} << 28 : uint64_t{1} << 32);
    const uint64_t cus = static_cast<uint64_t>(compute_units()), rows = (m + 127) / 128;
    const uint64_t wide = rows * ((n + 127) / 128), narrow = rows * ((n + 63) / 64);
    const uint64_t rounds = std::min((narrow + cus - 1) / cus * 21, (wide + cus - 1) / cus * 40);
    return work >= uint64_t{1} << 30 &&
           rounds * cus * 128 * 128 * 4 <= 7 * 40 * static_cast<uint64_t>(m) * n;
}

// Whether a small 16-bit product's odd operands along K are worth copying for the
// register-fed kernel: what the copies' few microseconds win is the chain of odd
// loads along K, which that kernel's 16 x 16 tiles cut into more pieces.  us a
// call, as they are / copied, A along K and both: 1023 x 511 x 1023 12.3 / 10.9 and
// 18.1 / 13.2, 101 x 501 x 8191 9.5 / 9.3 and 12.1 / 15.5, 700 x 701 x 699 10.6 /
// 11.0 and 14.1 / 13.2, 333 x 777 x 555 8.2 / 8.1 and 10.2 / 9.1, 511 x 1001 x 511
// 9.0 / 8.8 and 11.8 / 9.3, 1023 x 4095 x 1023 65 / 38 and 102 / 44; in 16 x 16
// tiles 255 x 1001 x 255 5.2 / 7.7 and 6.7 / 8.0, 255 x 2049 x 255 13.2 / 11.4 and
// 20.1 / 9.4, 16 x 2049 x 4097 28.7 / 22.9 and 29.5 / 14.9.
inline bool worth_sliced_copies(uint32_t m, uint32_t k, uint32_t n) {
    return k >= (sliced_tile(m, n) == 16 ? 2048 : 768);
}

// The in-place f32 kernel, in 128 x 128 or 128 x 64 tiles (`narrow32`).
template <typename O, bool A_KC, bool B_KC, class EPI = PlainStore>
void launch_inplace32(const float* a, const float* b, O* c, uint32_t m, uint32_t k, uint32_t n, bool accumulate,
                      hipStream_t s, const EPI& epi = EPI{}) {
    const uint32_t tiles = ((m + 127) / 128) * ((n + 127) / 128), narrow = ((m + 127) / 128) * ((n + 63) / 64);
    if constexpr (!EPI::kProgram) {
        if (narrow32(m, n)) {
            inplace32_kernel<O, A_KC, B_KC, 128, 64, EPI><<<narrow, kThreads, 0, s>>>(a, b, c, m, n, k, accumulate,
                                                                                     epi);
            return;
        }
    }
    inplace32_kernel<O, A_KC, B_KC, 128, 128, EPI><<<tiles, kThreads, 0, s>>>(a, b, c, m, n, k, accumulate, epi);
}

// The sliced kernel, in its tile for the product.
template <typename S, typename O, bool A_KC, bool B_KC, class EPI = PlainStore>
void launch_sliced(const S* a, const S* b, O* c, uint32_t m, uint32_t k, uint32_t n, bool accumulate, hipStream_t s,
                   const EPI& epi = EPI{}) {
    const uint32_t tile = sliced_tile(m, n);
    const uint32_t blocks = ((m + tile - 1) / tile) * ((n + tile - 1) / tile);
    if (tile == 64) {
        sliced_kernel<S, O, A_KC, B_KC, 4, 4, 4, 1, EPI><<<blocks, 256, 0, s>>>(a, b, c, m, n, k, accumulate, epi);
    } else if (tile == 32) {
        sliced_kernel<S, O, A_KC, B_KC, 2, 2, 4, 1, EPI><<<blocks, 256, 0, s>>>(a, b, c, m, n, k, accumulate, epi);
    } else if (sliced_waves(m, k, n, sizeof(S)) == 2) {
        sliced_kernel<S, O, A_KC, B_KC, 1, 1, 2, 1, EPI><<<blocks, 128, 0, s>>>(a, b, c, m, n, k, accumulate, epi);
    } else {
        sliced_kernel<S, O, A_KC, B_KC, 1, 1, 8, 4, EPI><<<blocks, 512, 0, s>>>(a, b, c, m, n, k, accumulate, epi);
    }
}

// The product as `tc_matmul` forms it, of operands the tiled kernels cannot read
// in place, which are first copied to rows of whole 16-byte words
// (gemm_padded.hip).  `*done` is false, with nothing launched, where that is not
// worth it, or the copies would pass the kernels' 2^31 bytes or have no memory.
int padded_product(uint32_t in_dtype, uint32_t out_dtype, uint32_t transposed, bool accumulate, uint64_t m, uint64_t k,
                   uint64_t n, const void* a, const void* b, void* c, hipStream_t s, bool* done);

}  // namespace tc
