// Matrix products of operands whose rows are not 16-byte aligned (an extent the
// word does not divide, or an operand at an odd address), where the register-fed
// kernel's odd loads are the slower way: each such operand is copied once to rows
// of whole 16-byte words, zeros after its own elements, and the product runs on
// the copies, C written where it belongs.
//
// The copy is bandwidth-bound and both operands' go in one launch: 5.6 us of the
// 22.3 at bf16 2047 x 1001 x 1531 (14 MB), 20.4 of 206 at 4097^3 (6.5 TB/s); it grows
// with the sides where the product grows with the sides times K.  gemm_rules.hpp
// has the lines between these, with both sides' times.

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemm_kernels.hpp"
#include "gemm_rules.hpp"

namespace tc {
namespace {

// One operand's copy: `rows` of `cols` elements to `out_rows` of `ld`.
struct Padding {
    const void* src;
    void* dst;
    uint32_t rows, cols, out_rows, words;  // words of 16 bytes a copied row holds
    DivMod words_div;
    uint32_t blocks;
};

template <typename S>
__global__ void __launch_bounds__(256) pad_kernel(Padding first, Padding second) {
    constexpr uint32_t V = 16 / sizeof(S);
    const bool one = blockIdx.x < first.blocks;
    const Padding& p = one ? first : second;
    const uint32_t block = one ? blockIdx.x : blockIdx.x - first.blocks;
    const uint32_t total = p.out_rows * p.words;
    for (uint64_t item = static_cast<uint64_t>(block) * 256 + threadIdx.x; item < total;
         item += static_cast<uint64_t>(p.blocks) * 256) {
        const uint32_t at = static_cast<uint32_t>(item), row = p.words_div.div(at), col = (at - row * p.words) * V;
        const S* src = static_cast<const S*>(p.src) + static_cast<uint64_t>(row) * p.cols + col;
        uint4 word{0, 0, 0, 0};
        if (row < p.rows) {
            if (col + V <= p.cols) {
                word = load_any_word<false>(src);
            } else {
                S v[V] = {};
                for (uint32_t e = 0; e < V; e++) {
                    if (col + e < p.cols) v[e] = src[e];
                }
                __builtin_memcpy(&word, v, 16);
            }
        }
        static_cast<uint4*>(p.dst)[at] = word;
    }
}

template <typename S>
Padding padding(const void* src, uint64_t rows, uint64_t cols, uint64_t out_rows, uint64_t ld) {
    Padding p{};
    p.src = src;
    p.rows = static_cast<uint32_t>(rows);
    p.cols = static_cast<uint32_t>(cols);
    p.out_rows = static_cast<uint32_t>(out_rows);
    p.words = static_cast<uint32_t>(ld * sizeof(S) / 16);
    p.words_div = DivMod(p.words);
    p.blocks = blocks_for(out_rows * p.words, 1);
    return p;
}

enum class Kernel { sliced, tiled, persistent };

template <typename S, typename O, bool A_KC, bool B_KC>
void launch(Kernel kernel, const S* a, const S* b, O* c, uint32_t m, uint32_t k, uint32_t n, bool accumulate,
            const PaddedStore& store, hipStream_t s) {
    if constexpr (std::is_same<S, float>::value) {
        launch_inplace32<O, A_KC, B_KC>(a, b, c, m, k, n, accumulate, s, store);
    } else if (kernel == Kernel::persistent) {
        gemm16x16_persistent_kernel<S, O, A_KC, B_KC, PaddedStore>
            <<<compute_units(), 512, 0, s>>>(a, b, c, m, n, k, accumulate, store);
    } else if (kernel == Kernel::tiled) {
        launch_direct16<S, O, A_KC, B_KC>(a, b, c, m, k, n, accumulate, s, store);
    } else if constexpr (A_KC) {
        launch_sliced<S, O, A_KC, B_KC>(a, b, c, m, k, n, accumulate, s, store);
    }
}

template <typename S, typename O>
int product(uint32_t transposed, bool accumulate, uint64_t m, uint64_t k, uint64_t n, const void* a, const void* b,
            void* c, hipStream_t s, bool* done) {
    constexpr bool kF32 = std::is_same<S, float>::value;
    constexpr uint64_t V = 16 / sizeof(S);
    const bool a_kc = transposed != TC_LEFT, b_kc = transposed == TC_RIGHT;
    const uint32_t m32 = static_cast<uint32_t>(m), n32 = static_cast<uint32_t>(n);
    const auto whole = [](uint64_t x, uint64_t step) { return (x + step - 1) / step * step; };
    const uint64_t rows_a = a_kc ? m : k, cols_a = a_kc ? k : m, rows_b = b_kc ? n : k, cols_b = b_kc ? k : n;
    const bool odd_a = cols_a % V != 0 || !aligned16(a), odd_b = cols_b % V != 0 || !aligned16(b);
    const bool along_k = (a_kc && odd_a) || (b_kc && odd_b);
    *done = false;
    Kernel kernel;
    if (!small_product(m32, n32, kF32) && worth_tiled_copies(m32, static_cast<uint32_t>(k), n32, kF32, along_k)) {
        // From a 256 x 256 tile a CU up, the persistent 16-bit kernel.
        kernel = !kF32 && ((m + 255) / 256) * ((n + 255) / 256) >= static_cast<uint64_t>(compute_units())
                     ? Kernel::persistent
                     : Kernel::tiled;
    } else if (!kF32 && along_k && worth_sliced_copies(m32, static_cast<uint32_t>(k), n32)) {
        kernel = Kernel::sliced;
    } else {
        return TC_OK;
    }
    // The persistent kernel takes whole pairs of 64-deep steps: both operands
    // copied, K rounded up with zeros.  The register-fed one reads an operand
    // across K quickly wherever its rows start.
    const bool both = kernel == Kernel::persistent;
    const uint64_t depth = both ? whole(k, 128) : k;
    const bool copy_a = both || (odd_a && (a_kc || kernel != Kernel::sliced));
    const bool copy_b = both || (odd_b && (b_kc || kernel != Kernel::sliced));
    const uint64_t lda = copy_a ? whole(a_kc ? depth : m, V) : cols_a, ldb = copy_b ? whole(b_kc ? depth : n, V) : cols_b;
    const uint64_t out_a = a_kc ? m : depth, out_b = b_kc ? n : depth;
    const uint64_t limit = uint64_t{1} << 31, bytes_a = out_a * lda * sizeof(S), bytes_b = out_b * ldb * sizeof(S);
    if (bytes_a >= limit || bytes_b >= limit) return TC_OK;
    void* made_a = nullptr;
    void* made_b = nullptr;
    if ((copy_a && tc_alloc(bytes_a, &made_a) != TC_OK) || (copy_b && tc_alloc(bytes_b, &made_b) != TC_OK)) {
        if (made_a) tc_free(made_a);
        return TC_OK;
    }
    *done = true;
    Padding pa{}, pb{};
    if (copy_a) pa = padding<S>(a, rows_a, cols_a, out_a, lda);
    if (copy_b) pb = padding<S>(b, rows_b, cols_b, out_b, ldb);
    pa.dst = made_a;
    pb.dst = made_b;
    pad_kernel<S><<<pa.blocks + pb.blocks, 256, 0, s>>>(pa, pb);
    int status = check_launch("matmul");
    if (status == TC_OK) {
        const S* from_a = static_cast<const S*>(copy_a ? made_a : a);
        const S* from_b = static_cast<const S*>(copy_b ? made_b : b);
        O* pc = static_cast<O*>(c);
        const uint32_t k32 = static_cast<uint32_t>(depth);
        const PaddedStore store{static_cast<uint32_t>(lda), static_cast<uint32_t>(ldb)};
        if (a_kc && b_kc) {
            launch<S, O, true, true>(kernel, from_a, from_b, pc, m32, k32, n32, accumulate, store, s);
        } else if (a_kc) {
            launch<S, O, true, false>(kernel, from_a, from_b, pc, m32, k32, n32, accumulate, store, s);
        } else {
            launch<S, O, false, false>(kernel, from_a, from_b, pc, m32, k32, n32, accumulate, store, s);
        }
        status = check_launch("matmul");
    }
    // Stream order keeps the copies alive until the product has run.
    if (made_a) tc_free(made_a);
    if (made_b) tc_free(made_b);
    return status;
}

}  // namespace

int padded_product(uint32_t in_dtype, uint32_t out_dtype, uint32_t transposed, bool accumulate, uint64_t m, uint64_t k,
                   uint64_t n, const void* a, const void* b, void* c, hipStream_t s, bool* done) {
    if (in_dtype == TC_F32) return product<float, float>(transposed, accumulate, m, k, n, a, b, c, s, done);
    if (in_dtype == TC_BF16) {
        if (out_dtype == TC_F32) return product<bf16_t, float>(transposed, accumulate, m, k, n, a, b, c, s, done);
        return product<bf16_t, bf16_t>(transposed, accumulate, m, k, n, a, b, c, s, done);
    }
    if (out_dtype == TC_F32) return product<_Float16, float>(transposed, accumulate, m, k, n, a, b, c, s, done);
    return product<_Float16, _Float16>(transposed, accumulate, m, k, n, a, b, c, s, done);
}

}  // namespace tc
