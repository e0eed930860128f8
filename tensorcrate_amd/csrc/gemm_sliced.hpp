// The register-fed product kernel (`sliced_kernel`): small products, products
// with a long K over few tiles, and operands whose rows are not 16-byte
// aligned.  Shared by the library (gemm.hip) and the product kernels the
// runtime compiler builds with a program's epilogue compiled in; it includes
// only what hiprtc provides.
#pragma once

#include <type_traits>

#include "device.hpp"
#include "gemm_kernels.hpp"

namespace tc {

// `BYTES` bytes at `at`, whatever its alignment: one load instruction of
// that width (gfx950 loads words from any byte address).
template <int BYTES>
struct Word;
template <>
struct Word<2> {
    typedef uint16_t type;
};
template <>
struct Word<4> {
    typedef uint32_t type;
};
template <>
struct Word<8> {
    typedef u32x2 type;
};
template <>
struct Word<16> {
    typedef u32x4 type;
};
template <int BYTES>
__device__ __forceinline__ typename Word<BYTES>::type load_anywhere(const uint8_t* at) {
    typename Word<BYTES>::type v;
    __builtin_memcpy(&v, at, BYTES);
    return v;
}

// One operand of a wave's 16 V x kDepth chunks: V fragments of 16 rows (the
// tile's M or N index), each lane holding 16 bytes of consecutive k: lane l
// the k's (l / 16) * kLane .. of row l % 16 of each fragment.
//  - K-contiguous rows: fragment i is rows base + 16 i .. + 15, one 16-byte
//    load a lane.
//  - Row-contiguous storage: a lane loads V consecutive rows of each of its
//    kLane k's at once, so fragment i is rows base + V x + i, x = 0 .. 15,
//    and 16-bit values are paired along k in registers (v_perm_b32).
// Rows past the operand repeat its last ones; `owned` says which results a
// lane stands for.  `rows` is at least V where the storage is row-contiguous.
template <typename S, bool KC, int V>
struct SlicedOperand {
    static constexpr int kSize = sizeof(S);
    static constexpr int kLane = 16 / kSize;
    static constexpr int kDepth = 4 * kLane;
    // A chunk as loaded: the fragments themselves, or V values of each k.
    typedef typename std::conditional<KC, uint4, typename Word<(KC ? 16 : V * kSize)>::type>::type Raw;
    static constexpr int kRaw = KC ? V : kLane;
    const uint8_t* bytes;
    uint32_t base, rows, row_bytes;
    uint32_t offset[KC ? V : 1];
    uint32_t lane_k;

    __device__ __forceinline__ uint32_t row(int i, uint32_t x) const {
        if constexpr (KC) return base + 16 * i + x;
        return min(base + V * x, rows - V) + i;
    }
    __device__ __forceinline__ bool owned(int i, uint32_t x) const {
        const uint32_t r = row(i, x);
        if constexpr (KC) return r < rows;
        return r >= base + V * x;
    }
    __device__ __forceinline__ void init(const S* p, uint32_t first, uint32_t count, uint32_t ld, uint32_t lane) {
        bytes = reinterpret_cast<const uint8_t*>(p);
        base = first, rows = count, row_bytes = ld * kSize;
        lane_k = lane / 16 * kLane;
        if constexpr (KC) {
#pragma unroll
            for (int i = 0; i < V; i++) offset[i] = min(row(i, lane % 16), rows - 1) * row_bytes + lane_k * kSize;
        } else {
            offset[0] = lane_k * row_bytes + row(0, lane % 16) * kSize;
        }
    }
    // The chunk at k0, all of it inside K.
    __device__ __forceinline__ void load(Raw (&raw)[kRaw], uint32_t k0) const {
        if constexpr (KC) {
            const uint8_t* from = bytes + k0 * kSize;
#pragma unroll
            for (int i = 0; i < V; i++) raw[i] = __builtin_bit_cast(uint4, load_anywhere<16>(from + offset[i]));
        } else {
            const uint8_t* from = bytes + static_cast<uint64_t>(k0) * row_bytes;
#pragma unroll
            for (int r = 0; r < kLane; r++) {
                raw[r] = load_anywhere<V * kSize>(from + static_cast<uint64_t>(r) * row_bytes + offset[0]);
            }
        }
    }
    // The chunk at k0, its k's from K on zero.
    __device__ __forceinline__ void load_edge(uint4 (&fragment)[V], uint32_t k0, uint32_t K) const {
        typedef typename std::conditional<kSize == 2, uint16_t, uint32_t>::type Bits;
#pragma unroll
        for (int i = 0; i < V; i++) {
            Bits value[kLane];
#pragma unroll
            for (int r = 0; r < kLane; r++) {
                const uint32_t k = k0 + lane_k + r;
                const uint64_t at = KC ? static_cast<uint64_t>(k0 + r) * kSize + offset[KC ? i : 0]
                                       : static_cast<uint64_t>(k0 + r) * row_bytes + offset[0] + i * kSize;
                value[r] = 0;
                if (k < K) value[r] = load_anywhere<kSize>(bytes + at);
            }
            __builtin_memcpy(&fragment[i], value, 16);
        }
    }
    __device__ static __forceinline__ uint32_t part(const Raw& word, int d) {
        if constexpr (sizeof(Raw) <= 4) {
            return word;
        } else {
            return word[d];
        }
    }
    // The fragments of a chunk.
    __device__ static __forceinline__ void arrange(uint4 (&fragment)[V], const Raw (&raw)[kRaw]) {
        uint32_t out[V][4];
        if constexpr (KC) {
#pragma unroll
            for (int i = 0; i < V; i++) fragment[i] = raw[i];
            return;
        } else if constexpr (kSize == 4) {
#pragma unroll
            for (int i = 0; i < V; i++)
#pragma unroll
                for (int r = 0; r < 4; r++) out[i][r] = part(raw[r], i);
        } else if constexpr (V == 1) {
#pragma unroll
            for (int r = 0; r < 4; r++) out[0][r] = raw[2 * r] | static_cast<uint32_t>(raw[2 * r + 1]) << 16;
        } else {
#pragma unroll
            for (int d = 0; d < V / 2; d++) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const uint32_t even = part(raw[2 * r], d), odd = part(raw[2 * r + 1], d);
                    out[2 * d][r] = __builtin_amdgcn_perm(odd, even, 0x05040100);
                    out[2 * d + 1][r] = __builtin_amdgcn_perm(odd, even, 0x07060302);
                }
            }
        }
#pragma unroll
        for (int i = 0; i < V; i++) fragment[i] = make_uint4(out[i][0], out[i][1], out[i][2], out[i][3]);
    }
};

// One chunk's matrix-core steps for one 16 x 16 tile.
template <typename S>
__device__ __forceinline__ f32x4 sliced_step(const uint4& a, const uint4& b, f32x4 c) {
    if constexpr (std::is_same<S, float>::value) {
        const f32x4 x = __builtin_bit_cast(f32x4, a), y = __builtin_bit_cast(f32x4, b);
#pragma unroll
        for (int e = 0; e < 4; e++) c = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], c, 0, 0, 0);
        return c;
    } else {
        return Mfma16x16<S>::step(a, b, c);
    }
}

// Two wait states between what wrote these fragments and the matrix-core step
// that reads them.  gfx950 needs them after any vector instruction; the
// compiler counts them, but not (ROCm 7.2) where that step begins a basic
// block entered by falling through from the write: the step then read the
// last register's old value.  Written into the data flow, they hold there.
template <int VA, int VB>
__device__ __forceinline__ void settle(uint4 (&fa)[VA], uint4 (&fb)[VB]) {
    u32x4 v[8] = {};
    static_assert(VA + VB <= 8, "the fragments of one chunk");
#pragma unroll
    for (int i = 0; i < VA; i++) v[i] = __builtin_bit_cast(u32x4, fa[i]);
#pragma unroll
    for (int j = 0; j < VB; j++) v[VA + j] = __builtin_bit_cast(u32x4, fb[j]);
    if constexpr (VA + VB <= 2) {
        asm volatile("s_nop 1" : "+v"(v[0]), "+v"(v[1]));
    } else if constexpr (VA + VB <= 4) {
        asm volatile("s_nop 1" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
    } else {
        asm volatile("s_nop 1" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]),
                     "+v"(v[7]));
    }
#pragma unroll
    for (int i = 0; i < VA; i++) fa[i] = __builtin_bit_cast(uint4, v[i]);
#pragma unroll
    for (int j = 0; j < VB; j++) fb[j] = __builtin_bit_cast(uint4, v[VA + j]);
}

// C[M x N] (+)= A . B on 16 VA x 16 VB tiles, operands in the layout they are
// stored in, a block a tile.  Its W waves each compute the whole tile over
// every W-th piece of K: U chunks at a time, loaded straight into the matrix
// cores' registers one turn ahead of their use, with no LDS and no barrier
// until the waves' sums are added through LDS, in their order.
//
// What bounds a small product is the chain of steps along K and how many
// compute units get a tile: the tiled kernels' 128-wide tiles give a 512^3
// product 32 blocks of 16 steps, each a load, a barrier and a wait.  Here the
// tile is small enough for a block a compute unit, and K's chain is cut by W.
// Measured (us a call, with the launch, tiled kernel before / this one):
// f32 512^3 24.2 / 5.8, f32 1024^3 44.9 / 22.4, f32 256 x 8192 x 256 327 / 27,
// bf16 1024^3 14.8 / 9.3, bf16 16 x 4096 x 4096 with B transposed 42.4 / 11.1;
// operands whose rows are not 16-byte aligned, which the tiled kernels cannot
// read: f32 1153 x 255 x 1153 16.4 (17.5 with copies), bf16 1023 x 255 x 1023 8.4
// (9.1).  At 2048 x 1024 x 1536
// aligned it is past its range: bf16 15.5 / 21.8, the waves' rereading of
// their operands from L2 then costing more than the tiled kernel's barriers.
template <typename S, typename O, bool A_KC, bool B_KC, int VA, int VB, int W, int U, class EPI = PlainStore>
__global__ void __launch_bounds__(W * 64) sliced_kernel(const S* __restrict__ A, const S* __restrict__ B,
                                                        O* __restrict__ C, uint32_t M, uint32_t N, uint32_t K,
                                                        bool accumulate, EPI epi) {
    using OA = SlicedOperand<S, A_KC, VA>;
    using OB = SlicedOperand<S, B_KC, VB>;
    constexpr uint32_t kDepth = OA::kDepth;
    __shared__ f32x4 shares[W][VA * VB][64];
    uint32_t tm, tn;
    tile_of(blockIdx.x, (M + 16 * VA - 1) / (16 * VA), (N + 16 * VB - 1) / (16 * VB), tm, tn);
    const uint32_t lane = threadIdx.x % 64;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    OA a;
    OB b;
    a.init(A, tm * 16 * VA, M, row_a(epi, A_KC ? K : M), lane);
    b.init(B, tn * 16 * VB, N, row_b(epi, B_KC ? K : N), lane);

    f32x4 acc[VA][VB];
#pragma unroll
    for (int i = 0; i < VA; i++)
#pragma unroll
        for (int j = 0; j < VB; j++) acc[i][j] = f32x4{};
    auto multiply = [&](const uint4(&fa)[VA], const uint4(&fb)[VB]) {
#pragma unroll
        for (int i = 0; i < VA; i++)
#pragma unroll
            for (int j = 0; j < VB; j++) acc[i][j] = sliced_step<S>(fa[i], fb[j], acc[i][j]);
    };

    // This wave's turns: its U-chunk pieces of K, W apart.
    const uint32_t turns = K / (kDepth * U);
    const uint32_t mine = turns > wave ? (turns - wave + W - 1) / W : 0;
    typename OA::Raw ra[2][U][OA::kRaw];
    typename OB::Raw rb[2][U][OB::kRaw];
    auto load = [&](int slot, uint32_t i) {
        const uint32_t k0 = (wave + i * W) * (U * kDepth);
#pragma unroll
        for (int u = 0; u < U; u++) {
            a.load(ra[slot][u], k0 + u * kDepth);
            b.load(rb[slot][u], k0 + u * kDepth);
        }
        __builtin_amdgcn_sched_barrier(0);  // the loads first, then what waits for the ones before
    };
    auto compute = [&](int slot) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            uint4 fa[VA], fb[VB];
            OA::arrange(fa, ra[slot][u]);
            OB::arrange(fb, rb[slot][u]);
            if constexpr (sizeof(S) == 2 && !(A_KC && B_KC)) settle(fa, fb);
            multiply(fa, fb);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    if (mine > 0) {
        load(0, 0);
        for (uint32_t i = 0; i + 1 < mine; i += 2) {
            load(1, i + 1);
            compute(0);
            load(0, min(i + 2, mine - 1));  // after the last pair: a harmless reload
            compute(1);
        }
        if (mine % 2 != 0) compute(0);
    }
    // What is left of K, chunk by chunk over the waves.
    uint32_t chunk = turns * U;
    for (uint32_t k0 = chunk * kDepth; k0 < K; k0 += kDepth, chunk++) {
        if (chunk % W != wave) continue;
        uint4 fa[VA], fb[VB];
        if (k0 + kDepth <= K) {
            a.load(ra[0][0], k0);
            b.load(rb[0][0], k0);
            OA::arrange(fa, ra[0][0]);
            OB::arrange(fb, rb[0][0]);
        } else {
            a.load_edge(fa, k0, K);
            b.load_edge(fb, k0, K);
        }
        settle(fa, fb);
        multiply(fa, fb);
    }

#pragma unroll
    for (int i = 0; i < VA; i++)
#pragma unroll
        for (int j = 0; j < VB; j++) shares[wave][i * VB + j][lane] = acc[i][j];
    __syncthreads();
    // A row of 16 x 16 tiles a wave: lane l holds, of each, column l % 16 and
    // rows 4 (l / 16) + e by the fragments' own indexes.
    for (uint32_t i = wave; i < VA; i += W) {
        f32x4 v[VB];
#pragma unroll
        for (int j = 0; j < VB; j++) {
            v[j] = shares[0][i * VB + j][lane];
#pragma unroll
            for (int w = 1; w < W; w++) v[j] += shares[w][i * VB + j][lane];
        }
        const uint32_t x = lane % 16, y = lane / 16 * 4;
        if constexpr (EPI::kProgram) {
            constexpr int E = EPI::kElems;
            static_assert(4 * VB % E == 0, "whole groups of elements");
#pragma unroll
            for (int q = 0; q < 4 * VB; q += E) {
                bool live[E];
                uint32_t rows[E], cols[E];
                float product[E];
#pragma unroll
                for (int n = 0; n < E; n++) {
                    const int e = (q + n) / VB, j = (q + n) % VB;
                    rows[n] = a.row(i, y + e), cols[n] = b.row(j, x);
                    live[n] = a.owned(i, y + e) && b.owned(j, x);
                    product[n] = v[j][e];
                }
                epi.group(live, rows, cols, N, product);
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                if (!a.owned(i, y + e)) continue;
                O* to = C + static_cast<uint64_t>(a.row(i, y + e)) * N;
                if (!B_KC && !accumulate && b.owned(0, x)) {
                    // V consecutive columns in one store.
                    O out[VB];
#pragma unroll
                    for (int j = 0; j < VB; j++) out[j] = Elem<O>::narrow(v[j][e]);
                    __builtin_memcpy(to + b.row(0, x), out, sizeof(out));
                    continue;
                }
#pragma unroll
                for (int j = 0; j < VB; j++) {
                    if (b.owned(j, x)) store_out(to, b.row(j, x), v[j][e], accumulate);
                }
            }
        }
    }
}

}  // namespace tc
