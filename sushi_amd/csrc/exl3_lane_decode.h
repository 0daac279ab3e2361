// The lane decoder shared by the GEMV and the GEMM: one lane's 32 codewords of a 16x16 trellis tile, from its
// aligned stream words, to 16 packed f16 weight pairs (t, t+1).  Lane chunk j of a tile holds codewords 32j..32j+31,
// the weights of output columns j and j+8 over all 16 k rows (tensorCorePerm, beamivalice/sushi
// src/exl3/expert_exl3.zig:379-398): pair i = 4qq + p covers rows 2qq + 8(p & 1) + {0, 1} of column j (p < 2) or
// j + 8 (p >= 2).
#pragma once
#include "exl3_common.cuh"

#include <type_traits>

namespace exl3 {

// Codeword v of the lane as (window index, high half?): for K = 1, 2, 4 the window ending at codeword v + 16/K
// carries codeword v in its high half, so half the windows serve two codewords.
template <int N>
struct Pairing {
    static constexpr bool ON = N == 16 || N == 32 || N == 64;
    static constexpr int STEP = ON ? 256 / N : 32;
    __device__ static constexpr bool hi(int v) { return ON && ((v / STEP) % 2 == 0); }
    __device__ static constexpr int win(int v) { return hi(v) ? v + STEP : v; }
    static constexpr int win_of(int v) { return ON && (v / STEP) % 2 == 0 ? v + STEP : v; }  // on host and device
};

// A scheduling fence: nothing moves across it, so each phase below stays one batch of independent instructions.
__device__ __forceinline__ void phase_fence() { __builtin_amdgcn_sched_barrier(0); }

// A pair of hash / pair family weights times 2^12 (exact: they are the codebook values over 4096), as the
// reconstruction returns them.  The matrix cores take them unscaled (codebook_scale).
__device__ __forceinline__ uint32_t scale_h2_4096(uint32_t v) {
    __half2 h = __builtin_bit_cast(__half2, v);
    h = __hmul2(h, __half2(__float2half(4096.0f), __float2half(4096.0f)));
    return __builtin_bit_cast(uint32_t, h);
}

// f(std::integral_constant<int, 0>) .. f(std::integral_constant<int, N - 1>): an unrolled loop whose index is a constant
// to the code it runs.
template <int N, class F>
__device__ __forceinline__ void unrolled(F f) {
    if constexpr (N > 0) {
        unrolled<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// The clean codewords cw(0) .. cw(C - 1) of a lane into c (CW: a constexpr map), in two fenced phases for the paired
// rates: the windows that hold them, then their halves.
template <int N, int C, bool MASKED, class CW>
__device__ __forceinline__ void lane_codewords(const uint32_t (&A)[LaneBits<N>::AW], const DecodeV &v, uint32_t (&c)[C],
                                               CW) {
    using P = Pairing<N>;
    if constexpr (P::ON) {
        uint32_t win[32];
        unrolled<C>([&](auto ic) __attribute__((always_inline)) {
            constexpr int u = CW::at(decltype(ic)::value);
            if constexpr (CW::first(decltype(ic)::value, P::win(u))) win[P::win(u)] = lane_codeword<N>(A, P::win(u));
        });
        phase_fence();
        unrolled<C>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value, u = CW::at(i);
            c[i] = window_codeword<MASKED, P::hi(u)>(win[P::win(u)], v);
        });
    } else {
        unrolled<C>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            c[i] = lane_codeword_clean<N, MASKED>(A, CW::at(i), v);
        });
    }
    phase_fence();
}

// Products, masks and sums of C clean codewords (consecutive ones a weight pair) into C / 2 packed pairs, in fenced
// phases: within a phase no instruction depends on another, so no result is read by the instruction right after it and
// the hazard recognizer inserts no wait states (gfx950 needs one between an SDWA write and its reader, and counts none
// for writes in asm).
template <int FAM, int C>
__device__ __forceinline__ void hash_weights(uint32_t (&c)[C], const DecodeV &v, uint32_t (&w)[C / 2]) {
#pragma unroll
    for (int i = 0; i < C; i++) c[i] = hash_product<FAM>(c[i], v);
    phase_fence();
    if constexpr (FAM == FAM_3INST) {
#pragma unroll
        for (int i = 0; i < C; i++) c[i] = hash_add<FAM>(c[i], v);
        phase_fence();
    }
#pragma unroll
    for (int i = 0; i < C; i++) c[i] = hash_halves<FAM>(c[i], v);
    phase_fence();
#pragma unroll
    for (int i = 0; i < C; i += 2) half_sum_low(w[i / 2], c[i]);
    phase_fence();
#pragma unroll
    for (int i = 0; i < C; i += 2) half_sum_high(w[i / 2], c[i + 1]);
    phase_fence();
}

// Codeword orders.  `first(i, w)`: no earlier position's window is w.
template <int N, int C, class At>
struct CodewordOrder {
    static constexpr int at(int i) { return At::at(i); }
    static constexpr bool first(int i, int win) {
        for (int q = 0; q < i; q++)
            if (Pairing<N>::win_of(At::at(q)) == win) return false;
        return true;
    }
};
struct OrderAll {  // all 32 in order
    static constexpr int at(int i) { return i; }
};
template <int G>
struct OrderGroup {  // group G of two, 16 codewords
    static constexpr int at(int i) { return 16 * G + i; }
};
template <int H, int G>
struct OrderHalf {  // group G of two of the half decode: column j + 8 H, 8 codewords
    static constexpr int at(int i) { return 2 * (2 * H + ((i >> 1) & 1) + 4 * (2 * G + (i >> 2))) + (i & 1); }
};

// The weights of the lane's chunk, unscaled for the hash / pair families (the x4096 is applied by the caller).
// The hash-product families run all 32 codewords together where the rate pairs its windows (two codewords each), else in
// two groups of 16, half the temporaries.
template <int FAM, int N, bool MASKED>
__device__ __forceinline__ void decode_weights(const uint32_t (&A)[LaneBits<N>::AW], const DecodeK &k,
                                               uint32_t (&w)[16]) {
    using P = Pairing<N>;
    if constexpr (FAM == FAM_MUL1) {
        uint32_t win[32];
#pragma unroll
        for (int v = 0; v < 32; v++) {
            if (P::win(v) == v) {
                win[v] = lane_codeword<N>(A, v);
                if constexpr (MASKED) win[v] &= k.wmask | (k.wmask << 16);
            }
        }
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t x0 = win[P::win(2 * i)], x1 = win[P::win(2 * i + 1)];
            const uint32_t c0 = P::hi(2 * i) ? x0 >> 16 : x0, c1 = P::hi(2 * i + 1) ? x1 >> 16 : x1;
            w[i] = pack_h2(decode1<FAM_MUL1>(c0, k), decode1<FAM_MUL1>(c1, k));
        }
    } else if constexpr (FAM == FAM_PAIR) {
        const DecodeV v = decode_vgprs<FAM>(k);
        // Both weights of a pair decode from the odd codeword (decodePair, expert_exl3.zig:298-301).  Two groups of eight
        // pairs: 16 codewords with both their half arrays at once took 82-86 VGPRs in the decode GEMV (67-78 in groups,
        // but for n = 24 and 40), past the 80 that keep three workgroups on a CU.  Routed + shared layer of 128 experts,
        // 2048 x 768, 32 tokens, together / in groups: n = 32 121 / 115 us, n = 48 130 / 126 us, n = 64 127 / 122 us.
        unrolled<2>([&](auto gc) __attribute__((always_inline)) {
            constexpr int g = decltype(gc)::value;
            uint32_t h0[8], h1[8];
            unrolled<8>([&](auto ic) __attribute__((always_inline)) {
                constexpr int i = decltype(ic)::value;
                h1[i] = lane_codeword_clean<N, MASKED>(A, 2 * (8 * g + i) + 1, v);
            });
            phase_fence();
#pragma unroll
            for (int i = 0; i < 8; i++) h1[i] = hash_product<FAM>(h1[i], v);
            phase_fence();
#pragma unroll
            for (int i = 0; i < 8; i++) {
                h0[i] = h1[i] & v.mask;
                h1[i] = __builtin_amdgcn_alignbit(h1[i], h1[i], 32u - k.rot) & v.flip;
            }
            phase_fence();
#pragma unroll
            for (int i = 0; i < 8; i++) half_sum_low(w[8 * g + i], h0[i]);
            phase_fence();
#pragma unroll
            for (int i = 0; i < 8; i++) half_sum_high(w[8 * g + i], h1[i]);
            phase_fence();
        });
    } else {
        const DecodeV v = decode_vgprs<FAM>(k);
        if constexpr (P::ON) {
            uint32_t c[32];
            lane_codewords<N, 32, MASKED>(A, v, c, CodewordOrder<N, 32, OrderAll>{});
            hash_weights<FAM, 32>(c, v, w);
        } else {
            unrolled<2>([&](auto gc) __attribute__((always_inline)) {
                constexpr int g = decltype(gc)::value;
                using O = OrderGroup<g>;
                uint32_t c[16], p[8];
                lane_codewords<N, 16, MASKED>(A, v, c, CodewordOrder<N, 16, O>{});
                hash_weights<FAM, 16>(c, v, p);
                unrolled<8>([&](auto ic) __attribute__((always_inline)) {
                    constexpr int i = decltype(ic)::value;
                    w[O::at(2 * i) / 2] = p[i];
                });
            });
        }
    }
}

// Half of the lane's chunk, for the hash-product families (MCG, 3INST, hash rows): the 8 weight pairs of column
// j + 8 H (pairs i with (i & 2) == 2 H, in the order 2H, 2H+1, 2H+4, 2H+5, ..., 2H+13), so two waves can share one
// chunk's decode.  Output pair q holds rows 2 (q >> 1) + 8 (q & 1) + {0, 1} of that column; unscaled.  The phases run
// over two groups of 8 codewords, so few registers are live beside a caller's accumulators.
template <int FAM, int N, bool MASKED, int H>
__device__ __forceinline__ void decode_weights_half(const uint32_t (&A)[LaneBits<N>::AW], const DecodeK &k,
                                                    uint32_t (&w)[8]) {
    static_assert(FAM != FAM_PAIR && FAM != FAM_MUL1, "the half decoder serves the hash-product families");
    const DecodeV v = decode_vgprs<FAM>(k);
    unrolled<2>([&](auto gc) __attribute__((always_inline)) {
        constexpr int g = decltype(gc)::value;
        uint32_t c[8], p[4];
        unrolled<8>([&](auto ic) __attribute__((always_inline)) {
            constexpr int i = decltype(ic)::value;
            c[i] = lane_codeword_clean<N, MASKED>(A, OrderHalf<H, g>::at(i), v);
        });
        phase_fence();
        hash_weights<FAM, 8>(c, v, p);
#pragma unroll
        for (int q = 0; q < 4; q++) w[4 * g + q] = p[q];
    });
}

// ------------------------------------------------------------------------------------------------------------
// Per-tile rates (a seeded K1 / K2 tile mix, a layout extension: the reference fixes a rate per tensor or
// per expert group, src/exl3/layout.zig:56-62, and decodes every tile at its own n with decodeTile,
// src/exl3/expert_exl3.zig:338-357).  A segment is the 8 tiles (k-tile row tk, output group s) one wave reads; they
// lie contiguous from the segment's word offset, tile o at TILED_NA halfwords when bit o of the segment's mask is set,
// else TILED_NB, so tile o starts 16 o - 8 popcount(mask below o) words in.  Each lane decodes its chunk at its own
// tile's rate.
// The lane's words of its tile: A[0..1] as load_lane_words<16> reads them (k1), else A[0..2] as load_lane_words<32>.
// `row` is the segment's wave-uniform start and lane_words its tile's offset (words); loads take the scalar-base form.
__device__ __forceinline__ void load_lane_words_tiled(const uint32_t *__restrict__ row, uint32_t lane_words, int j,
                                                      bool k1, uint32_t (&A)[3]) {
    typedef __attribute__((address_space(1))) const uint32_t global_u32;
    const char *base = reinterpret_cast<const char *>(row);
    auto at = [&](uint32_t w) __attribute__((always_inline)) {
        return *(global_u32 *)(base + (uint32_t)((lane_words + w) * 4u));
    };
    const uint32_t i0 = k1 ? (uint32_t)((j + 7) & 7) : (uint32_t)((2 * j + 15) & 15);
    const uint32_t i1 = k1 ? (uint32_t)j : (uint32_t)(2 * j);
    const uint32_t i2 = k1 ? (uint32_t)j : (uint32_t)(2 * j + 1);  // unused at n = 16 (a repeat of A[1])
    A[0] = at(i0);
    A[1] = at(i1);
    A[2] = at(i2);
}

// The lane's 16 weight pairs at its own rate.  Both rates pair codewords in 32-bit windows (Pairing<16>: window s
// ending at codeword 16 + s carries codeword s in its high half; Pairing<32>: the windows ending at codewords 8 + s
// and 16 + s (s >= 8) carry s and 8 + s), so only the window extraction depends on the rate; the products, masks and
// sums run once over 16 windows in the n = 32 arrangement (codewords 0-7 = high halves 0-7, 8-15 = low 0-7, 16-23 =
// high 8-15, 24-31 = low 8-15).  At n = 16 the middle two groups of that arrangement hold codewords 16-23 and 8-15,
// so a k1 lane swaps pairs 4-7 with 8-11 at the end.  ka / kb: the constants at n = 16 / 32.
template <int FAM, bool MASKED>
__device__ __forceinline__ void decode_weights_tiled(const uint32_t (&A)[3], bool k1, const DecodeK &ka,
                                                     const DecodeK &kb, uint32_t (&w)[16]) {
    static_assert(FAM != FAM_PAIR && FAM != FAM_MUL1, "per-tile rates serve the hash-product families");
    const uint32_t A16[2] = {A[0], A[1]};
    DecodeV v = decode_vgprs<FAM>(kb);
    if constexpr (FAM == FAM_HASH) {  // the rows differ by rate: the lane's own
        v.mult = k1 ? in_vgpr(ka.mult) : v.mult;
        v.mask = k1 ? in_vgpr(ka.mask0) : v.mask;
    }
    uint32_t win[16], c[32];
#pragma unroll
    for (int s = 0; s < 16; s++) {
        const uint32_t c16 = lane_codeword<16>(A16, 16 + s);
        const uint32_t c32 = lane_codeword<32>(A, s < 8 ? 8 + s : 16 + s);
        win[s] = k1 ? c16 : c32;
    }
    phase_fence();
    // codeword u of the n = 32 arrangement
#pragma unroll
    for (int u = 0; u < 32; u++) {
        const uint32_t x = win[u < 8 ? u : u < 16 ? u - 8 : u < 24 ? u - 8 : u - 16];
        c[u] = (u & 8) ? window_codeword<MASKED, false>(x, v) : window_codeword<MASKED, true>(x, v);
    }
    phase_fence();
    hash_weights<FAM, 32>(c, v, w);
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t a = w[4 + q], b = w[8 + q];
        w[4 + q] = k1 ? b : a;
        w[8 + q] = k1 ? a : b;
    }
}

// The mask of segment `seg` (8 bits, one per tile), read through its aligned 32-bit word so the load stays a scalar
// one (the host checks that the table is 4-byte aligned; its length, a multiple of 8, keeps the word inside it).
__device__ __forceinline__ uint32_t seg_mask(const uint8_t *k1, size_t seg) {
    const uint32_t w = reinterpret_cast<const uint32_t *>(k1)[seg >> 2];
    return (w >> (8u * (uint32_t)(seg & 3))) & 0xFFu;
}

}  // namespace exl3
