// Trellis encoder search on the GPU: the two-pass tail-biting Viterbi of src/encoder/encode.zig:170-309
// (`Encoder.encodeTile` / `packStates`), one 16x16 tile per search, T tiles per workgroup.
//
// Per step the search scores every codeword of the window once per tile: cw = (fresh << kr) | e over the
// 2^(w - k_next) edges e (the bits the next codeword keeps) and the 2^k_next fresh high bits, error
// fma(value(cw) - x, value(cw) - x, cost[cw >> k]) in f32 against the f16 path cost of its predecessor, and keeps per
// edge the first minimum as an f16 cost and a one-byte backpointer.  The arithmetic is the reference's, so the codes
// are the same: f32 squared error fused with the predecessor's cost, f16 path costs clamped at 65504, first minimum.
//
// Layout: the workgroup's threads own edges; each thread decodes a codeword once and scores it for all T tiles of the
// workgroup, so the decode is shared.  The two cost rows of every tile live in LDS (T x 2 x 2^(w - kmin) halves); the
// backpointers (256 x 2^(w - kmin) bytes per tile) go to the caller's workspace, one slot per workgroup, and are
// walked back by one lane per tile.  Codeword values are decoded on the fly (decode1), bit-exact with the engine's.
#include "exl3_kernels.h"

// The f64 squared error is summed term by term as the reference does; no multiply-add contraction in this file
// (the path costs' fused multiply-add is written out as fmaf).
#pragma clang fp contract(off)

namespace exl3 {

namespace {

constexpr int ENC_THREADS = 512;
constexpr float H_INF = 65504.0f;

__device__ __forceinline__ int fresh_bits(int n, int t) {
    return (((t + 1) * n) >> 4) - ((t * n) >> 4);
}

// tensorCorePerm (src/exl3/expert_exl3.zig:379-398): trellis index i -> row-major tile position.
__device__ __forceinline__ int tensor_core_perm(int i) {
    const int lane = i >> 3, j = i & 7;
    const int r0 = (lane & 3) * 2, c0 = lane >> 2;
    const int r = r0 + (j & 1) + ((j & 2) ? 8 : 0);
    return r * 16 + c0 + (j >= 4 ? 8 : 0);
}

__device__ __forceinline__ uint16_t f32_to_f16_bits(float v) { return __half_as_ushort(__float2half_rn(v)); }
__device__ __forceinline__ float f16_bits_to_f32(uint16_t h) { return __half2float(__ushort_as_half(h)); }

// One step of the search for all T tiles: scores every codeword, writes each edge's minimum and backpointer.  The first
// step, which has no predecessor's cost, is a body of its own (FIRST): with its branch in the scoring loop, a dozen
// instructions a score, the loop's time hung on where the compiler happened to place it (two builds of the same loop
// 2 - 8% apart).  MCG, branch in the loop (those two builds) / a body of its own: n = 80 w = 12, 64 tiles 1430 - 1535 /
// 1175 us, 1024 tiles 4300 - 4350 / 1890 us; n = 40 w = 15, 2048 tiles 13.5 - 13.9 / 10.9 ms; n = 24 w = 16, 256 tiles
// 7.4 - 7.7 / 6.0 ms.
template <int FAM, int T, bool FIRST>
__device__ __forceinline__ void search_step(int ri, int n, int w, const DecodeK &dk, const float *xs,
                                            const uint16_t *prev, uint16_t *curr, uint8_t *back, size_t back_tile,
                                            int stride, bool pinned, const int *pin) {
    const int k = fresh_bits(n, ri);
    const int k_next = fresh_bits(n, (ri + 1) & 255);
    const int kr = w - k_next;
    const int edges = 1 << kr;
    const int kk = 1 << k_next;
    float target[T];
#pragma unroll
    for (int t = 0; t < T; t++) target[t] = xs[t * 256 + ri];
    uint8_t *row = back + (size_t)ri * stride;
    for (int e = threadIdx.x; e < edges; e += ENC_THREADS) {
        float best[T];
        int bf[T];
#pragma unroll
        for (int t = 0; t < T; t++) { best[t] = H_INF; bf[t] = 0; }
        for (int fresh = 0; fresh < kk; fresh++) {
            const uint32_t cw = ((uint32_t)fresh << kr) | (uint32_t)e;
            const uint32_t pred = cw >> k;
            const float v = __half2float(decode1<FAM>(cw, dk));
#pragma unroll
            for (int t = 0; t < T; t++) {
                const float dh = v - target[t];
                float err;
                if constexpr (FIRST) {
                    if (pinned && (int)pred != pin[t]) {
                        err = H_INF;
                    } else {
                        const float sq = dh * dh;
                        err = sq < H_INF ? sq : H_INF;
                    }
                } else {
                    err = __builtin_fmaf(dh, dh, f16_bits_to_f32(prev[t * 2 * stride + pred]));
                }
                if (err < best[t]) { best[t] = err; bf[t] = fresh; }
            }
        }
#pragma unroll
        for (int t = 0; t < T; t++) {
            curr[t * 2 * stride + e] = f32_to_f16_bits(best[t]);
            row[t * back_tile + e] = (uint8_t)bf[t];
        }
    }
}

// A workgroup's paths to its outputs: packed codes, and where asked the squared error and the decoded values.
template <int FAM>
__device__ __forceinline__ void write_outputs(int T, int n, const DecodeK &dk, int64_t tile0, int64_t count,
                                              const uint16_t *path, uint32_t *words, const float *xs,
                                              uint16_t *__restrict__ packed, double *__restrict__ sse,
                                              float *__restrict__ recon) {
    const int tid = threadIdx.x;
    // packStates: step t's fresh k bits (the state's low bits), MSB first, end at bitEnd(t) of a stream read as
    // 32-bit words whose bit 31 comes first; stored little-endian, a word is the halfword pair (lo, hi).
    for (int i = tid; i < T * 64; i += ENC_THREADS) words[i] = 0u;
    __syncthreads();
    for (int i = tid; i < T * 256; i += ENC_THREADS) {
        const int t = i >> 8, s = i & 255;
        const int k = fresh_bits(n, s);
        const int end = ((s + 1) * n) >> 4;
        const uint32_t field = (uint32_t)path[i] & ((1u << k) - 1u);
        const int p0 = end - k;
        const int j0 = p0 >> 5, o0 = p0 & 31;
        if (o0 + k <= 32) {
            atomicOr(&words[t * 64 + j0], field << (32 - o0 - k));
        } else {
            const int hi = 32 - o0;  // bits in the first word
            atomicOr(&words[t * 64 + j0], field >> (k - hi));
            atomicOr(&words[t * 64 + j0 + 1], field << (32 - (k - hi)));
        }
    }
    __syncthreads();
    for (int i = tid; i < T * (n / 2); i += ENC_THREADS) {
        const int t = i / (n / 2), j = i % (n / 2);
        if (tile0 + t < count) {
            const uint32_t v = words[t * 64 + j];
            packed[(tile0 + t) * n + 2 * j] = (uint16_t)(v & 0xFFFFu);
            packed[(tile0 + t) * n + 2 * j + 1] = (uint16_t)(v >> 16);
        }
    }
    // The values the decoder will produce, back in row-major tile order.
    if (recon != nullptr)
        for (int i = tid; i < T * 256; i += ENC_THREADS) {
            const int t = i >> 8, j = i & 255;
            if (tile0 + t < count)
                recon[(tile0 + t) * 256 + tensor_core_perm(j)] = __half2float(decode1<FAM>(path[i], dk));
        }
    // The path's squared error in f64, summed in trellis order as the reference does.
    if (sse != nullptr && tid < T && tile0 + tid < count) {
        double acc = 0.0;
        for (int i = 0; i < 256; i++) {
            const double d = (double)xs[tid * 256 + i] - (double)__half2float(decode1<FAM>(path[tid * 256 + i], dk));
            acc += d * d;
        }
        sse[tile0 + tid] = acc;
    }
}

template <int FAM, int T>
__global__ __launch_bounds__(ENC_THREADS) void encode_search_kernel(const float *__restrict__ tiles, int64_t count,
                                                                    int n, int w, DecodeK dk,
                                                                    uint16_t *__restrict__ packed,
                                                                    double *__restrict__ sse,
                                                                    float *__restrict__ recon,
                                                                    uint8_t *__restrict__ back_ws, int stride) {
    extern __shared__ __align__(16) unsigned char enc_lds[];
    // LDS: cost rows [T][2][stride] u16, then x [T][256] f32, paths [T][256] u16, packed words [T][64] u32,
    // the final-edge reduction [ENC_THREADS / 64][T] u32 and the pins [T].
    uint16_t *costs = reinterpret_cast<uint16_t *>(enc_lds);
    float *xs = reinterpret_cast<float *>(enc_lds + (size_t)T * 2 * stride * 2);
    uint16_t *path = reinterpret_cast<uint16_t *>(xs + T * 256);
    uint32_t *words = reinterpret_cast<uint32_t *>(path + T * 256);
    uint32_t *red = words + T * 64;
    int *pin = reinterpret_cast<int *>(red + (ENC_THREADS / 64) * T);

    const size_t back_tile = (size_t)256 * stride;
    uint8_t *back = back_ws + (size_t)blockIdx.x * T * back_tile;
    const int64_t batches = (count + T - 1) / T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    for (int64_t b = blockIdx.x; b < batches; b += gridDim.x) {
        const int64_t tile0 = b * T;
        // Inputs, permuted into trellis order (tensorCorePerm): x[i] = tile[perm[i]].
        for (int i = tid; i < T * 256; i += ENC_THREADS) {
            const int t = i >> 8, j = i & 255;
            const int64_t tile = tile0 + t < count ? tile0 + t : count - 1;
            xs[i] = tiles[tile * 256 + tensor_core_perm(j)];
        }
        __syncthreads();
        for (int pass = 0; pass < 2; pass++) {
            const int roll = pass == 0 ? 128 : 0;
            int cur = 0;
            for (int step = 0; step < 256; step++) {
                const int ri = (step + roll) & 255;
                const uint16_t *prev = costs + cur * stride;
                uint16_t *curr = costs + (cur ^ 1) * stride;
                if (step == 0)
                    search_step<FAM, T, true>(ri, n, w, dk, xs, prev, curr, back, back_tile, stride, pass == 1, pin);
                else
                    search_step<FAM, T, false>(ri, n, w, dk, xs, prev, curr, back, back_tile, stride, pass == 1, pin);
                cur ^= 1;
                __syncthreads();
            }
            // The edge the traceback starts from: pass 0 the first cheapest final edge (an f16 cost is >= 0, so its
            // bits order as the values do and (bits << 16 | edge) orders by cost, then edge); pass 1 the pin.
            if (pass == 0) {
                const int final_edges = 1 << (w - fresh_bits(n, 0));
#pragma unroll
                for (int t = 0; t < T; t++) {
                    uint32_t key = 0xFFFFFFFFu;
                    for (int e = tid; e < final_edges; e += ENC_THREADS) {
                        const uint32_t c = costs[t * 2 * stride + cur * stride + e];
                        const uint32_t kv = (c << 16) | (uint32_t)e;
                        key = kv < key ? kv : key;
                    }
                    for (int off = 32; off > 0; off >>= 1) {
                        const uint32_t o = (uint32_t)__shfl_xor((int)key, off);
                        key = o < key ? o : key;
                    }
                    if (lane == 0) red[wave * T + t] = key;
                }
                __syncthreads();
                if (tid < T) {
                    uint32_t key = 0xFFFFFFFFu;
                    for (int v = 0; v < ENC_THREADS / 64; v++) key = red[v * T + tid] < key ? red[v * T + tid] : key;
                    pin[tid] = (int)(key & 0xFFFFu);
                }
                __syncthreads();
            }
            // Traceback, one lane per tile.
            if (tid < T) {
                const int t = tid;
                int edge = pin[t];
                const uint8_t *bt = back + (size_t)t * back_tile;
                for (int step_i = 255; step_i >= 0; step_i--) {
                    const int ri = (step_i + roll) & 255;
                    const int k = fresh_bits(n, ri);
                    const int kr = w - fresh_bits(n, (ri + 1) & 255);
                    const int state = ((int)bt[(size_t)ri * stride + edge] << kr) | edge;
                    edge = state >> k;
                    if (pass == 1) {
                        path[t * 256 + ri] = (uint16_t)state;
                    } else if (ri == 0) {
                        break;
                    }
                }
                pin[t] = edge;
            }
            __syncthreads();
        }
        write_outputs<FAM>(T, n, dk, tile0, count, path, words, xs, packed, sse, recon);
        __syncthreads();
    }
}

// The uniform search, for rates whose steps all take the same K = 2, 3 or 4 fresh bits (n = 32, 48, 64).
//
// Bound: the VALU.  Every step scores the same codewords, and the 2^K edges of a group (e >> K equal) share the 2^K
// predecessors fresh << (kr - K) | e >> K.  So a thread owns B blocks of NE consecutive edges of a group for the whole
// search: their NE x 2^K values are decoded once, into VGPRs, a predecessor's cost is read and widened once for NE
// edges, and what is left per score is a subtract, a multiply-add and the selection: with four edges, 6.2 instructions a
// score in the compiled loop, 3.6 in the steps without backpointers, each score's share of the reads and addresses
// included.  4096 tiles at n = 32, w = 12, MCG: 2.13 ms by the general search, 1.20 ms here.  Where the blocks are fewer
// than the threads, the threads split into sets that take the tiles in turn.  Only the steps that a traceback walks keep
// backpointers: the first half of pass 0 takes minima alone.
//
// A block's backpointers, NE * K bits, are a byte: a step's row is a quarter byte an edge (2 bits) or half (3 and 4
// bits; a half and one with a single tile a workgroup at 12 bits).  The traceback reads rows in chunks that half a wave
// copies to LDS (the cost rows are dead by then), the next chunk in flight while the half wave walks this one, its lanes
// in step along the one path: a lane that followed the chain through memory waited its latency 384 times.
//
// Step 0 has no predecessor: pass 0 starts from zero costs, pass 1 from zero at the pinned edge and 65504 elsewhere,
// whose scores never beat the starting 65504 (as the reference's: no such edge has a backpointer or a lower cost).
constexpr int CHUNK_BYTES = 2048;  // a tile's backpointer rows copied to LDS at a time: 32 or 64 bytes a lane

template <int NE, int K, int B, bool BACK>
__device__ __forceinline__ void uniform_step(const float (&v)[B][1 << K][NE], const float *xs, int ri, int T, int set,
                                             int sets, int block, const uint16_t *prev, uint16_t *curr, int stride,
                                             int pstep, uint8_t *row, size_t back_tile) {
    constexpr int KK = 1 << K;
    for (int t = set; t < T; t += sets) {
        const float target = xs[t * 256 + ri];
#pragma unroll
        for (int b = 0; b < B; b++) {
            const int blk = block + b * ENC_THREADS;
            const uint16_t *pc = prev + (size_t)t * 2 * stride + ((blk * NE) >> K);
            float best[NE];
            uint32_t bf[NE];
#pragma unroll
            for (int f = 0; f < KK; f++) {
                const float pcost = f16_bits_to_f32(pc[f * pstep]);
#pragma unroll
                for (int j = 0; j < NE; j++) {
                    const float dh = v[b][f][j] - target;
                    const float err = __builtin_fmaf(dh, dh, pcost);
                    if (f == 0) {
                        best[j] = __builtin_fminf(H_INF, err);
                        bf[j] = 0;
                    } else {
                        if (BACK) bf[j] = err < best[j] ? (uint32_t)f : bf[j];
                        best[j] = __builtin_fminf(best[j], err);
                    }
                }
            }
            uint16_t h[NE];
            uint32_t bits = 0;
#pragma unroll
            for (int j = 0; j < NE; j++) {
                h[j] = f32_to_f16_bits(best[j]);
                bits |= bf[j] << (K * j);
            }
            __builtin_memcpy(__builtin_assume_aligned(curr + (size_t)t * 2 * stride + blk * NE, NE * 2), h, NE * 2);
            if (BACK) row[(size_t)t * back_tile + blk] = (uint8_t)bits;
        }
    }
}

// Up to 16 values a thread are bound to the 128 VGPRs of two workgroups a CU, one's barriers under the other's steps (the
// 32 values of K = 2 and 3 with two blocks fit them too).
template <int FAM, int NE, int K, int B>
__global__ __launch_bounds__(ENC_THREADS, (B * NE << K) <= 16 ? 4 : 2) void encode_uniform_kernel(
    const float *__restrict__ tiles, int64_t count, int T, int w, DecodeK dk, uint16_t *__restrict__ packed,
    double *__restrict__ sse, float *__restrict__ recon, uint8_t *__restrict__ back_ws) {
    static_assert(NE * K <= 8, "a block's backpointers are one byte");
    constexpr int KK = 1 << K;
    extern __shared__ __align__(16) unsigned char enc_lds[];
    const int kr = w - K, stride = 1 << kr, blocks = stride / NE;
    // The general kernel's LDS layout.
    uint16_t *costs = reinterpret_cast<uint16_t *>(enc_lds);
    float *xs = reinterpret_cast<float *>(enc_lds + (size_t)T * 2 * stride * 2);
    uint16_t *path = reinterpret_cast<uint16_t *>(xs + T * 256);
    uint32_t *words = reinterpret_cast<uint32_t *>(path + T * 256);
    uint32_t *red = words + T * 64;
    int *pin = reinterpret_cast<int *>(red + (ENC_THREADS / 64) * T);

    const size_t back_tile = (size_t)256 * blocks;
    uint8_t *back = back_ws + (size_t)blockIdx.x * T * 256 * stride;
    const int64_t batches = (count + T - 1) / T;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int block = B == 1 ? tid & (blocks - 1) : tid;
    const int set = B == 1 ? tid / blocks : 0, sets = B == 1 ? ENC_THREADS / blocks : 1;
    const int pstep = 1 << (kr - K);

    float v[B][KK][NE];
#pragma unroll
    for (int b = 0; b < B; b++)
#pragma unroll
        for (int f = 0; f < KK; f++)
#pragma unroll
            for (int j = 0; j < NE; j++)
                v[b][f][j] = __half2float(
                    decode1<FAM>(((uint32_t)f << kr) | (uint32_t)((block + b * ENC_THREADS) * NE + j), dk));

    // Traceback geometry: half a wave per tile (T <= 16), rows of `blocks` bytes, chunks of `rows` rows that fit the
    // tile's cost rows (1024 bytes at the narrowest, n = 64 at 12 bits).
    const int ht = tid >> 5, hl = tid & 31;
    const int chunk = 4 * stride < CHUNK_BYTES ? 4 * stride : CHUNK_BYTES;
    // Rows wider than a chunk are walked in place.
    const int rows = blocks <= chunk ? chunk / blocks : 0;

    for (int64_t bt = blockIdx.x; bt < batches; bt += gridDim.x) {
        const int64_t tile0 = bt * T;
        for (int i = tid; i < T * 256; i += ENC_THREADS) {
            const int t = i >> 8, j = i & 255;
            const int64_t tile = tile0 + t < count ? tile0 + t : count - 1;
            xs[i] = tiles[tile * 256 + tensor_core_perm(j)];
        }
        for (int pass = 0; pass < 2; pass++) {
            const int roll = pass == 0 ? 128 : 0;
            for (int i = tid; i < T << kr; i += ENC_THREADS) {
                const int t = i >> kr, e = i & (stride - 1);
                costs[t * 2 * stride + e] = pass == 0 || e == pin[t] ? 0 : 0x7BFF;
            }
            __syncthreads();
            for (int step = 0; step < 256; step++) {
                const int ri = (step + roll) & 255;
                const uint16_t *prev = costs + (step & 1) * stride;
                uint16_t *curr = costs + ((step & 1) ^ 1) * stride;
                uint8_t *row = back + (size_t)ri * blocks;
                if (pass == 0 && step < 128)
                    uniform_step<NE, K, B, false>(v, xs, ri, T, set, sets, block, prev, curr, stride, pstep, row,
                                                  back_tile);
                else
                    uniform_step<NE, K, B, true>(v, xs, ri, T, set, sets, block, prev, curr, stride, pstep, row,
                                                 back_tile);
                __syncthreads();
            }
            if (pass == 0) {  // the first cheapest final edge (256 steps: the last costs are in row 0)
                for (int t = 0; t < T; t++) {
                    uint32_t key = 0xFFFFFFFFu;
                    for (int e = tid; e < stride; e += ENC_THREADS) {
                        const uint32_t kv = ((uint32_t)costs[t * 2 * stride + e] << 16) | (uint32_t)e;
                        key = kv < key ? kv : key;
                    }
                    for (int off = 32; off > 0; off >>= 1) {
                        const uint32_t o = (uint32_t)__shfl_xor((int)key, off);
                        key = o < key ? o : key;
                    }
                    if (lane == 0) red[wave * T + t] = key;
                }
                __syncthreads();
                if (tid < T) {
                    uint32_t key = 0xFFFFFFFFu;
                    for (int u = 0; u < ENC_THREADS / 64; u++) key = red[u * T + tid] < key ? red[u * T + tid] : key;
                    pin[tid] = (int)(key & 0xFFFFu);
                }
                __syncthreads();
            }
            // Traceback of trellis steps 127 .. 0 (pass 0) or 255 .. 0 (pass 1), whose rows lie in order of ri.
            if (ht < T) {
                const uint8_t *src = back + (size_t)ht * back_tile;
                const int top = pass == 0 ? 128 : 256;
                int edge = pin[ht];
                auto walk = [&](const uint8_t *r, int ri) {
                    const int fresh = ((uint32_t)r[edge / NE] >> (K * (edge & (NE - 1)))) & (KK - 1);
                    const int state = (fresh << kr) | edge;
                    edge = state >> K;
                    if (pass == 1) path[ht * 256 + ri] = (uint16_t)state;
                };
                if (rows != 0) {
                    unsigned char *stage = enc_lds + (size_t)ht * 4 * stride;
                    uint4 q0, q1, q2, q3;  // a chunk's shares of this lane, 512 bytes apart
                    // (`two` holds for every chunk there is, 1024 bytes at the least; without the condition the compiler
                    // lays the kernel out another way and 4096 tiles at n = 32, w = 12 take 1204 us instead of 1195)
                    const bool two = chunk > 512, four = chunk > 1024;
                    auto fetch = [&](int c) {
                        const uint8_t *from = src + (size_t)c * chunk + hl * 16;
                        q0 = *reinterpret_cast<const uint4 *>(from);
                        if (two) q1 = *reinterpret_cast<const uint4 *>(from + 512);
                        if (four) q2 = *reinterpret_cast<const uint4 *>(from + 1024);
                        if (four) q3 = *reinterpret_cast<const uint4 *>(from + 1536);
                    };
                    const int chunks = top / rows;
                    fetch(chunks - 1);
                    for (int c = chunks - 1; c >= 0; c--) {
                        unsigned char *to = stage + hl * 16;
                        *reinterpret_cast<uint4 *>(to) = q0;
                        if (two) *reinterpret_cast<uint4 *>(to + 512) = q1;
                        if (four) *reinterpret_cast<uint4 *>(to + 1024) = q2;
                        if (four) *reinterpret_cast<uint4 *>(to + 1536) = q3;
                        if (c > 0) fetch(c - 1);
                        // The half wave runs in step: its stores are ordered before its own reads.
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                        for (int r = rows - 1; r >= 0; r--)
                            walk(stage + r * blocks, c * rows + r);
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                    }
                } else {
                    for (int ri = top - 1; ri >= 0; ri--) walk(src + (size_t)ri * blocks, ri);
                }
                if (hl == 0) pin[ht] = edge;
            }
            __syncthreads();
        }
        write_outputs<FAM>(T, K * 16, dk, tile0, count, path, words, xs, packed, sse, recon);
        __syncthreads();
    }
}

template <int FAM, int NE, int K, int B>
hipError_t launch_uniform(const EncodeArgs &a, hipStream_t s) {
    const size_t lds = encode_lds_bytes(a.tiles_per_wg, a.stride);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&encode_uniform_kernel<FAM, NE, K, B>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((encode_uniform_kernel<FAM, NE, K, B>), dim3((unsigned)a.grid), dim3(ENC_THREADS), lds, s,
                       a.tiles, a.count, a.tiles_per_wg, a.w, a.k, a.packed, a.sse, a.recon, a.back);
    return hipGetLastError();
}

// NE edges a thread: four at K = 2, where they are the whole group; two at K = 3 and 4, whose larger groups would take
// the VGPRs of a second workgroup (K = 3, 4 edges: 150, and 700 tiles 627 us against 407); fewer at 12 bits where one
// tile a workgroup would leave threads without edges.
template <int FAM, int K>
hipError_t launch_uniform_k(const EncodeArgs &a, hipStream_t s) {
    constexpr int NE = K == 2 ? 4 : 2;
    if constexpr (K < 4)
        if (a.tiles_per_wg == 1 && a.w == 12) return launch_uniform<FAM, K == 2 ? 2 : 1, K, 1>(a, s);
    switch (a.stride / NE / ENC_THREADS) {
    case 0:
    case 1: return launch_uniform<FAM, NE, K, 1>(a, s);
    case 2: return launch_uniform<FAM, NE, K, 2>(a, s);
    case 4: return launch_uniform<FAM, NE, K, 4>(a, s);
    default:  // 8: K = 2, 3 at a 16-bit window
        if constexpr (K < 4) return launch_uniform<FAM, NE, K, 8>(a, s);
        return hipErrorInvalidValue;
    }
}

template <int FAM, int T>
hipError_t launch_encode(const EncodeArgs &a, hipStream_t s) {
    const size_t lds = encode_lds_bytes(T, a.stride);
    if (lds > 64 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&encode_search_kernel<FAM, T>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((encode_search_kernel<FAM, T>), dim3((unsigned)a.grid), dim3(ENC_THREADS), lds, s, a.tiles,
                       a.count, a.n, a.w, a.k, a.packed, a.sse, a.recon, a.back, a.stride);
    return hipGetLastError();
}

template <int FAM>
hipError_t launch_encode_t(const EncodeArgs &a, hipStream_t s) {
    // The uniform search copies backpointer rows by 16 bytes, so it wants an aligned workspace.
    if (a.w >= 12 && a.w <= 16 && (reinterpret_cast<uintptr_t>(a.back) & 15) == 0) {
        if (a.n == 32) return launch_uniform_k<FAM, 2>(a, s);
        if (a.n == 48) return launch_uniform_k<FAM, 3>(a, s);
        if (a.n == 64) return launch_uniform_k<FAM, 4>(a, s);
    }
    switch (a.tiles_per_wg) {
    case 16: return launch_encode<FAM, 16>(a, s);
    case 8: return launch_encode<FAM, 8>(a, s);
    case 4: return launch_encode<FAM, 4>(a, s);
    case 2: return launch_encode<FAM, 2>(a, s);
    default: return launch_encode<FAM, 1>(a, s);
    }
}

}  // namespace

size_t encode_lds_bytes(int tiles_per_wg, int stride) {
    const size_t t = (size_t)tiles_per_wg;
    return t * 2 * stride * 2 + t * 256 * 4 + t * 256 * 2 + t * 64 * 4 + (ENC_THREADS / 64) * t * 4 + t * 4;
}

hipError_t run_encode(int fam, const EncodeArgs &a, hipStream_t s) {
    if (a.count == 0) return hipSuccess;
    switch (fam) {
    case FAM_MCG: return launch_encode_t<FAM_MCG>(a, s);
    case FAM_MUL1: return launch_encode_t<FAM_MUL1>(a, s);
    default: return launch_encode_t<FAM_3INST>(a, s);
    }
}

}  // namespace exl3
