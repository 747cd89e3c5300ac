// gfx950 reference-order GEMV of the halo_mi355x library (HALO_MI_GEMV_GGUF_REF): GGUF rows of any
// of the 16 types at any alignment, 8 sums per output in cpu::detail::dot's order
// (backends/cpu/kernel_common.h:16-27 of the reference), so y is bit-identical to the CPU backend.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "device.h"
#include "launch.h"

namespace halo_mi {
namespace {

using namespace dev;

// What bounds it: the CPU's order leaves 8 independent sums per output, each a chain of cols / 8
// products added one at a time, with the product rounded before its addition (no fused
// multiply-add). So the kernel is bound by vector instructions (decode, multiply, add), not by HBM.
//
// Lane l of a wave holds sum j = l % 8 of the rows l / 8 + 8 i, i < R, for NV vectors. Per chunk of
// CH elements of K:
//   - the wave brings its rows' bytes into its own piece of LDS with 16-byte loads at whatever
//     alignment the rows have (the next chunk's loads are in flight while this one is computed);
//   - the workgroup stages x in LDS by sum: element 8 s + j of a vector at [j][s], so the four
//     products of a 32-element slot that lane j takes (elements j, j + 8, j + 16, j + 24) need one
//     16-byte read; two buffers, one barrier per chunk;
//   - every weight is decoded once per launch and vector group and used for NV vectors.
// With 8 or 16 vectors a lane takes two rows, so each 16-byte read of x feeds 16 instructions: with
// one row the LDS path (8 cycles per read and CU) and the four SIMDs' 8 multiply-adds would be
// equally busy.
//
// Measured on MI355X against one thread per sum with byte loads and every weight decoded once per
// vector: IQ4_NL 5120 x 17408 at 1 vector 646 -> 62 us, Q3_K 17408 x 5120 at 64 vectors 14470 ->
// 439 us (13 T multiply-adds/s; the two rounded operations alone take about 290 us).
template <uint32_t T, int NV>
constexpr uint32_t chunk_elems() {
    // at most 640 bytes of a row and 16 x loads per thread and chunk
    uint32_t ch = NV == 1 ? 1024u : NV == 2 ? 512u : 256u;
    while (ch / block_elems(T) * block_bytes(T) > 640 && ch > 128 && ch / 2 % block_elems(T) == 0) ch /= 2;
    return ch;
}

// Threads per workgroup: single waves for few vectors (8 rows each, so 5120 rows are 640 workgroups
// over 256 CUs; four-wave workgroups would leave 96 CUs idle), four for many (they share x).
template <int NV>
constexpr uint32_t ref_threads() {
    return NV <= 4 ? 64u : 256u;
}

// The weights of elements j, j + 8, j + 16, j + 24 of slot `s` (32 elements) of the row piece `row`.
template <uint32_t T>
__device__ __forceinline__ void slot4(const uint8_t* row, uint32_t s, uint32_t j, float w[4]) {
#pragma clang fp contract(off)
    if constexpr (T == kIQ4_NL || T == kIQ4_XS) {
        // bytes j and j + 8 of the slot's 16 code bytes; four table lookups at once
        constexpr bool xs = T == kIQ4_XS;
        const uint8_t* blk = xs ? row + s / 8 * 136 : row + s * 18;
        const uint8_t* qs = xs ? blk + 8 + 16 * (s % 8) : blk + 2;
        const float d0 = h2f(*reinterpret_cast<const uint16_t*>(blk));
        float d = d0;
        if constexpr (xs)
            d = d0 * (float)iq4xs_ls(*reinterpret_cast<const uint16_t*>(blk + 2), *reinterpret_cast<const uint32_t*>(blk + 4), s % 8);
        const uint32_t q = (uint32_t)qs[j] | ((uint32_t)qs[j + 8] << 8);
        const uint32_t v = iq4_lookup4<false>((q & 0x0F0Fu) | ((q & 0xF0F0u) << 12));
#pragma unroll
        for (int k = 0; k < 4; ++k) w[k] = d * sbyte(v, k);
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) w[k] = gguf_elem<T, true>(row, 32 * s + j + 8 * k);
    }
}

// 16 bytes at p of which `avail` may be read (the others come back as zero).
__device__ __forceinline__ uint4 load_piece(const uint8_t* p, uint64_t avail) {
    uint4 v{0, 0, 0, 0};
    if (avail >= 16) {
        __builtin_memcpy(&v, p, 16);
    } else {
        uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
        for (uint32_t b = 0; b < 15; ++b)
            if (b < avail) w[b / 4] |= (uint32_t)p[b] << (8 * (b % 4));
        v = uint4{w[0], w[1], w[2], w[3]};
    }
    return v;
}

template <uint32_t T, int NV, int R>
__global__ __launch_bounds__(ref_threads<NV>()) void k_gemv_gguf_ref(const uint8_t* __restrict__ w, uint64_t w_stride,
                                                                     const float* __restrict__ x, uint64_t x_stride,
                                                                     float* __restrict__ y, uint64_t y_stride, uint32_t rows,
                                                                     uint32_t cols, uint32_t n_vec) {
#pragma clang fp contract(off)
    constexpr uint32_t BE = block_elems(T), BB = block_bytes(T), TH = ref_threads<NV>(), WAVES = TH / 64;
    constexpr uint32_t CH = chunk_elems<T, NV>(), CHB = CH / BE * BB;
    constexpr uint32_t PIECES = (CHB + 15) / 16, WR = 8 * R, NLD = (WR * PIECES + 63) / 64;
    constexpr uint32_t RS = PIECES * 16 + 16;  // LDS bytes of a row's piece: the rows start on different banks
    constexpr uint32_t XS = CH / 8 + 4;        // LDS floats of one sum's x: the 8 sums start on different banks
    constexpr uint32_t XLD = NV * CH / TH;     // x loads per thread and chunk
    static_assert(NV * CH % TH == 0 && CH % 32 == 0 && CH % BE == 0 && XS % 4 == 0);
    __shared__ __align__(16) uint8_t wl[WAVES][WR * RS];
    __shared__ __align__(16) float xl[2][NV * 8 * XS];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, j = lane & 7u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t row0 = (blockIdx.x * WAVES + wave) * WR, t0 = blockIdx.y * NV;
    const uint32_t full = cols - cols % 8u, nch = full / CH + (full % CH != 0);
    const uint64_t row_len = (uint64_t)(cols / BE) * BB;

    uint4 wreg[NLD];
    float xreg[XLD];
    auto load = [&](uint32_t c) __attribute__((always_inline)) {
        const uint64_t b0 = (uint64_t)c * CHB, left = row_len - b0;
        const uint32_t here = (uint32_t)min((uint64_t)CHB, left);  // this chunk's bytes of a row
#pragma unroll
        for (uint32_t i = 0; i < NLD; ++i) {
            const uint32_t e = lane + 64 * i, r = e / PIECES, o = e % PIECES * 16;
            wreg[i] = uint4{0, 0, 0, 0};
            if (r < WR && o < here)  // rows past the end read the last row; their sums are not stored
                wreg[i] = load_piece(w + (uint64_t)min(row0 + r, rows - 1) * w_stride + b0 + o, left - o);
        }
#pragma unroll
        for (uint32_t i = 0; i < XLD; ++i) {
            const uint32_t e = tid + TH * i, v = e / CH, k = c * CH + e % CH;
            xreg[i] = k < full ? x[(uint64_t)min(t0 + v, n_vec - 1) * x_stride + k] : 0.0f;
        }
    };
    auto store = [&](uint32_t c) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t i = 0; i < NLD; ++i) {
            const uint32_t e = lane + 64 * i, r = e / PIECES, o = e % PIECES * 16;
            if (r < WR) *reinterpret_cast<uint4*>(&wl[wave][r * RS + o]) = wreg[i];
        }
#pragma unroll
        for (uint32_t i = 0; i < XLD; ++i) {
            const uint32_t e = tid + TH * i, v = e / CH, k = e % CH;
            xl[c & 1u][(v * 8 + k % 8) * XS + k / 8] = xreg[i];
        }
    };

    float p[R][NV];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int v = 0; v < NV; ++v) p[r][v] = 0.0f;
    if (nch > 0) {
        load(0);
        store(0);
    }
    __syncthreads();
    for (uint32_t c = 0; c < nch; ++c) {
        if (c + 1 < nch) load(c + 1);
        const uint32_t steps = min(CH, full - c * CH) / 8;  // additions of each sum in this chunk
        const uint8_t* rp = &wl[wave][lane / 8 * RS];
        const float* xp = &xl[c & 1u][j * XS];
        auto slot = [&](const uint8_t* piece, uint32_t sl, uint32_t s) __attribute__((always_inline)) {
            float q[R][4];
#pragma unroll
            for (int r = 0; r < R; ++r) slot4<T>(piece + r * 8 * RS, sl, j, q[r]);
#pragma unroll
            for (int v = 0; v < NV; ++v) {
                const float4 xv = *reinterpret_cast<const float4*>(xp + v * 8 * XS + 4 * s);
                const float xe[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                for (int k = 0; k < 4; ++k)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float prod = xe[k] * q[r][k];
                        p[r][v] = p[r][v] + prod;
                    }
            }
        };
        if constexpr (BE == 256) {
            for (uint32_t b = 0; b < steps / 32; ++b)
#pragma unroll
                for (uint32_t sl = 0; sl < 8; ++sl) slot(rp + b * BB, sl, b * 8 + sl);
        } else {
#pragma unroll 4
            for (uint32_t s = 0; s < steps / 4; ++s) slot(rp + s * (32 / BE * BB), 0, s);
            if constexpr (BE == 1) {  // a last slot of fewer than four additions
                for (uint32_t k = steps & ~3u; k < steps; ++k)
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        const float q = gguf_elem<T, true>(rp + r * 8 * RS, 8 * k + j);
#pragma unroll
                        for (int v = 0; v < NV; ++v) {
                            const float prod = xp[v * 8 * XS + k] * q;
                            p[r][v] = p[r][v] + prod;
                        }
                    }
            }
        }
        if (c + 1 < nch) store(c + 1);
        __syncthreads();
    }
    // ((p0+p4)+(p1+p5)) + ((p2+p6)+(p3+p7)), then + tail, exactly as the CPU dot
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const float a = p[r][v] + __shfl_down(p[r][v], 4, 8);  // lanes 0..3: p_j + p_{j+4}
            const float b = a + __shfl_down(a, 1, 8);              // lane 0: left, lane 2: right
            const float s = b + __shfl_down(b, 2, 8);              // lane 0: left + right
            const uint32_t n = row0 + 8 * r + lane / 8;
            if (j == 0 && n < rows && t0 + v < n_vec) {
                const float* xt = x + (uint64_t)(t0 + v) * x_stride;
                float tail = 0.0f;
                if constexpr (BE == 1)
                    for (uint32_t i = full; i < cols; ++i) {
                        const float prod = xt[i] * gguf_elem<T>(w + (uint64_t)n * w_stride, i);
                        tail = tail + prod;
                    }
                y[(uint64_t)(t0 + v) * y_stride + n] = s + tail;
            }
        }
}

// Few rows and vectors: the same sums with the products computed ahead by other waves, one vector
// (blockIdx.y) per workgroup. A lone wave per 8 rows leaves the chip idle (5120 rows: 640 waves on 1024
// SIMDs) and pays decode, multiply and add in one dependent stream. Here a workgroup takes 8 rows with one
// chain wave and kOneProducers producer waves: in round r producer i turns chunk r * kOneProducers + i
// (kOneChunk elements of K) into products in LDS, one 16-byte quad per lane and slot, and the chain wave
// adds the round before in order (lane l: sum l % 8 of row l / 8, as above). Rows' bytes and x are loaded
// kOneAhead rounds ahead (a round is shorter than a memory round trip). The chain wave's place in the
// workgroup changes with the workgroup, so every SIMD gets as many of them.
// What bounds it is the length of a round (1.7 us at 5120 x 17408), not the issue rate: the producers'
// instructions (about 28 per slot of 4 x 64 products) are 16 of IQ4_NL's 57 us there and the chain's adds 7,
// but a producer writes a chunk's bytes, waits, reads them, writes the products and meets the barrier
// one after the other.
// Measured on MI355X against k_gemv_gguf_ref, us. One vector: 5120 x 17408 IQ4_NL 62 -> 57, Q3_K 92 -> 75, Q6_K
// 99 -> 70; 1024 x 5120 19 -> 14, 29 -> 17, 30 -> 16; 8192 x 5120 22 -> 22, 33 -> 31, 35 -> 28; 10240 x 5120 27 -> 32,
// 40 -> 42, 42 -> 39; 17408 x 5120 35 -> 47, 53 -> 62, 52 -> 56. Two vectors of 1024 x 5120: 20 -> 14, 30 -> 18, 30 ->
// 17; eight of them 28 -> 21, 43 -> 27, 44 -> 24.
constexpr uint32_t kOneProducers = 2, kOneChunk = 256, kOneAhead = 3;
// LDS of a workgroup: 36.9-39.7 KB for the quantized types, 43.5 for the 16-bit ones, 51.7 for F32
template <uint32_t T>
constexpr uint32_t one_lds_bytes() {
    constexpr uint32_t row = (kOneChunk / block_elems(T) * block_bytes(T) + 15) / 16 * 16 + 16;
    return kOneProducers * (8 * row + 4 * 8 * (kOneChunk / 8 + 4)) + 2 * kOneProducers * (kOneChunk / 32) * 64 * 16;
}

template <uint32_t T>
__global__ __launch_bounds__(64 * (kOneProducers + 1)) void k_gemv_gguf_one(const uint8_t* __restrict__ w, uint64_t w_stride,
                                                                            const float* __restrict__ x, uint64_t x_stride,
                                                                            float* __restrict__ y, uint64_t y_stride, uint32_t rows,
                                                                            uint32_t cols) {
#pragma clang fp contract(off)
    constexpr uint32_t BE = block_elems(T), BB = block_bytes(T), P = kOneProducers, CH = kOneChunk, CHB = CH / BE * BB;
    constexpr uint32_t PIECES = (CHB + 15) / 16, NLD = (8 * PIECES + 63) / 64;
    constexpr uint32_t RS = PIECES * 16 + 16, XS = CH / 8 + 4, XLD = CH / 64, SLOTS = CH / 32;
    x += blockIdx.y * x_stride;
    y += blockIdx.y * y_stride;
    __shared__ __align__(16) uint8_t wl[P][8 * RS];
    __shared__ __align__(16) float xl[P][8 * XS];
    __shared__ float4 prod[2][P][SLOTS][64];
    static_assert(sizeof(wl) + sizeof(xl) + sizeof(prod) == one_lds_bytes<T>());
    const uint32_t lane = threadIdx.x & 63u, j = lane & 7u;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t role = (wave + P + 1 - blockIdx.x % (P + 1)) % (P + 1);  // P: the chain wave; else producer
    const uint32_t row0 = blockIdx.x * 8;
    const uint32_t full = cols - cols % 8u, nch = full / CH + (full % CH != 0), rounds = nch / P + (nch % P != 0);
    const uint64_t row_len = (uint64_t)(cols / BE) * BB;
    auto chunk_steps = [&](uint32_t c) __attribute__((always_inline)) { return min(CH, full - c * CH) / 8; };

    if (role < P) {
        uint4 wreg[kOneAhead][NLD];
        float xreg[kOneAhead][XLD];
        auto load = [&](uint32_t c, uint4 (&wr)[NLD], float (&xr)[XLD]) __attribute__((always_inline)) {
            if (c >= nch) return;
            const uint64_t b0 = (uint64_t)c * CHB, left = row_len - b0;
            const uint32_t here = (uint32_t)min((uint64_t)CHB, left);
#pragma unroll
            for (uint32_t i = 0; i < NLD; ++i) {
                const uint32_t e = lane + 64 * i, r = e / PIECES, o = e % PIECES * 16;
                wr[i] = uint4{0, 0, 0, 0};
                if (r < 8 && o < here) wr[i] = load_piece(w + (uint64_t)min(row0 + r, rows - 1) * w_stride + b0 + o, left - o);
            }
#pragma unroll
            for (uint32_t i = 0; i < XLD; ++i) {
                const uint32_t k = c * CH + lane + 64 * i;
                xr[i] = k < full ? x[k] : 0.0f;
            }
        };
        auto produce = [&](uint32_t c, uint32_t buf, const uint4 (&wr)[NLD], const float (&xr)[XLD]) __attribute__((always_inline)) {
#pragma unroll
            for (uint32_t i = 0; i < NLD; ++i) {
                const uint32_t e = lane + 64 * i, r = e / PIECES, o = e % PIECES * 16;
                if (r < 8) *reinterpret_cast<uint4*>(&wl[role][r * RS + o]) = wr[i];
            }
#pragma unroll
            for (uint32_t i = 0; i < XLD; ++i) {
                const uint32_t k = lane + 64 * i;
                xl[role][k % 8 * XS + k / 8] = xr[i];
            }
            __builtin_amdgcn_wave_barrier();  // (LDS keeps a wave's own order)
            const uint8_t* rp = &wl[role][lane / 8 * RS];
            const float* xp = &xl[role][j * XS];
            auto slot = [&](const uint8_t* piece, uint32_t sl, uint32_t s) __attribute__((always_inline)) {
                float q[4];
                slot4<T>(piece, sl, j, q);
                const float4 xv = *reinterpret_cast<const float4*>(xp + 4 * s);
                return float4{xv.x * q[0], xv.y * q[1], xv.z * q[2], xv.w * q[3]};
            };
            // a part of a chunk is whole blocks; past it (and in a plain type's last slot) the
            // products are of whatever LDS holds and are not added
            const uint32_t slots = (chunk_steps(c) + 3) / 4;
            if (slots == SLOTS) {
                float4 o[SLOTS];  // written after the last slot's reads: a write between would hold them back
#pragma unroll
                for (uint32_t s = 0; s < SLOTS; ++s) {
                    if constexpr (BE == 256) o[s] = slot(rp, s, s);
                    else o[s] = slot(rp + s * (32 / BE * BB), 0, s);
                }
#pragma unroll
                for (uint32_t s = 0; s < SLOTS; ++s) prod[buf][role][s][lane] = o[s];
            } else {
                for (uint32_t s = 0; s < slots; ++s) {
                    if constexpr (BE == 256) prod[buf][role][s][lane] = slot(rp, s, s);
                    else prod[buf][role][s][lane] = slot(rp + s * (32 / BE * BB), 0, s);
                }
            }
        };
#pragma unroll
        for (uint32_t d = 0; d < kOneAhead; ++d) load(d * P + role, wreg[d], xreg[d]);
        for (uint32_t r0 = 0; r0 < rounds + 1; r0 += kOneAhead) {
#pragma unroll
            for (uint32_t d = 0; d < kOneAhead; ++d) {
                const uint32_t r = r0 + d, c = r * P + role;
                if (r > rounds) break;
                if (c < nch) {
                    produce(c, r & 1u, wreg[d], xreg[d]);
                    load(c + kOneAhead * P, wreg[d], xreg[d]);
                }
                __syncthreads();
            }
        }
        return;
    }
    __builtin_amdgcn_s_setprio(2);
    float p = 0.0f;
    for (uint32_t r = 0; r < rounds + 1; ++r) {
        if (r > 0) {
            const uint32_t buf = (r - 1) & 1u;
#pragma unroll
            for (uint32_t i = 0; i < P; ++i) {
                const uint32_t c = (r - 1) * P + i;
                const uint32_t steps = c < nch ? chunk_steps(c) : 0u;
                if (steps == CH / 8) {
                    float4 q[SLOTS];
#pragma unroll
                    for (uint32_t s = 0; s < SLOTS; ++s) q[s] = prod[buf][i][s][lane];
#pragma unroll
                    for (uint32_t s = 0; s < SLOTS; ++s) {
                        p = p + q[s].x;
                        p = p + q[s].y;
                        p = p + q[s].z;
                        p = p + q[s].w;
                    }
                } else {
                    for (uint32_t k = 0; k < steps; ++k) p = p + reinterpret_cast<const float*>(&prod[buf][i][k / 4][lane])[k % 4];
                }
            }
        }
        __syncthreads();
    }
    const float a = p + __shfl_down(p, 4, 8);  // the CPU dot's combine, as above
    const float b = a + __shfl_down(a, 1, 8);
    const float sum = b + __shfl_down(b, 2, 8);
    const uint32_t n = row0 + lane / 8;
    if (j == 0 && n < rows) {
        float tail = 0.0f;
        if constexpr (BE == 1)
            for (uint32_t i = full; i < cols; ++i) {
                const float pr = x[i] * gguf_elem<T>(w + (uint64_t)n * w_stride, i);
                tail = tail + pr;
            }
        y[n] = sum + tail;
    }
}

struct RefArgs {
    const uint8_t* w;
    uint64_t w_stride;
    const float* x;
    uint64_t x_stride;
    float* y;
    uint64_t y_stride;
    uint32_t rows, cols;
};

// `n` vectors from t0 on, NV per workgroup (the last group may be short)
template <uint32_t T, int NV, int R>
void launch_ref_nv(const RefArgs& a, uint32_t t0, uint32_t n, hipStream_t st) {
    constexpr uint32_t per = ref_threads<NV>() / 64 * 8 * R;  // rows per workgroup
    constexpr uint32_t kMaxGroups = 32768;                    // grid.y stays within the launch limits
    for (uint32_t k = 0; k < n; k += kMaxGroups * NV) {
        const uint32_t m = std::min(n - k, kMaxGroups * NV);
        hipLaunchKernelGGL((k_gemv_gguf_ref<T, NV, R>), dim3((a.rows - 1) / per + 1, (m + NV - 1) / NV), dim3(ref_threads<NV>()),
                           0, st, a.w, a.w_stride, a.x + (uint64_t)(t0 + k) * a.x_stride, a.x_stride,
                           a.y + (uint64_t)(t0 + k) * a.y_stride, a.y_stride, a.rows, a.cols, m);
    }
}

template <uint32_t T>
void launch_ref(const RefArgs& a, uint32_t n_vec, hipStream_t st) {
    // Large vector groups decode least and small ones fill the chip soonest: a group's time hardly depends
    // on its rows until there is about a wave per SIMD (1024). What decides is therefore the call's work in
    // units of 8 rows of one vector. While its products-ahead workgroups are all resident at once (four per CU by
    // the LDS of the quantized types, three for the others; 256 CUs) they win, then groups of 1, 2 and 4 vectors
    // in turn. The types that decode slowest skip the groups of one; the 256-element blocks but Q5_K's, whose
    // decoding outweighs what a group of four adds, go to 4 sooner.
    // Groups of 16 with two rows per lane take over at 1024 waves of them, one of 8 what is left of a large matrix.
    // Groups of one and two take every vector (a launch of its own costs the whole chain again); beside groups of
    // 4, one or two vectors left over go on their own (three fill a group).
    // Measured on MI355X, us, Q4_K of 5120 columns either side of each line: 1024 units ahead 19, groups of one 23;
    // 1280 31 and 25; 2048 groups of one 27, of two 33; 3072 47 and 37 (2560: Q4_K 34 and 36, but Q5_0 51 and 47); 6144 of
    // two 48, of four 47; 7680 70 and 48. Slow types: 1280 units of Q3_K 5120 x 1024 ahead / of one / of two 13.1 / 13.9 /
    // 12.8; 4096 units of two and four IQ3_S 81 and 60, Q6_K 54 and 47, but Q5_K 44 and 58, Q8_0 39 and 65. Against
    // the products ahead for one vector only, groups of two next and groups of four from 4096 units on: 0.77x the
    // time over 16 types, 16 sizes and 1 to 64 vectors (IQ3_S 1024 x 5120 at two 67 -> 22), none slower by more than 4%.
    constexpr bool kSlow = T == kQ3_K || T == kQ6_K || T == kIQ3_S, kSooner = block_elems(T) == 256 && T != kQ5_K;
    constexpr uint64_t kAhead = 256 * (163840 / one_lds_bytes<T>()), kOnes = kSlow ? 0 : 2048, kTwos = 6144;
    const uint64_t w = (a.rows - 1) / 8 + 1;  // units of one vector
    for (uint32_t t = 0; t < n_vec;) {
        const uint32_t left = n_vec - t, g16 = left / 16 + (left % 16 > 8 ? 1 : 0), g4 = (left + 1) / 4;
        const bool fours = left > 2 && (kSooner ? (uint64_t)a.rows * g4 >= 8 * 1024 : w * (left + left % 2) > kTwos);
        uint32_t n = left;
        if ((uint64_t)a.rows * g16 >= 16 * 1024) {
            n = std::min(left, 16 * g16);
            launch_ref_nv<T, 16, 2>(a, t, n, st);
        } else if (left > 4 && left <= 8 && a.rows >= 32 * 1024) {
            launch_ref_nv<T, 8, 2>(a, t, n, st);
        } else if (w * left <= kAhead) {
            hipLaunchKernelGGL((k_gemv_gguf_one<T>), dim3((uint32_t)w, n), dim3(64 * (kOneProducers + 1)), 0, st, a.w, a.w_stride,
                               a.x + (uint64_t)t * a.x_stride, a.x_stride, a.y + (uint64_t)t * a.y_stride, a.y_stride, a.rows, a.cols);
        } else if (w * left <= kOnes || left == 1) {
            launch_ref_nv<T, 1, 1>(a, t, n, st);
        } else if (!fours) {
            launch_ref_nv<T, 2, 1>(a, t, n, st);
        } else {
            n = std::min(left, 4 * g4);
            launch_ref_nv<T, 4, 1>(a, t, n, st);
        }
        t += n;
    }
}

}  // namespace

int launch_gemv_gguf_ref(uint32_t type, const uint8_t* w, uint64_t w_stride, const float* x, uint64_t x_stride, float* y,
                         uint64_t y_stride, uint32_t rows, uint32_t cols, uint32_t n_vec, hipStream_t st) {
    const RefArgs a{w, w_stride, x, x_stride, y, y_stride, rows, cols};
    switch (type) {
        case kF32: launch_ref<kF32>(a, n_vec, st); break;
        case kF16: launch_ref<kF16>(a, n_vec, st); break;
        case kBF16: launch_ref<kBF16>(a, n_vec, st); break;
        case kQ4_0: launch_ref<kQ4_0>(a, n_vec, st); break;
        case kQ4_1: launch_ref<kQ4_1>(a, n_vec, st); break;
        case kQ5_0: launch_ref<kQ5_0>(a, n_vec, st); break;
        case kQ5_1: launch_ref<kQ5_1>(a, n_vec, st); break;
        case kQ8_0: launch_ref<kQ8_0>(a, n_vec, st); break;
        case kQ2_K: launch_ref<kQ2_K>(a, n_vec, st); break;
        case kQ3_K: launch_ref<kQ3_K>(a, n_vec, st); break;
        case kQ4_K: launch_ref<kQ4_K>(a, n_vec, st); break;
        case kQ5_K: launch_ref<kQ5_K>(a, n_vec, st); break;
        case kQ6_K: launch_ref<kQ6_K>(a, n_vec, st); break;
        case kIQ4_NL: launch_ref<kIQ4_NL>(a, n_vec, st); break;
        case kIQ3_S: launch_ref<kIQ3_S>(a, n_vec, st); break;
        case kIQ4_XS: launch_ref<kIQ4_XS>(a, n_vec, st); break;
        default: return set_error(HALO_MI_E_UNSUPPORTED, "gemv_gguf_ref: type %u has no decoder", type);
    }
    return hip_status(hipGetLastError(), "gemv_gguf_ref launch");
}

}  // namespace halo_mi
