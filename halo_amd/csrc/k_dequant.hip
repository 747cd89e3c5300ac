// gfx950 kernels of the halo_mi355x library: GGUF <-> SLAB repack, exact dequantization
// (bit-identical to tensor::dequantize_row, src/tensor/quant.cpp:430-435 of the reference) and
// a fill kernel for workspace initialisation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <type_traits>

#include "device.h"
#include "launch.h"

namespace halo_mi {
namespace {

using namespace dev;

// ==========================================================================================
// Repack / unpack / dequantize
// ==========================================================================================

// One thread per (slab, kRepackBlocks consecutive blocks, row), row fastest: the 64 threads of a
// (slab, block) read or write each of the block's slot records as one contiguous 1 KB, and each
// works on its own row's block with 16-byte accesses at whatever alignment the row has, all in
// registers. Bound by HBM: the rows' accesses are one line apart per lane, and a thread of a
// 32-weight format takes several blocks so that it uses most of a line at once. Measured on MI355X,
// 17408 x 5120, repack / unpack us (bytes moved one by one through a block in scratch memory, and
// unpack with the blocks of a row side by side, before): Q4_0 61 / 125 -> 32 / 58, Q8_0 120 / 304 ->
// 42 / 70, Q4_K 22 (its own 16-byte path) / 589 -> 18 / 26, Q5_K 174 / 738 -> 21 / 30, Q6_K 223 / 886
// -> 34 / 42 (73 MB: 4.4 TB/s read and written), IQ4_XS 136 / 609 -> 17 / 25. (With a branch around every load
// for the rows past the last Q4_K took 22, Q6_K 39 and Q4_K 17408 x 17408 94, against its older path's 86.)
template <uint32_t T>
constexpr uint32_t kRepackBlocks = T == kQ4_0 ? 8u : T == kQ8_0 ? 4u : 1u;
// A matrix that gives too few threads that way to fill the chip takes one block per thread (repack_blocks).
constexpr uint64_t kRepackThreads = 16384;

__device__ __forceinline__ uint4 ld16(const uint8_t* p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}
__device__ __forceinline__ void st16(uint8_t* p, const uint4& v) { __builtin_memcpy(p, &v, 16); }
__device__ __forceinline__ void unwords(const uint4& v, uint32_t w[4]) {
    w[0] = v.x;
    w[1] = v.y;
    w[2] = v.z;
    w[3] = v.w;
}

// The two slot records of 32 bytes holding 64 4-bit codes (a: bytes 0..15, c: 16..31): the low
// nibbles' slot, then the high nibbles'; and back.
__device__ __forceinline__ void nibbles_to_slots(const uint4& a4, const uint4& c4, uint4& lo, uint4& hi) {
    uint32_t a[4], c[4], l[4], h[4];
    unwords(a4, a);
    unwords(c4, c);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        l[k] = (a[k] & 0x0F0F0F0Fu) | ((c[k] & 0x0F0F0F0Fu) << 4);
        h[k] = ((a[k] >> 4) & 0x0F0F0F0Fu) | (c[k] & 0xF0F0F0F0u);
    }
    lo = uint4{l[0], l[1], l[2], l[3]};
    hi = uint4{h[0], h[1], h[2], h[3]};
}
// (the map is its own inverse: lo, hi -> a, c)

template <uint32_t T>
__device__ __forceinline__ void repack_block(const uint8_t* __restrict__ s, bool live, uint8_t* __restrict__ out, const SlabGeom& g,
                                             uint32_t r, uint32_t b) {
    // (past the last row s is the first row's block: every load is issued without a branch of its own)
    auto in = [&](uint32_t o) __attribute__((always_inline)) {
        const uint4 v = ld16(s + o);
        return uint4{live ? v.x : 0u, live ? v.y : 0u, live ? v.z : 0u, live ? v.w : 0u};
    };
    auto in2 = [&](uint32_t o) __attribute__((always_inline)) {
        uint16_t v;
        __builtin_memcpy(&v, s + o, 2);
        return live ? v : (uint16_t)0;
    };
    auto rec = [&](uint64_t off, uint64_t i, uint32_t bytes) __attribute__((always_inline)) { return out + off + (i * 64 + r) * bytes; };
    if constexpr (T == kQ4_0 || T == kQ8_0) {
        const uint16_t d = in2(0);
        const uint4 q = in(2);
        if constexpr (T == kQ4_0) {
            *reinterpret_cast<uint4*>(rec(g.q_off, b, 16)) = q;
        } else {
            const uint4 q1 = in(18);
            *reinterpret_cast<uint4*>(rec(g.q_off, 2 * (uint64_t)b, 16)) = q;
            *reinterpret_cast<uint4*>(rec(g.q_off, 2 * (uint64_t)b + 1, 16)) = q1;
        }
        *reinterpret_cast<uint16_t*>(rec(g.aux_off, b, 2)) = d;
    } else if constexpr (T == kIQ4_XS) {
        uint2 hdr;
        __builtin_memcpy(&hdr, s, 8);
        if (!live) hdr = uint2{0, 0};
        uint4 q[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) q[j] = in(8 + 16 * j);
        *reinterpret_cast<uint2*>(rec(g.aux_off, b, 8)) = hdr;
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) *reinterpret_cast<uint4*>(rec(g.q_off, (uint64_t)b * 8 + j, 16)) = q[j];
    } else if constexpr (T == kQ4_K || T == kQ5_K) {
        constexpr uint32_t Q = T == kQ4_K ? 16 : 48;
        const uint4 hdr = in(0);
        uint4 q[8], qh[2];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) q[i] = in(Q + 16 * i);
        if constexpr (T == kQ5_K) {
            qh[0] = in(16);
            qh[1] = in(32);
        }
        *reinterpret_cast<uint4*>(rec(T == kQ4_K ? g.aux_off : g.sc_off, b, 16)) = hdr;
#pragma unroll
        for (uint32_t grp = 0; grp < 4; ++grp) {  // sub-blocks 2 grp (low nibbles), 2 grp + 1 (high)
            uint4 lo, hi;
            nibbles_to_slots(q[2 * grp], q[2 * grp + 1], lo, hi);
            *reinterpret_cast<uint4*>(rec(g.q_off, (uint64_t)b * 8 + 2 * grp, 16)) = lo;
            *reinterpret_cast<uint4*>(rec(g.q_off, (uint64_t)b * 8 + 2 * grp + 1, 16)) = hi;
        }
        if constexpr (T == kQ5_K) {  // bit j of qh dword i -> bit i of the bytes of slot j's word
            uint32_t h[8];
            unwords(qh[0], h);
            unwords(qh[1], h + 4);
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                uint32_t w = 0;
#pragma unroll
                for (uint32_t i = 0; i < 8; ++i) w |= ((h[i] >> j) & 0x01010101u) << i;
                *reinterpret_cast<uint32_t*>(rec(g.aux_off, (uint64_t)b * 8 + j, 4)) = w;
            }
        }
    } else {  // Q6_K
        uint4 q[8], qh[4];
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) q[i] = in(16 * i);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) qh[i] = in(128 + 16 * i);
        const uint4 sc = in(192);
        const uint16_t d = in2(208);
        *reinterpret_cast<uint4*>(rec(g.sc_off, b, 16)) = sc;
        *reinterpret_cast<uint16_t*>(rec(g.d_off, b, 2)) = d;
#pragma unroll
        for (uint32_t n = 0; n < 2; ++n) {
            // 32 code bytes 64 n + 32 p: slots 4 n + p (low nibbles) and 4 n + 2 + p (high)
#pragma unroll
            for (uint32_t p = 0; p < 2; ++p) {
                uint4 lo, hi;
                nibbles_to_slots(q[4 * n + 2 * p], q[4 * n + 2 * p + 1], lo, hi);
                *reinterpret_cast<uint4*>(rec(g.q_off, (uint64_t)b * 8 + 4 * n + p, 16)) = lo;
                *reinterpret_cast<uint4*>(rec(g.q_off, (uint64_t)b * 8 + 4 * n + 2 + p, 16)) = hi;
            }
            uint32_t h[8];
            unwords(qh[2 * n], h);
            unwords(qh[2 * n + 1], h + 4);
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {  // slot 4 n + k: bits 2 k .. 2 k + 1 (q6_qh_byte's places)
                uint32_t w[2];
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    auto t = [&](uint32_t x) __attribute__((always_inline)) { return (h[x] >> (2 * k)) & 0x03030303u; };
                    w[i] = t(2 * i + 1) | (t(2 * i + 5) << 2) | (t(2 * i) << 4) | (t(2 * i + 4) << 6);
                }
                *reinterpret_cast<uint2*>(rec(g.aux_off, (uint64_t)b * 8 + 4 * n + k, 8)) = uint2{w[0], w[1]};
            }
        }
    }
}

// repack_block's inverse: the block's GGUF bytes at d.
template <uint32_t T>
__device__ __forceinline__ void unpack_block(const uint8_t* __restrict__ src, uint8_t* __restrict__ d, const SlabGeom& g, uint32_t r,
                                             uint32_t b) {
    auto rec = [&](uint64_t off, uint64_t i, uint32_t bytes) __attribute__((always_inline)) { return src + off + (i * 64 + r) * bytes; };
    auto q = [&](uint64_t i) __attribute__((always_inline)) { return *reinterpret_cast<const uint4*>(rec(g.q_off, i, 16)); };
    if constexpr (T == kQ4_0 || T == kQ8_0) {
        __builtin_memcpy(d, rec(g.aux_off, b, 2), 2);
        if constexpr (T == kQ4_0) {
            st16(d + 2, q(b));
        } else {
            st16(d + 2, q(2 * (uint64_t)b));
            st16(d + 18, q(2 * (uint64_t)b + 1));
        }
    } else if constexpr (T == kIQ4_XS) {
        const uint2 hdr = *reinterpret_cast<const uint2*>(rec(g.aux_off, b, 8));
        __builtin_memcpy(d, &hdr, 8);
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) st16(d + 8 + 16 * j, q((uint64_t)b * 8 + j));
    } else if constexpr (T == kQ4_K || T == kQ5_K) {
        constexpr uint32_t Q = T == kQ4_K ? 16 : 48;
        st16(d, *reinterpret_cast<const uint4*>(rec(T == kQ4_K ? g.aux_off : g.sc_off, b, 16)));
        if constexpr (T == kQ5_K) {
            uint32_t h[8] = {};
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                const uint32_t w = *reinterpret_cast<const uint32_t*>(rec(g.aux_off, (uint64_t)b * 8 + j, 4));
#pragma unroll
                for (uint32_t i = 0; i < 8; ++i) h[i] |= ((w >> i) & 0x01010101u) << j;
            }
            st16(d + 16, uint4{h[0], h[1], h[2], h[3]});
            st16(d + 32, uint4{h[4], h[5], h[6], h[7]});
        }
#pragma unroll
        for (uint32_t grp = 0; grp < 4; ++grp) {
            uint4 a, c;
            nibbles_to_slots(q((uint64_t)b * 8 + 2 * grp), q((uint64_t)b * 8 + 2 * grp + 1), a, c);
            st16(d + Q + 32 * grp, a);
            st16(d + Q + 32 * grp + 16, c);
        }
    } else {  // Q6_K
#pragma unroll
        for (uint32_t n = 0; n < 2; ++n) {
#pragma unroll
            for (uint32_t p = 0; p < 2; ++p) {
                uint4 a, c;
                nibbles_to_slots(q((uint64_t)b * 8 + 4 * n + p), q((uint64_t)b * 8 + 4 * n + 2 + p), a, c);
                st16(d + 64 * n + 32 * p, a);
                st16(d + 64 * n + 32 * p + 16, c);
            }
            uint32_t h[8] = {};
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint2 w2 = *reinterpret_cast<const uint2*>(rec(g.aux_off, (uint64_t)b * 8 + 4 * n + k, 8));
                const uint32_t w[2] = {w2.x, w2.y};
#pragma unroll
                for (uint32_t i = 0; i < 2; ++i) {
                    h[2 * i + 1] |= (w[i] & 0x03030303u) << (2 * k);
                    h[2 * i + 5] |= ((w[i] >> 2) & 0x03030303u) << (2 * k);
                    h[2 * i] |= ((w[i] >> 4) & 0x03030303u) << (2 * k);
                    h[2 * i + 4] |= ((w[i] >> 6) & 0x03030303u) << (2 * k);
                }
            }
            st16(d + 128 + 32 * n, uint4{h[0], h[1], h[2], h[3]});
            st16(d + 128 + 32 * n + 16, uint4{h[4], h[5], h[6], h[7]});
        }
        st16(d + 192, *reinterpret_cast<const uint4*>(rec(g.sc_off, b, 16)));
        __builtin_memcpy(d + 208, rec(g.d_off, b, 2), 2);
    }
}

template <uint32_t T, uint32_t NB>
__global__ __launch_bounds__(256) void k_repack_slab(const uint8_t* __restrict__ src, uint64_t src_stride, uint32_t rows, uint32_t cols,
                                                     uint8_t* __restrict__ dst) {
    const SlabGeom g = slab_geom(T, cols);
    const uint32_t nblk = cols / block_elems(T), groups = (nblk + NB - 1) / NB;
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t r = (uint32_t)(idx % kSlabRows);
    const uint64_t slab = idx / kSlabRows / groups, row = slab * kSlabRows + r;
    if (slab * kSlabRows >= rows) return;
    const uint32_t b0 = (uint32_t)(idx / kSlabRows % groups) * NB;
    const bool live = row < rows;
#pragma unroll
    for (uint32_t k = 0; k < NB; ++k)
        if (b0 + k < nblk)
            repack_block<T>(src + (live ? row : 0) * src_stride + (uint64_t)(b0 + k) * block_bytes(T), live, dst + slab * g.slab_bytes, g,
                            r, b0 + k);
}

template <uint32_t T, uint32_t NB>
__global__ __launch_bounds__(256) void k_unpack_slab(const uint8_t* __restrict__ src, uint32_t rows, uint32_t cols,
                                                     uint8_t* __restrict__ dst, uint64_t dst_stride) {
    const SlabGeom g = slab_geom(T, cols);
    const uint32_t nblk = cols / block_elems(T), groups = (nblk + NB - 1) / NB;
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t r = (uint32_t)(idx % kSlabRows);
    const uint64_t slab = idx / kSlabRows / groups, row = slab * kSlabRows + r;
    if (row >= rows) return;
    const uint32_t b0 = (uint32_t)(idx / kSlabRows % groups) * NB;
#pragma unroll
    for (uint32_t k = 0; k < NB; ++k)
        if (b0 + k < nblk)
            unpack_block<T>(src + slab * g.slab_bytes, dst + row * dst_stride + (uint64_t)(b0 + k) * block_bytes(T), g, r, b0 + k);
}

// The table row of output row r: first_row + r, or ids[r] (GET_ROWS). An id outside the table
// returns false, and the thread of the row's first element reports it in *status.
__device__ __forceinline__ bool table_row(const int32_t* ids, uint32_t table_rows, uint32_t first_row, uint64_t r,
                                          bool first, uint32_t* status, uint64_t& row) {
    if (!ids) {
        row = first_row + r;
        return true;
    }
    const int32_t id = ids[r];
    if (id < 0 || (uint32_t)id >= table_rows) {
        if (first && status) atomicOr(status, kStatusBadIndex);
        return false;
    }
    row = (uint64_t)id;
    return true;
}

// Dequantize / GET_ROWS: a block of kDqThreads threads takes E elements of one output row per thread, consecutive
// ones (blocks of a row follow each other, so the row's index is one scalar division): with four a wave stores
// 1 KB at once. Bound by launch and load latency at a prefill chunk's sizes: 512 rows of 5120 from a Q6_K SLAB
// table 7.9 -> 5.7 us (one thread per 32-element slot stored 4 bytes at a 128-byte pitch), from a GGUF table
// 8.7 -> 6.5 us (one thread per element with 64-bit divisions); Q4_K 7.2 -> 4.7 and 8.8 -> 6.3.
constexpr uint32_t kDqThreads = 256;
// Elements of a GGUF call from which a thread takes four: with rows aligned for 16-byte stores, and with others.
// Below, the chip has threads to spare, and a thread's four byte-wise decodes in a row add latency (MI355X, one and
// four elements per thread, means of the 16 types, us: 1 x 5120 2.0 and 2.2, 64 x 5120 2.4 and 2.6, 102 x 5120 2.82 and
// 2.88; on other rows 64 x 5120 2.5 and 3.0, 512 x 2048 4.2 and 4.4; one per thread with 64-bit divisions 2.1, 2.6, 3.05;
// 2.7, 4.5. From there on four gain: 512 x 2048 aligned 4.0 and 3.5, 4096 x 5120 56 and 30, on other rows 55 and 37).
constexpr uint64_t kDqQuadElems = 1ull << 20, kDqQuadElemsOther = 1ull << 22;

// Stores w[0..3] at o[i..i+3], of which the first `left` exist; 16-byte stores where the row is aligned.
__device__ __forceinline__ void store4(float* o, uint32_t i, uint32_t left, const float w[4]) {
    if (left >= 4 && (reinterpret_cast<uintptr_t>(o + i) & 15u) == 0) {
        *reinterpret_cast<float4*>(o + i) = float4{w[0], w[1], w[2], w[3]};
    } else {
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k)
            if (k < left) o[i + k] = w[k];
    }
}

template <uint32_t T, uint32_t E>
__global__ __launch_bounds__(kDqThreads) void k_dequant_gguf(const uint8_t* __restrict__ w, uint64_t w_stride, uint32_t cols,
                                                             uint32_t first_row, uint32_t blocks_per_row,
                                                             float* __restrict__ out, uint64_t out_stride,
                                                             const int32_t* __restrict__ ids, uint32_t table_rows,
                                                             uint32_t* status) {
    const uint32_t r = blockIdx.x / blocks_per_row;
    const uint32_t i = (blockIdx.x % blocks_per_row) * (E * kDqThreads) + E * threadIdx.x;
    if (i >= cols) return;
    uint64_t row;
    if (!table_row(ids, table_rows, first_row, r, i == 0, status, row)) return;
    const uint8_t* p = w + row * w_stride;
    if constexpr (E == 1) {
        out[r * out_stride + i] = gguf_elem<T>(p, i);
    } else {
        static_assert(E == 4);
        float v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) v[k] = i + k < cols ? gguf_elem<T>(p, i + k) : 0.0f;
        store4(out + r * out_stride, i, cols - i, v);
    }
}

// Exact fp32 weights 4 k .. 4 k + 3 of slot s of the row at lane r of `slab` (the reference's
// expressions). Dword i = k % 4 of the slot's code record holds them, in the low nibbles (k < 4) or
// the high ones.
template <uint32_t T>
__device__ __forceinline__ void slab_quad_weights(const uint8_t* __restrict__ slab, const SlabGeom& g, uint32_t r,
                                                  uint32_t s, uint32_t k, float w[4]) {
#pragma clang fp contract(off)
    const uint32_t i = k & 3u, high = k >> 2;
    const uint64_t sr = (uint64_t)s * 64 + r, br = (uint64_t)(s / 8) * 64 + r;
    auto word = [&](uint64_t off) __attribute__((always_inline)) { return *reinterpret_cast<const uint32_t*>(slab + off); };
    auto half = [&](uint64_t off) __attribute__((always_inline)) { return h2f(*reinterpret_cast<const uint16_t*>(slab + off)); };
    if constexpr (T == kQ8_0) {
        const float d = half(g.aux_off + sr * 2);
        const uint32_t q = word(g.q_off + (((uint64_t)s * 2 + high) * 64 + r) * 16 + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = sbyte(q, e) * d;
        return;
    }
    const uint32_t q = word(g.q_off + sr * 16 + 4 * i);
    const uint32_t nib = (high ? q >> 4 : q) & 0x0F0F0F0Fu;
    if constexpr (T == kQ4_0) {
        const float d = half(g.aux_off + sr * 2);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = (ubyte(nib, e) - 8.0f) * d;
    } else if constexpr (T == kQ4_K || T == kQ5_K) {
        const uint4 hdr = *reinterpret_cast<const uint4*>(slab + (T == kQ4_K ? g.aux_off : g.sc_off) + br * 16);
        float d1, m1;
        q4k_scales(hdr, s % 8, d1, m1);
        uint32_t c = nib;
        if constexpr (T == kQ5_K) {
            const uint32_t qh = word(g.aux_off + sr * 4);
            c |= (high ? qh >> i : qh << (4 - i)) & 0x10101010u;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = d1 * ubyte(c, e) - m1;
    } else if constexpr (T == kIQ4_XS) {
        const uint2 hdr = *reinterpret_cast<const uint2*>(slab + g.aux_off + br * 8);
        const float dl = h2f((uint16_t)(hdr.x & 0xFFFFu)) * (float)iq4xs_ls(hdr.x >> 16, hdr.y, s % 8);
        const uint32_t c = iq4_lookup4(nib);
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = dl * (ubyte(c, e) - 128.0f);
    } else {  // Q6_K: the top bits as q6_slot_bytes_gemv (gemv_device.h) places them
        const uint32_t h = word(g.aux_off + sr * 8 + 4 * (i >> 1));
        const uint32_t top = (high ? ((i & 1u) ? h << 2 : h >> 2) : ((i & 1u) ? h << 4 : h)) & 0x30303030u;
        const int8_t sc = *reinterpret_cast<const int8_t*>(slab + g.sc_off + br * 16 + 2 * (s % 8) + high);
        const float dA = half(g.d_off + br * 2) * (float)sc;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = dA * (ubyte(nib | top, e) - 32.0f);
    }
}

template <uint32_t T>
__global__ __launch_bounds__(kDqThreads) void k_dequant_slab(const uint8_t* __restrict__ w, uint32_t cols, uint32_t first_row,
                                                             uint32_t blocks_per_row, float* __restrict__ out,
                                                             uint64_t out_stride, const int32_t* __restrict__ ids,
                                                             uint32_t table_rows, uint32_t* status) {
    const SlabGeom g = slab_geom(T, cols);
    const uint32_t r = blockIdx.x / blocks_per_row;
    const uint32_t i = (blockIdx.x % blocks_per_row) * (4 * kDqThreads) + 4 * threadIdx.x;
    if (i >= cols) return;
    uint64_t row;
    if (!table_row(ids, table_rows, first_row, r, i == 0, status, row)) return;
    float v[4];
    slab_quad_weights<T>(w + (row / kSlabRows) * g.slab_bytes, g, (uint32_t)(row % kSlabRows), i / kSlot, i % kSlot / 4, v);
    store4(out + r * out_stride, i, cols - i, v);
}

__global__ void k_fill_u32(uint32_t* p, uint64_t n, uint32_t v) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// The read floor: a plain stream over n16 16-byte words, U nontemporal loads in flight per
// thread, grid-stride. The words are folded into one value per thread that is stored only if it
// equals a constant no input here produces, so the loads stay and nothing is written.
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

template <int U>
__global__ __launch_bounds__(256) void k_stream_read(const u32x4_t* __restrict__ p, uint64_t n16, uint32_t* sink) {
    uint32_t acc = 0;
    const uint64_t stride = (uint64_t)gridDim.x * 256 * U;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 * U + threadIdx.x; i < n16; i += stride) {
        u32x4_t v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint64_t k = i + (uint64_t)u * 256;
            v[u] = __builtin_nontemporal_load(p + (k < n16 ? k : n16 - 1));
        }
#pragma unroll
        for (int u = 0; u < U; ++u) acc += v[u].x ^ v[u].y ^ v[u].z ^ v[u].w;
    }
    if (acc == 0x9E3779B9u) sink[blockIdx.x * 256 + threadIdx.x] = acc;
}
}  // namespace

int launch_stream_read(const void* p, uint64_t bytes, uint32_t workgroups, uint32_t unroll, uint32_t* sink, hipStream_t st) {
    const uint64_t n16 = bytes / 16;
    const dim3 grid(workgroups), block(256);
    switch (unroll) {
        case 2: hipLaunchKernelGGL(k_stream_read<2>, grid, block, 0, st, static_cast<const u32x4_t*>(p), n16, sink); break;
        case 4: hipLaunchKernelGGL(k_stream_read<4>, grid, block, 0, st, static_cast<const u32x4_t*>(p), n16, sink); break;
        case 8: hipLaunchKernelGGL(k_stream_read<8>, grid, block, 0, st, static_cast<const u32x4_t*>(p), n16, sink); break;
        default: hipLaunchKernelGGL(k_stream_read<16>, grid, block, 0, st, static_cast<const u32x4_t*>(p), n16, sink); break;
    }
    return hip_status(hipGetLastError(), "stream_read launch");
}

// Calls launch(blocks per thread, grid) for a repack or unpack: a thread per row (of whole slabs) and kRepackBlocks
// blocks, or one block where those are fewer than kRepackThreads (MI355X, Q4_0 with 8 and with 1, us: repack 64 x 17408
// 4.4 and 2.1, 1000 x 1024 4.1 and 2.2; unpack 64 x 17408 5.8 and 2.4; Q8_0 with 4 and 1: 64 x 17408 4.8 and 2.5).
template <uint32_t T, typename F>
static void repack_blocks(uint32_t rows, uint32_t cols, F launch) {
    const uint64_t padded = ((uint64_t)rows + kSlabRows - 1) / kSlabRows * kSlabRows, nblk = cols / block_elems(T);
    auto with = [&](auto nb) {
        const uint64_t threads = padded * ((nblk + nb() - 1) / nb());
        if (nb() > 1 && threads < kRepackThreads) return false;
        launch(nb, dim3((uint32_t)((threads + 255) / 256)));
        return true;
    };
    if (!with(std::integral_constant<uint32_t, kRepackBlocks<T>>{})) with(std::integral_constant<uint32_t, 1>{});
}

// Calls f(integral constant) with the SLAB type
template <typename F>
static void with_slab_type(uint32_t type, F f) {
    switch (type) {
        case kQ4_0: f(std::integral_constant<uint32_t, kQ4_0>{}); break;
        case kQ8_0: f(std::integral_constant<uint32_t, kQ8_0>{}); break;
        case kQ4_K: f(std::integral_constant<uint32_t, kQ4_K>{}); break;
        case kQ5_K: f(std::integral_constant<uint32_t, kQ5_K>{}); break;
        case kIQ4_XS: f(std::integral_constant<uint32_t, kIQ4_XS>{}); break;
        default: f(std::integral_constant<uint32_t, kQ6_K>{}); break;
    }
}

int launch_repack_slab(uint32_t type, const uint8_t* src, uint64_t src_stride, uint32_t rows, uint32_t cols,
                       uint8_t* dst, hipStream_t st) {
    with_slab_type(type, [&](auto t) {
        repack_blocks<t()>(rows, cols, [&](auto nb, dim3 grid) {
            hipLaunchKernelGGL((k_repack_slab<t(), nb()>), grid, dim3(256), 0, st, src, src_stride, rows, cols, dst);
        });
    });
    return hip_status(hipGetLastError(), "repack_slab launch");
}

int launch_unpack_slab(uint32_t type, const uint8_t* src, uint32_t rows, uint32_t cols, uint8_t* dst,
                       uint64_t dst_stride, hipStream_t st) {
    with_slab_type(type, [&](auto t) {
        repack_blocks<t()>(rows, cols, [&](auto nb, dim3 grid) {
            hipLaunchKernelGGL((k_unpack_slab<t(), nb()>), grid, dim3(256), 0, st, src, rows, cols, dst, dst_stride);
        });
    });
    return hip_status(hipGetLastError(), "unpack_slab launch");
}

// Calls launch(grid, first table row, out, ids) for output rows [0, n_rows) in ranges whose blocks
// fit one grid (`per` blocks per row).
template <typename F>
static int dequant_blocks(uint32_t n_rows, uint32_t per, uint32_t first_row, float* out, uint64_t out_stride,
                          const int32_t* ids, F launch) {
    const uint32_t most = std::max((1u << 23) / per, 1u);  // rows per launch (under 2^32 threads)
    for (uint32_t r = 0; r < n_rows; r += std::min(most, n_rows - r)) {
        const uint32_t n = std::min(most, n_rows - r);
        if (int rc = launch(dim3(n * per), first_row + r, out + (uint64_t)r * out_stride, ids ? ids + r : nullptr)) return rc;
    }
    return HALO_MI_OK;
}

int launch_dequant_gguf(uint32_t type, const uint8_t* w, uint64_t w_stride, uint32_t cols, uint32_t first_row,
                        uint32_t n_rows, float* out, uint64_t out_stride, hipStream_t st, const int32_t* ids,
                        uint32_t table_rows, uint32_t* status) {
    const bool aligned = (reinterpret_cast<uintptr_t>(out) % 16 | out_stride % 4) == 0;
    const bool quads = (uint64_t)n_rows * cols >= (aligned ? kDqQuadElems : kDqQuadElemsOther);
    const uint32_t per = (cols - 1) / ((quads ? 4 : 1) * kDqThreads) + 1;
    const dim3 block(kDqThreads);
#define HALO_MI_DQ(T)                                                                                                                                   \
    case T:                                                                                                                                             \
        if (quads) hipLaunchKernelGGL((k_dequant_gguf<T, 4>), grid, block, 0, st, w, w_stride, cols, first, per, o, out_stride, id, table_rows, status); \
        else hipLaunchKernelGGL((k_dequant_gguf<T, 1>), grid, block, 0, st, w, w_stride, cols, first, per, o, out_stride, id, table_rows, status);       \
        break
    return dequant_blocks(n_rows, per, first_row, out, out_stride, ids, [&](dim3 grid, uint32_t first, float* o, const int32_t* id) {
    switch (type) {
        HALO_MI_DQ(kF32);
        HALO_MI_DQ(kF16);
        HALO_MI_DQ(kBF16);
        HALO_MI_DQ(kQ4_0);
        HALO_MI_DQ(kQ4_1);
        HALO_MI_DQ(kQ5_0);
        HALO_MI_DQ(kQ5_1);
        HALO_MI_DQ(kQ8_0);
        HALO_MI_DQ(kQ2_K);
        HALO_MI_DQ(kQ3_K);
        HALO_MI_DQ(kQ4_K);
        HALO_MI_DQ(kQ5_K);
        HALO_MI_DQ(kQ6_K);
        HALO_MI_DQ(kIQ4_NL);
        HALO_MI_DQ(kIQ3_S);
        HALO_MI_DQ(kIQ4_XS);
        default: return set_error(HALO_MI_E_UNSUPPORTED, "dequant: type %u has no decoder", type);
    }
    return hip_status(hipGetLastError(), "dequant_gguf launch");
    });
#undef HALO_MI_DQ
}

int launch_dequant_slab(uint32_t type, const uint8_t* w, uint32_t cols, uint32_t first_row, uint32_t n_rows, float* out,
                        uint64_t out_stride, hipStream_t st, const int32_t* ids, uint32_t table_rows, uint32_t* status) {
    const uint32_t per = (cols - 1) / (4 * kDqThreads) + 1;
    const dim3 block(kDqThreads);
#define HALO_MI_DQ(T) hipLaunchKernelGGL(k_dequant_slab<T>, grid, block, 0, st, w, cols, first, per, o, out_stride, id, table_rows, status)
    return dequant_blocks(n_rows, per, first_row, out, out_stride, ids, [&](dim3 grid, uint32_t first, float* o, const int32_t* id) {
    switch (type) {
        case kQ4_0: HALO_MI_DQ(kQ4_0); break;
        case kQ8_0: HALO_MI_DQ(kQ8_0); break;
        case kQ4_K: HALO_MI_DQ(kQ4_K); break;
        case kQ5_K: HALO_MI_DQ(kQ5_K); break;
        case kIQ4_XS: HALO_MI_DQ(kIQ4_XS); break;
        default: HALO_MI_DQ(kQ6_K); break;
    }
    return hip_status(hipGetLastError(), "dequant_slab launch");
    });
#undef HALO_MI_DQ
}

int launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t st) {
    hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, st, p, n, v);
    return hip_status(hipGetLastError(), "fill launch");
}

}  // namespace halo_mi
