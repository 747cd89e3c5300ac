// gfx950 kernels of the RMS norm in front of the matmul (cpu::rms_norm,
// backends/cpu/ops_basic.cpp:18-33 of the reference):
//   mean = dot(x, x) / cols   (cpu::detail::dot, backends/cpu/kernel_common.h:16-27)
//   inv  = 1 / sqrt(mean + eps)
//   out  = (x * inv) * w
// Every kernel computes the sum of squares in the CPU's order, so the results are bitwise the
// CPU's: k_rms_norm_rows writes the normalized rows (the reference-order GEMV's input, and the
// RMS_NORM op itself); k_norm_to_frag writes them in bf16 as the GEMM's staged x, and k_rms_inv_rows
// only inv per row, for rows too wide for that.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "device.h"
#include "launch.h"
#include "norm_device.h"

namespace halo_mi {
namespace {

constexpr uint32_t kNormBlock = 512;
constexpr uint32_t kNormManyBlock = 256;  // for more rows than fit at once (launch_rms_norm)
constexpr uint32_t kNormChunk = 8192;  // floats of a row staged in LDS at a time
constexpr uint32_t kChainStride = dev::norm_chain_stride(kNormChunk);  // LDS floats per chain row (padded)
constexpr uint32_t kNormLds = dev::norm_lds_floats(kNormChunk);        // the chain rows, then the result

// 1 / sqrt(dot(x, x) / cols + eps) of one row, for the whole block, in cpu::detail::dot's order
// (norm_device.h): each chunk's squares are staged in LDS transposed (every load of the chunk is
// issued before the first is used: one memory round trip per chunk), lanes 0..7 of wave 0 carry
// the 8 chain sums across the chunks, then wave 0 combines them and thread 0 finishes. PT: loads
// per thread and chunk, PT * BLOCK >= min(cols, kNormChunk). v: the last chunk's elements,
// v[i] at tid + i * BLOCK (the whole row when it is one chunk); `meanwhile` runs while the
// chains do, after the last chunk's loads.
template <uint32_t BLOCK, uint32_t PT, typename F>
__device__ __forceinline__ float row_rms_inv(const float* __restrict__ x, uint32_t cols, float eps, float* lds, float (&v)[PT],
                                             F meanwhile) {
#pragma clang fp contract(off)
    const uint32_t tid = threadIdx.x;
    const uint32_t full = cols - cols % 8u;
    float p = 0.0f;
    for (uint32_t c0 = 0; c0 < cols; c0 += kNormChunk) {
        const uint32_t here = min(kNormChunk, cols - c0), n = min(here, full - min(c0, full));  // n: a multiple of 8
#pragma unroll
        for (uint32_t i = 0; i < PT; ++i) v[i] = x[c0 + min(tid + i * BLOCK, here - 1)];  // past the end: not used
        if (c0 + here == cols) meanwhile();
#pragma unroll
        for (uint32_t i = 0; i < PT; ++i) {
            const uint32_t e = tid + i * BLOCK;
            if (e < n) lds[(e % 8) * kChainStride + e / 8] = v[i] * v[i];
        }
        __syncthreads();
        if (tid < 8) p = dev::norm_chain_ahead(lds + tid * kChainStride, n / 8, p);
        __syncthreads();
    }
    if (tid < 64) {
        const float inv = dev::norm_finish(p, x, full, cols, eps, tid);
        if (tid == 0) lds[8 * kChainStride] = inv;
    }
    __syncthreads();
    return lds[8 * kChainStride];
}

// grid rows, block BLOCK. out may be x (each element is read before it is written, by
// the same thread, after the whole row has been summed). KEEP: a row of one chunk stays in registers,
// and the norm weights are loaded before the chains: what remains is the row's one round trip to
// memory and the chains (3 rows of 5120: 7.3 -> 5.6 us in the kernel trace, against 256 threads that
// read the row again for the output; 512 rows 11.0 -> 9.0). Else the row is read again for the output.
template <uint32_t BLOCK, uint32_t PT, bool KEEP>
__global__ __launch_bounds__(BLOCK) void k_rms_norm_rows(const float* x, uint64_t x_stride,
                                                              const float* __restrict__ w, float* out,
                                                              uint64_t out_stride, uint32_t cols, float eps) {
#pragma clang fp contract(off)
    __shared__ float lds[kNormLds];
    const float* xr = x + (uint64_t)blockIdx.x * x_stride;
    float* o = out + (uint64_t)blockIdx.x * out_stride;
    const uint32_t tid = threadIdx.x;
    const bool one = KEEP && cols <= kNormChunk;
    float v[PT], wv[PT];
    const float inv = row_rms_inv<BLOCK, PT>(xr, cols, eps, lds, v, [&]() __attribute__((always_inline)) {
        if (one) {
#pragma unroll
            for (uint32_t i = 0; i < PT; ++i) wv[i] = w[min(tid + i * BLOCK, cols - 1)];
        }
    });
    for (uint32_t c0 = 0; c0 < cols; c0 += kNormChunk) {
        const uint32_t n = min(kNormChunk, cols - c0);
        if (!one) {  // every load of a chunk before the first store: one memory round trip per chunk
#pragma unroll
            for (uint32_t i = 0; i < PT; ++i) {
                const uint32_t e = c0 + min(tid + i * BLOCK, n - 1);
                v[i] = xr[e];
                wv[i] = w[e];
            }
        }
#pragma unroll
        for (uint32_t i = 0; i < PT; ++i) {
            const uint32_t e = tid + i * BLOCK;
            if (e < n) {
                const float t = v[i] * inv;
                o[c0 + e] = t * wv[i];
            }
        }
    }
}

template <uint32_t BLOCK, uint32_t PT>
__global__ __launch_bounds__(BLOCK) void k_rms_inv_rows(const float* __restrict__ x, uint64_t x_stride,
                                                             uint32_t cols, float eps, float* __restrict__ inv) {
    __shared__ float lds[kNormLds];
    float v[PT];
    const float s = row_rms_inv<BLOCK, PT>(x + (uint64_t)blockIdx.x * x_stride, cols, eps, lds, v, []() {});
    if (threadIdx.x == 0) inv[blockIdx.x] = s;
}

// The GEMM's staged x with the fused norm: rows of x normalized as cpu::rms_norm rounds them,
// (x * inv) * w, then to bf16 (RNE) in the A-fragment order of k_x_to_frag (k_gemm.hip): the 8
// values of octet o (k = 8 o ..) of row m at 16-byte entry ((m / 32) * (cols / 16) + o / 2) * 64 +
// 32 (o % 2) + m % 32; rows in [n_vec, m_pad) are zero. One launch in place of k_rms_inv_rows and
// k_x_to_frag, with x read once.
// A workgroup takes kFragRows rows: their chains run side by side in one wave, in the time of one
// row's 8, and their entries of an octet are one 32-byte run. What bounds it is one round trip to
// memory and the chains; the rows stay in registers meanwhile. Thread t has octets t / 2 + 256 i of
// row t % 2. Measured on MI355X, what the norm adds to a Q4_K 5120 x 5120 GEMM at 13 / 64 / 200 / 512
// rows of x: 5.4 / 5.8 / 6.0 / 6.9 us with the two launches, 3.0 / 3.0 / 2.4 / 3.4 here; 4 rows and
// 1024 threads 4.9 / 4.9 / 4.4 / 3.2, one row and 256 threads 2.7 / 2.6 / 2.4 / 4.9.
constexpr uint32_t kFragRows = 2, kFragBlock = 512, kFragOcts = kFragBlock / kFragRows;
constexpr uint32_t kFragMaxCols = 8192;  // LDS for the squares of kFragRows rows
// LDS floats of a row's squares; rows start 32 banks apart, so a wave's writes (32 octets of 2 rows) do not collide
__host__ __device__ constexpr uint32_t frag_row_floats(uint32_t cols) {
    return 8 * dev::norm_chain_stride(cols) + ((32 - 8 * dev::norm_chain_stride(cols)) & 63u);
}

template <uint32_t IT>
__global__ __launch_bounds__(kFragBlock) void k_norm_to_frag(const float* __restrict__ x, uint64_t x_stride, uint32_t n_vec, uint32_t cols,
                                                             float eps, const float* __restrict__ w, uint4* __restrict__ out) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) float lds[];
    const uint32_t tid = threadIdx.x, row = tid % kFragRows, m = blockIdx.x * kFragRows + row, octs = cols / 8;
    const uint32_t cs = dev::norm_chain_stride(cols), rs = frag_row_floats(cols);
    const bool live = m < n_vec;
    float v[IT][8], wv[IT][8];
    auto load8 = [](const float* p, float (&d)[8]) __attribute__((always_inline)) {
        const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
        d[0] = a.x;
        d[1] = a.y;
        d[2] = a.z;
        d[3] = a.w;
        d[4] = b.x;
        d[5] = b.y;
        d[6] = b.z;
        d[7] = b.w;
    };
    if (blockIdx.x * kFragRows < n_vec) {  // (the whole workgroup: a block of padding rows only writes zeros)
#pragma unroll
        for (uint32_t i = 0; i < IT; ++i) {
            const uint32_t o = min(tid / kFragRows + kFragOcts * i, octs - 1);  // past the end: not used
            load8(x + (uint64_t)min(m, n_vec - 1) * x_stride + 8 * o, v[i]);
        }
#pragma unroll
        for (uint32_t i = 0; i < IT; ++i) {
            const uint32_t o = tid / kFragRows + kFragOcts * i;
#pragma unroll
            for (uint32_t e = 0; e < 8; ++e)
                if (o < octs) lds[row * rs + e * cs + o] = v[i][e] * v[i][e];
        }
        __syncthreads();
        // the norm weights' elements, 4-byte loads (norm_w has no more alignment), while the chains run
#pragma unroll
        for (uint32_t i = 0; i < IT; ++i) {
            const uint32_t o = min(tid / kFragRows + kFragOcts * i, octs - 1);
#pragma unroll
            for (uint32_t e = 0; e < 8; ++e) wv[i][e] = w[8 * o + e];
        }
        if (tid < 64) {
            const uint32_t r = tid / 8 % kFragRows;  // (lanes 16 .. 63 repeat the rows)
            const float p = dev::norm_chain_ahead(lds + r * rs + tid % 8 * cs, octs, 0.0f);
            const float inv = dev::norm_finish(p, x, cols, cols, eps, tid % 8);
            if (tid < 8 * kFragRows && tid % 8 == 0) lds[kFragRows * rs + r] = inv;
        }
        __syncthreads();
    }
    const float inv = live ? lds[kFragRows * rs + row] : 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < IT; ++i) {
        const uint32_t o = tid / kFragRows + kFragOcts * i;
        dev::bf16x8 b{};
        if (live) {
#pragma unroll
            for (uint32_t e = 0; e < 8; ++e) {
                const float t = v[i][e] * inv;
                b[e] = (__bf16)(t * wv[i][e]);
            }
        }
        if (o < octs) out[((uint64_t)(m / 32) * (octs / 2) + o / 2) * 64 + 32 * (o % 2) + m % 32] = __builtin_bit_cast(uint4, b);
    }
}

// Calls f(integral constant PT) with the least of 4, 8, 12, 16 loads per thread that cover a chunk of the row
template <typename F>
void with_loads(uint32_t cols, F f) {
    const uint32_t pt = (std::min(cols, kNormChunk) + kNormBlock - 1) / kNormBlock;
    if (pt <= 4) f(std::integral_constant<uint32_t, 4>{});
    else if (pt <= 8) f(std::integral_constant<uint32_t, 8>{});
    else if (pt <= 12) f(std::integral_constant<uint32_t, 12>{});
    else f(std::integral_constant<uint32_t, 16>{});
}

}  // namespace

int launch_rms_norm(const float* x, uint64_t x_stride, const float* w, float* out, uint64_t out_stride, uint32_t rows,
                    uint32_t cols, float eps, hipStream_t st) {
    if (rows == 0 || cols == 0) return HALO_MI_OK;
    // A kept row costs registers: with 16 loads per thread (above 6144 columns) a CU holds one
    // workgroup, with 6 to 12 two, where the form that reads the row again holds four. So rows that would
    // wait for a second round of those take that form (MI355X, kept over read again: 8192 columns 0.84 at 256 rows,
    // 1.26 at 257, 1.24 at 512, 1.54 at 520, 1.70 at 3000; 5120 columns 0.82 at 512, 1.07 at 520, 1.11 at 3000; 4096
    // 0.77 at 512, 1.01 at 520, 1.08 at 700, 1.11 at 3000; 3072 1.00 at 1024, 1.07 at 3000; 2048 0.65 at 512, 0.63 at 3000).
    const bool many = cols > 6144 ? rows > 256 : cols > 3072 ? rows > 512 : cols > 2048 && rows > 1024;
    auto launch = [&](auto kernel, uint32_t block) {
        hipLaunchKernelGGL(kernel, dim3(rows), dim3(block), 0, st, x, x_stride, w, out, out_stride, cols, eps);
    };
    if (many && cols > 6144) launch(k_rms_norm_rows<kNormManyBlock, 32, false>, kNormManyBlock);
    else if (many) launch(k_rms_norm_rows<kNormManyBlock, 24, false>, kNormManyBlock);
    else with_loads(cols, [&](auto pt) { launch(k_rms_norm_rows<kNormBlock, pt(), true>, kNormBlock); });
    return hip_status(hipGetLastError(), "rms_norm launch");
}

bool norm_to_frag_fits(uint32_t cols) { return cols > 0 && cols <= kFragMaxCols && cols % 32 == 0; }

int launch_norm_to_frag(const float* x, uint64_t x_stride, uint32_t n_vec, uint32_t m_pad, uint32_t cols, float eps, const float* w,
                        __bf16* out, hipStream_t st) {
    const size_t lds = (kFragRows * frag_row_floats(cols) + kFragRows) * sizeof(float);
    const dim3 grid(m_pad / kFragRows), block(kFragBlock);
    uint4* o = reinterpret_cast<uint4*>(out);
    switch ((cols / 8 + kFragOcts - 1) / kFragOcts) {
        case 1: hipLaunchKernelGGL(k_norm_to_frag<1>, grid, block, lds, st, x, x_stride, n_vec, cols, eps, w, o); break;
        case 2: hipLaunchKernelGGL(k_norm_to_frag<2>, grid, block, lds, st, x, x_stride, n_vec, cols, eps, w, o); break;
        case 3: hipLaunchKernelGGL(k_norm_to_frag<3>, grid, block, lds, st, x, x_stride, n_vec, cols, eps, w, o); break;
        default: hipLaunchKernelGGL(k_norm_to_frag<4>, grid, block, lds, st, x, x_stride, n_vec, cols, eps, w, o); break;
    }
    return hip_status(hipGetLastError(), "norm staging launch");
}

int launch_rms_inv(const float* x, uint64_t x_stride, uint32_t rows, uint32_t cols, float eps, float* inv,
                   hipStream_t st) {
    if (rows == 0 || cols == 0) return HALO_MI_OK;
    auto launch = [&](auto kernel, uint32_t block) {
        hipLaunchKernelGGL(kernel, dim3(rows), dim3(block), 0, st, x, x_stride, cols, eps, inv);
    };
    // A CU holds three workgroups of 512 threads, or four of 256, which take longer for a row: those where they
    // save a round (MI355X, what the whole 64-row GEMM of normed x takes with 512 and 256 threads, us: 10240 columns
    // 768 rows 37.2 and 38.0, 800 43.0 and 39.2, 1024 45.9 and 41.3, 1100 48.1 and 48.0; 12288 columns 1500 rows 85.3
    // and 85.9, 1024 49.7 and 44.6).
    const bool many = cols > 6144 && (rows + 767) / 768 > (rows + 1023) / 1024;
    if (many) launch(k_rms_inv_rows<kNormManyBlock, 32>, kNormManyBlock);
    else with_loads(cols, [&](auto pt) { launch(k_rms_inv_rows<kNormBlock, pt()>, kNormBlock); });
    return hip_status(hipGetLastError(), "rms_inv launch");
}

}  // namespace halo_mi
