// gfx950 kernels of the LM head's argmax (Backend::lm_head, include/halo/backend/backend.h:433-460
// of the reference; semantics of CpuBackend::lm_head, src/backend/cpu_backend.cpp:669-770):
//   stage 1: one ArgPart per 64 rows and vector, from a logits buffer (the slab GEMV writes the
//            same parts in its epilogue, so the fused path skips this stage);
//   stage 2: each vector's parts -> its result words {index, value bits, poisoned}, and the
//            optional dense ids and scattered ids.
// The ranking is a total order on (value, index) (higher value, then lower index), so neither
// stage depends on the reduction order: the result is the CPU's argmax over the same values.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "device.h"
#include "launch.h"

namespace halo_mi {
namespace {

using namespace dev;

// grid (parts, n_vec), block 64: part p of vector v covers rows [64 p, 64 p + 64)
__global__ __launch_bounds__(64) void k_argmax_parts(const float* __restrict__ logits, uint64_t stride, uint32_t rows,
                                                     uint32_t valid_rows, ArgPart* __restrict__ parts) {
    const uint32_t p = blockIdx.x, v = blockIdx.y, lane = threadIdx.x;
    const uint32_t row = p * 64 + lane;
    const bool live = row < rows;
    const float val = live ? logits[(uint64_t)v * stride + row] : 0.0f;
    const bool nan = live && val != val;
    const bool rank = live && !nan && (valid_rows == 0 || row < valid_rows);
    float bv;
    uint32_t bi, any_nan;
    wave_argmax(val, row, rank, nan, bv, bi, any_nan);
    if (lane == 0) parts[(uint64_t)v * gridDim.x + p] = ArgPart{bv, bi, any_nan, 0u};
}

// grid n_vec, block BLOCK. A poisoned vector (any NaN logit) reports {kNoIndex, quiet NaN, 1}
// (cpu_backend.cpp:745-747); one with no ranked row {kNoIndex, 0, 0} (TopKEntry's default,
// include/halo/backends/cpu/ops.h:351-355). ids: the winning index, 0 for either of those
// (cpu_backend.cpp:756-760); ids_scatter[ids_slots[v]] likewise, a slot past the end dropped.
// Bound by its launch and one round trip to the parts: kFinishLoads of them are in flight per thread, so
// a 248320-row head's 3880 parts take one round, and the ranking runs in registers (MI355X, that head
// with one vector, norm and logits: 194.5 -> 190.6 us; ARGMAX alone over 248320 logits 9.6 -> 6.1; against 256
// threads with one load at a time and a tree in LDS). Up to 256 parts 256 threads hold them all: with many
// vectors the idle waves of the larger block cost more than its loads save (512 vectors of 64 / 1000
// logits 5.5 / 7.2 us with 256 threads, 6.0 / 7.8 with 1024).
constexpr uint32_t kFinishBlock = 1024, kFinishSmallBlock = 256, kFinishLoads = 4;
template <uint32_t BLOCK>
__global__ __launch_bounds__(BLOCK) void k_argmax_finish(const ArgPart* __restrict__ parts, uint32_t n_parts,
                                                         uint32_t* __restrict__ result, int32_t* ids,
                                                         const uint32_t* ids_slots, int32_t* ids_scatter,
                                                         uint64_t scatter_len) {
    constexpr uint32_t kWaves = BLOCK / 64, LOADS = BLOCK == kFinishSmallBlock ? 1 : kFinishLoads;
    __shared__ float sv[kWaves];
    __shared__ uint32_t si[kWaves], sn[kWaves];
    const uint32_t v = blockIdx.x, tid = threadIdx.x, lane = tid & 63u;
    const ArgPart* mine = parts + (uint64_t)v * n_parts;
    float bv = 0.0f;
    uint32_t bi = kNoIndex, nan = 0;
    for (uint32_t i = tid; i < n_parts; i += BLOCK * LOADS) {
        ArgPart q[LOADS];
#pragma unroll
        for (uint32_t k = 0; k < LOADS; ++k) q[k] = mine[min(i + k * BLOCK, n_parts - 1)];  // (a part twice ranks once)
#pragma unroll
        for (uint32_t k = 0; k < LOADS; ++k) {
            nan |= q[k].nan;
            if (ranks_before(q[k].value, q[k].index, bv, bi)) {
                bv = q[k].value;
                bi = q[k].index;
            }
        }
    }
    float wv;
    uint32_t wi, wn;
    wave_argmax(bv, bi, bi != kNoIndex, nan != 0, wv, wi, wn);
    if (lane == 0) {
        sv[tid / 64] = wv;
        si[tid / 64] = wi;
        sn[tid / 64] = wn;
    }
    __syncthreads();
    if (tid >= 64) return;
    const bool held = lane < kWaves;
    wave_argmax(held ? sv[lane] : 0.0f, held ? si[lane] : kNoIndex, held && si[lane] != kNoIndex, held && sn[lane] != 0, bv, bi, nan);
    if (tid != 0) return;
    const bool poisoned = nan != 0;
    const uint32_t idx = poisoned ? kNoIndex : bi;
    result[3 * v] = idx;
    result[3 * v + 1] = poisoned ? 0x7FC00000u : __float_as_uint(bv);
    result[3 * v + 2] = poisoned ? 1u : 0u;
    const int32_t id = idx == kNoIndex ? 0 : (int32_t)idx;
    if (ids) ids[v] = id;
    if (ids_scatter) {
        const uint32_t slot = ids_slots[v];
        if (slot < scatter_len) ids_scatter[slot] = id;
    }
}

}  // namespace

int launch_argmax_parts(const float* logits, uint64_t stride, uint32_t rows, uint32_t n_vec, uint32_t valid_rows,
                        ArgPart* parts, hipStream_t st) {
    const uint32_t n_parts = (rows + 63) / 64;
    hipLaunchKernelGGL(k_argmax_parts, dim3(n_parts, n_vec), dim3(64), 0, st, logits, stride, rows, valid_rows, parts);
    return hip_status(hipGetLastError(), "argmax_parts launch");
}

int launch_argmax_finish(const ArgPart* parts, uint32_t n_parts, uint32_t n_vec, uint32_t* result, int32_t* ids,
                         const uint32_t* ids_slots, int32_t* ids_scatter, uint64_t scatter_len, hipStream_t st) {
    auto launch = [&](auto kernel, uint32_t block) {
        hipLaunchKernelGGL(kernel, dim3(n_vec), dim3(block), 0, st, parts, n_parts, result, ids, ids_slots, ids_scatter, scatter_len);
    };
    if (n_parts <= kFinishSmallBlock) launch(k_argmax_finish<kFinishSmallBlock>, kFinishSmallBlock);
    else launch(k_argmax_finish<kFinishBlock>, kFinishBlock);
    return hip_status(hipGetLastError(), "argmax_finish launch");
}

}  // namespace halo_mi
