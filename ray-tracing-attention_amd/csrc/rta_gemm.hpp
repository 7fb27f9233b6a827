// rta_gemm.hpp -- the arithmetic of the batched dequant-fused readouts on the gfx950 matrix
// cores (rta_tiled.hpp, rta_packed.hpp, rta_wide.hpp), their x slab in LDS and slab reduce.
//
// y[b, r] = sum_k W[r, k] x[b, k] with v_mfma_f32_16x16x32_f16 (fp32 accumulation).
//
//   x (A operand), prepared per (batch row, superblock of 256 columns): a power-of-two scale s puts max|x s| in [2^13, 2^14); x s is split
//   into binary16 hi + lo (22 significant bits) and both are multiplied in.  The
//   group sums the formats need (sum x over 32 for the Q4_K minimum, over 16 for
//   the Q6_K -32 offset) are prepared the same way, already in A-operand order.
//
//   Weights (B operand) are built in registers as exact binary16 values with one
//   packed multiply per two codes: a code c in the low bits of a half is the
//   subnormal c * 2^-24, and
//     Q4_K  low nibble  (c 2^-24) * (sc 2^10) = c sc 2^-14   (c sc <= 945)
//           high nibble (16 c 2^-24) * (sc 2^6) = c sc 2^-14
//     Q6_K  (4 c 2^-24) * (sc 2^8) = c sc 2^-14  (exact for |c sc| <= 2048; beyond,
//           |sc| > 32, it rounds to 11 bits, <= 2^-12 relative; the -32 offset is
//           applied exactly through the group sums)
//   so every product handed to the matrix cores is a normal binary16 (or zero).
//   The masks deliver code pairs (k, k+2); x is stored in the same order inside
//   every 8-value segment (slots 0..7 hold k = 0,2,1,3,4,6,5,7), and a common
//   permutation of k leaves the contraction unchanged.
//   Per superblock the MFMAs accumulate across all groups; the superblock's
//   scale d, the minimum / offset terms (one more MFMA over the group sums) and
//   the 1/s of x are applied once per superblock.
//
//   Lane l of a wave owns weight row l%16 and k segment l/16 (B operand), batch row l%16
//   and the same segment (A operand), and outputs (batch 4*(l/16)+e, row l%16).
//
//   Work split of up to 32 rows: the K range is cut into slabs of up to 8 (16 x rows) or 4
//   (32 x rows) superblocks, whose x a workgroup (8 waves, one per CU) keeps in LDS.  With
//   one slab the kernel applies the epilogue itself; with more it writes per-slab partial
//   sums that gemm_reduce_kernel adds in slab order (deterministic).
//
// Equivalent reference: the batched projection pipelines (optical_resident.cpp:168,343,
// matrixRows 4/8/16) and resident_batch2.comp (which accumulates in fp16; not copied).
#pragma once
#include <type_traits>
#include "rta_gemv.hpp"

namespace rta {


constexpr int kMaxBatchTile = 32;  // batch rows per GEMM launch
constexpr int kXStride = 256 + 8;  // f16 per staged x row (8 of padding spread the LDS banks)
constexpr int kGemmWaves = 8;      // waves per workgroup
constexpr int kSlabRowSb = 128;    // LDS holds (x rows) * (superblocks) <= 128

// Static LDS of the GEMM: the x slab (hi and lo planes), group-sum operands, 1/s.
template <int NBT>
struct GemmSmem {
    static constexpr int kRows = 16 * NBT;
    static constexpr int kSb = kSlabRowSb / kRows;   // superblocks per slab
    _Float16 x[kSb][2][kRows][kXStride];
    h8_t g[kSb][kRows][4];
    float inv[kSb][kRows];
};

// Adds the K-slab partials in slab order and applies the epilogue.  In kSwiglu the
// virtual rows interleave gate (even) and up (odd).  kLogits also writes per-block
// maxima pmax[b * gridDim.x + block] for the argmax.  A slab holds slab_batch rows.
template <int MODE, int NS>
__global__ void __launch_bounds__(256) gemm_reduce_kernel(const float* __restrict__ part, int nslab, int rows,
                                                          int batch, float* __restrict__ y, float* __restrict__ pmax,
                                                          int slab_batch) {
    const int total_rows = MODE == kSwiglu ? 2 * rows : rows;
    const int b = blockIdx.y;
    const int r = blockIdx.x * 256 + threadIdx.x;
    float v = -INFINITY;
    if (r < rows && b < batch) {
        // the slabs' values are loaded before the first add, 16 at a time above 16 slabs (24
        // slabs of 8 x 2048 results one by one: 6.7 us, so 3.9)
        float s = 0.0f, s2 = 0.0f;
        const float* p0 = part + (int64_t)b * total_rows;
        const int64_t ks = (int64_t)slab_batch * total_rows;
        constexpr int kAhead = NS == 0 ? 16 : NS;
        for (int k0 = 0; k0 < (NS == 0 ? nslab : 1); k0 += kAhead) {
            if constexpr (MODE == kSwiglu) {
                float2 gu[kAhead];
#pragma unroll
                for (int k = 0; k < kAhead; ++k)
                    gu[k] = *reinterpret_cast<const float2*>(p0 + min(k0 + k, nslab - 1) * ks + 2 * r);
#pragma unroll
                for (int k = 0; k < kAhead; ++k)
                    if (k0 + k < nslab) {
                        s += gu[k].x;
                        s2 += gu[k].y;
                    }
            } else {
                float t[kAhead];
#pragma unroll
                for (int k = 0; k < kAhead; ++k) t[k] = p0[min(k0 + k, nslab - 1) * ks + r];
#pragma unroll
                for (int k = 0; k < kAhead; ++k)
                    if (k0 + k < nslab) s += t[k];
            }
        }
        float* out = y + (int64_t)b * rows + r;
        if constexpr (MODE == kStore || MODE == kLogits) *out = s;
        else if constexpr (MODE == kAccumulate) *out += s;
        else *out = swiglu(s, s2);
        v = s;
    }
    if constexpr (MODE == kLogits) {
        v = wave_max_dpp(v);
        __shared__ float red[4];
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
        __syncthreads();
        if (threadIdx.x == 0 && b < batch)
            pmax[(int64_t)b * gridDim.x + blockIdx.x] = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    }
}

}  // namespace rta
