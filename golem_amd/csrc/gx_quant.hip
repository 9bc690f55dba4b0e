// gx_quant.hip - the activation quantisers of nn.Batch on the device.
//
// Q8_0 (Batch.quantizeBlock, nn/batch.go:109-143) and Q8_K (Batch.QuantizeK,
// nn/batch.go:159-213), bit for bit: IEEE division for the scale and its
// inverse (the inverse is 127/peak, a division, not 1/scale), golem's
// round-half-even (nearestInt), the Q8_0 scale rounded through fp16, and the
// Q8_K extreme taken as the first element of largest magnitude.
#include "gx_device.hpp"
#include "gx_internal.hpp"

namespace gx {
namespace {

// Four values a lane, a block per eight lanes (q8_0_quad).  x is [M][ldx];
// q [M][K], scales/qsum/corr [M][K/32]; q16 in panel order (q16_offset), over
// Mp = ceil(M/32)*32 tokens, the ones past M zero.  WIDE: x, q and q16 take
// one access a lane (rows 16-byte aligned, q 4, q16 8); else one a value.
// Bound by memory at many tokens, by the launch at few.  (One value a lane, a
// 64-bit division each and byte stores took 20 us at 2048 tokens of 2560;
// this takes 7.0 us, 26 MB in and out, and 2.0 us at one token either way.)
__global__ __launch_bounds__(256) void quantize_q8_0_kernel(const float *__restrict__ x, int ldx, int M, int Mp,
                                                            int K, bool wide, int8_t *__restrict__ q,
                                                            float *__restrict__ scales, int32_t *__restrict__ qsum,
                                                            float *__restrict__ corr, uint16_t *__restrict__ q16) {
    // Blocks of 32 values; M * K/32 fits 32 bits for any x the card can hold.
    const uint32_t index = blockIdx.x * 32u + (threadIdx.x >> 3), blocks = (uint32_t)K >> 5;
    if (index >= (uint32_t)(q16 ? Mp : M) * blocks)
        return;
    const uint32_t m = index / blocks, b = index - m * blocks;
    const int j = 4 * (threadIdx.x & 7);  // this lane's values of the block
    uint16_t *half = q16 ? q16 + q16_offset((int)m, (int)(32 * b) + j, (int)blocks) : nullptr;
    uint32_t packed = 0;
    if (m < (uint32_t)M) {
        const float *xr = x + (size_t)m * ldx + 32 * b + j;
        float v[4];
        if (wide) {
            const float4 v4 = *(const float4 *)xr;
            v[0] = v4.x, v[1] = v4.y, v[2] = v4.z, v[3] = v4.w;
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++)
                v[u] = xr[u];
        }
        float stored;
        int32_t sum;
        packed = q8_0_quad(v, &stored, &sum);
        int8_t *qr = q + (size_t)index * 32 + j;
        if (wide) {
            *(uint32_t *)qr = packed;
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++)
                qr[u] = (int8_t)(packed >> (8 * u));
        }
        if (j == 0) {
            scales[index] = stored;
            qsum[index] = sum;
            if (corr) {
                const float eight_scale = 8.0f * stored;
                corr[index] = eight_scale * (float)sum;
            }
        }
    }
    if (half) {  // the same integers as fp16 (exact: |n| <= 128); zero past M
        uint32_t h[4];
#pragma unroll
        for (int u = 0; u < 4; u++)
            h[u] = float_to_half_bits((float)(int8_t)(packed >> (8 * u)));
        if (wide) {
            *(uint2 *)half = make_uint2(h[0] | (h[1] << 16), h[2] | (h[3] << 16));
        } else {
#pragma unroll
            for (int u = 0; u < 4; u++)
                half[u] = (uint16_t)h[u];
        }
    }
}

// One wavefront per 256-element superblock, four consecutive elements per
// lane.  x is [M][ldx]; q [M][K], kscales [M][K/256], bsums [M][K/16].
__global__ __launch_bounds__(256) void quantize_q8_k_kernel(const float *__restrict__ x, int ldx, int M, int K,
                                                            int8_t *__restrict__ q, float *__restrict__ kscales,
                                                            int16_t *__restrict__ bsums) {
    const int lane = threadIdx.x & 63;
    const size_t sb = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int nsb = K / kSuper;
    if (sb >= (size_t)M * nsb)
        return;
    const int m = (int)(sb / nsb), b = (int)(sb % nsb);
    const float4 v4 = *(const float4 *)(x + (size_t)m * ldx + (size_t)b * kSuper + 4 * lane);
    const float v[4] = {v4.x, v4.y, v4.z, v4.w};
    int32_t gsum;
    float ks;
    const uint32_t packed = q8_k_wave(v, lane, &gsum, &ks);
    *(uint32_t *)(q + (size_t)m * K + (size_t)b * kSuper + 4 * lane) = packed;
    if ((lane & 3) == 0)
        bsums[(size_t)m * (K / 16) + (size_t)b * 16 + (lane >> 2)] = (int16_t)gsum;
    if (lane == 0)
        kscales[(size_t)m * nsb + b] = ks;
}

}  // namespace

int launch_quantize_q8_0(gx_ctx *ctx, const float *x, int ldx, int M, int K, int8_t *q, float *scales, int32_t *qsum,
                         float *corr, uint16_t *q16) {
    const int Mp = (M + 31) / 32 * 32;
    const size_t blocks = (size_t)(q16 ? Mp : M) * (K / 32);
    const bool wide = ldx % 4 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)q % 4 == 0 && (uintptr_t)q16 % 8 == 0;
    quantize_q8_0_kernel<<<(unsigned)((blocks + 31) / 32), 256, 0, ctx->stream>>>(x, ldx, M, Mp, K, wide, q, scales,
                                                                                  qsum, corr, q16);
    return check_launch("quantize_q8_0");
}

int launch_quantize_q8_k(gx_ctx *ctx, const float *x, int ldx, int M, int K, int8_t *q, float *kscales,
                         int16_t *bsums) {
    GX_CHECK(ldx % 4 == 0, "gx: the Q8_K quantiser needs ldx a multiple of 4");
    const size_t sbs = (size_t)M * (K / kSuper);
    const int per_block = 4;  // wavefronts per 256-thread block
    quantize_q8_k_kernel<<<(unsigned)((sbs + per_block - 1) / per_block), 64 * per_block, 0, ctx->stream>>>(
        x, ldx, M, K, q, kscales, bsums);
    return check_launch("quantize_q8_k");
}

}  // namespace gx
