// gx_gemm.hip - the Q4_0 x Q8_0 product for a batch of tokens (prefill) on
// int8 MFMA.
//
// golem reads a prompt through the same MatVecBatch as a single token, with
// the batch as the inner loop (nn/matrix.go:67-81, nn/pack_q4_0.go:159-221).
// Here the batch is a real dense contraction: v_mfma_i32_32x32x32_i8 takes one
// Q4_0 block (32 inputs) of 32 rows against the same block of 32 tokens and
// returns the exact per-block integers; the fp32 scales are applied to them
// per block in the canonical order of the matrix-vector kernel
// (gx_q4_0.hip), stretch by stretch, so a token's result is bit-identical
// whether it came through this kernel or that one.
//
// The per-block epilogue is what bounds this product: every output element
// needs float(isum) * (d_w * d_a) added to its sum, per block.  The scale
// product d_w[i] * d_a[j] of a 32x32 tile is an outer product of two fp16
// vectors (golem stores d_a, the Q8_0 scale, already rounded through fp16),
// so it comes from the matrix core too: v_mfma_f32_32x32x8_f16 with the two
// vectors in k = 0 and zeros elsewhere gives every product exactly (an
// 11-bit by 11-bit product fits fp32; the int8 kernel puts them in k = 0 and
// k = 4 and takes 2 d_w d_a).  The vector ALU is left with one fma per
// element per block.
//
// Two kernels: the int8 one below (loads straight into LDS, every Q4_0
// product of more than a few tokens, dense or grouped by expert) and an fp16
// one for callers that hold the activation's fp16 copy.  The weights'
// nibbles are widened to signed int8 (n - 8) in registers as they are read.
#include <algorithm>
#include <type_traits>

#include "gx_device.hpp"
#include "gx_internal.hpp"

namespace gx {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// A 32x32x8 f16 operand holding the fp16 bits `h` at k = 0 (lanes 0..31,
// element 0) and zeros everywhere else.
__device__ __forceinline__ v4h k0_operand(uint32_t h, bool first_half) {
    const uint2 bits = make_uint2(first_half ? (h & 0xFFFFu) : 0u, 0u);
    return __builtin_bit_cast(v4h, bits);
}

// The same operand in both halves of the wavefront (k = 0 and k = 4): the
// outer product then holds every d_w[i] * d_a[j] twice, 2 d_w d_a, exactly.
// `h` has its upper 16 bits clear (a u16 LDS read, or a VOP1 fp16 result).
__device__ __forceinline__ v4h k04_operand(uint32_t h) {
    return __builtin_bit_cast(v4h, make_uint2(h, 0u));
}

// {fp16(f), +0} as one dword, in one instruction.  Exact for a value that fp16
// holds, whatever the rounding (the Q8_0 activation scales are fp16 values).
__device__ __forceinline__ uint32_t half2_bits_rtz(float f) {
    return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(f, 0.0f));
}


// Blocks a pipeline stage holds (half a stretch).
constexpr int kStage = 4;

// A mixture-of-experts product runs grouped: workgroup row y of the grid is
// work item y, {expert, first, count}, covering units sorted[first ..
// first + count) of one expert (count 0: nothing to do).  Unit u reads
// activation row u / act_div and writes output row u.
struct Groups {
    const int32_t *work;
    const int32_t *sorted;
    int act_div;
    size_t matrix_bytes;
};

// ---- the fp16 product ------------------------------------------------------
//
// The same contraction with the per-block integers taken by
// v_mfma_f32_32x32x16_f16 from integer-valued fp16 operands: the weights
// (n - 8) and the Q8_0 values q, both exact in fp16.  Every product and every
// partial sum is an integer below 2^24 in magnitude, so the fp32 result is
// the exact per-block integer, already a float: the epilogue is one fma per
// element per block, where the int8 kernel needs a conversion and an fma.
//
// Tile: a workgroup owns 64 rows (one R64 tile) x 32*NWT tokens; wavefront w
// owns the 64 rows x token group w (32 tokens): two 32x32 MFMA tiles sharing
// the activation operand.  The rows' nibbles are widened to fp16 once per
// workgroup into LDS, four blocks per stage, double buffered: the next
// stage's nibbles are in flight while this one's MFMAs run.  Each wavefront
// reads its activation operands straight from the panel-ordered fp16 copy
// (q16_offset): one contiguous 1 KiB per operand, one block ahead.
constexpr int kFStage = 4;   // blocks per stage
constexpr int kFWRow = 40;   // halves per staged weight row (32 + pad: 80-byte rows)

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

// Four nibbles (one per byte, values 0..15) -> four fp16 values n - 8, as two
// dwords.  0x64 above a byte makes the fp16 1024 + n; subtracting 1032 is
// exact.
__device__ __forceinline__ void nibbles_to_f16(uint32_t n, uint32_t &lo, uint32_t &hi) {
    const uint32_t a = __builtin_amdgcn_perm(0x64646464u, n, 0x04010400u);
    const uint32_t b = __builtin_amdgcn_perm(0x64646464u, n, 0x04030402u);
    const v2h bias = {(_Float16)1032.0f, (_Float16)1032.0f};
    lo = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, a) - bias);
    hi = __builtin_bit_cast(uint32_t, __builtin_bit_cast(v2h, b) - bias);
}

// One block row of nibbles (16 bytes) -> its 32 fp16 weights in golem's
// order in LDS: [0,16) from the low nibbles of bytes 0..15, [16,32) from the
// high nibbles.
__device__ __forceinline__ void widen_row(const v4u &w, uint16_t *row) {
    const uint32_t words[4] = {w.x, w.y, w.z, w.w};
    uint32_t out[16];
#pragma unroll
    for (int k = 0; k < 4; k++) {
        nibbles_to_f16(words[k] & 0x0F0F0F0Fu, out[2 * k], out[2 * k + 1]);
        nibbles_to_f16((words[k] >> 4) & 0x0F0F0F0Fu, out[8 + 2 * k], out[8 + 2 * k + 1]);
    }
#pragma unroll
    for (int k = 0; k < 4; k++)
        *(v4u *)(row + 8 * k) = (v4u){out[4 * k], out[4 * k + 1], out[4 * k + 2], out[4 * k + 3]};
}

template <int NWT, bool DOTS>
__global__ __launch_bounds__(64 * NWT) void q4_0_gemm_f16_kernel(
    const uint8_t *__restrict__ W, size_t plane0_bytes, int B, int DC, const uint16_t *__restrict__ q16,
    const float *__restrict__ scales, int M, int tile0, int row_start, int row_end, const float *__restrict__ bias,
    float *__restrict__ y, int ldy, int32_t *__restrict__ dots) {
    constexpr int NT = 64 * NWT;
    constexpr int RW = (kFStage * kTileRows + NT - 1) / NT;  // 16-byte nibble chunks per thread per stage
    __shared__ __attribute__((aligned(16))) uint16_t wl[2][kFStage][kTileRows][kFWRow];
    __shared__ uint16_t dwl[2][kFStage][kTileRows];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = tid >> 6, li = lane & 31, g = lane >> 5;
    const int tile = tile0 + blockIdx.x;
    const int n0 = tile * kTileRows;
    const int Gn = (M + 31) / 32;
    const int G = blockIdx.y * NWT + wv;  // this wavefront's token group
    const int Gc = min(G, Gn - 1);
    const int t = 32 * G + li;            // this lane's token
    const float *srow = scales ? scales + (size_t)min(t, M - 1) * B : nullptr;
    const uint16_t *panel = q16 + (size_t)Gc * B * 1024 + 8 * lane;  // + (2b + h) * 512
    const int S = (B + kFStage - 1) / kFStage;
    const int nrows = row_end - row_start;

    // Stage h's nibbles: chunk c (block c / 64, row c % 64) for c = tid + NT i;
    // clamped past the last block (never used).  Scales: rows tid < 64, the
    // 8 bytes of the row's scale chunk that hold the stage's 4 blocks.
    v4u raw[RW];
    uint2 sraw = make_uint2(0, 0);
    auto fetch_w = [&](int h, v4u (&r)[RW], uint2 &sr) {
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const int c = min(tid + NT * i, kFStage * kTileRows - 1);
            const int b = min(h * kFStage + (c >> 6), B - 1);
            r[i] = *(const v4u *)(W + (((size_t)tile * B + b) * kTileRows + (c & 63)) * kChunk);
        }
        if (!DOTS && tid < kTileRows) {
            const int b0 = h * kFStage;
            sr = *(const uint2 *)(W + plane0_bytes + (((size_t)tile * DC + (b0 >> 3)) * kTileRows + tid) * kChunk +
                                  2 * (b0 & 7));
        }
    };
    auto commit_w = [&](int buf, const v4u (&r)[RW], const uint2 &sr) {
#pragma unroll
        for (int i = 0; i < RW; i++) {
            const int c = tid + NT * i;
            if (c < kFStage * kTileRows)
                widen_row(r[i], wl[buf][c >> 6][c & 63]);
        }
        if (!DOTS && tid < kTileRows) {
            dwl[buf][0][tid] = (uint16_t)(sr.x & 0xFFFFu);
            dwl[buf][1][tid] = (uint16_t)(sr.x >> 16);
            dwl[buf][2][tid] = (uint16_t)(sr.y & 0xFFFFu);
            dwl[buf][3][tid] = (uint16_t)(sr.y >> 16);
        }
    };

    v16f acc0, acc1, tot0, tot1;
#pragma unroll
    for (int e = 0; e < 16; e++)
        acc0[e] = acc1[e] = tot0[e] = tot1[e] = 0.0f;
    const v16f zero_f = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    // Activation operands a stage ahead, in two register sets that alternate
    // by stage (the stage loop is unrolled by two, so each set's registers are
    // fixed): slot j of a set holds block 4s + j's two panels and scale
    // (clamped past the last block; never used there).
    v8h PA0[kFStage], PA1[kFStage], PB0[kFStage], PB1[kFStage];
    float dA[kFStage], dB[kFStage];
#define GX_F16_LOAD_SET(P0, P1, DS, s)                                                                               \
    do {                                                                                                             \
        for (int j = 0; j < kFStage; j++) {                                                                          \
            const int bn = min((s) * kFStage + j, B - 1);                                                            \
            P0[j] = *(const v8h *)(panel + (size_t)(2 * bn) * 512);                                                  \
            P1[j] = *(const v8h *)(panel + (size_t)(2 * bn + 1) * 512);                                              \
            DS[j] = DOTS ? 0.0f : srow[bn];                                                                          \
        }                                                                                                            \
    } while (0)

// One stage, software-pipelined across the two row tiles: tile 0's MFMAs for
// block j, then tile 1's fmas for block j - 1 (results of the previous
// block's MFMAs), then tile 1's MFMAs for block j, then tile 0's fmas for
// block j -- each batch of fmas runs while an independent batch of MFMAs is
// in the matrix core.  `pend` is the block whose tile-1 fmas are pending (-1:
// none).
#define GX_F16_FMA(D, SC, ACC, TOT, bb)                                                                              \
    do {                                                                                                             \
        for (int e = 0; e < 16; e++)                                                                                 \
            ACC[e] = fmaf(D[e], SC[e], ACC[e]);                                                                      \
        if (((bb) & (kStretch - 1)) == kStretch - 1 || (bb) == B - 1) { /* a stretch ends */                         \
            for (int e = 0; e < 16; e++) {                                                                           \
                TOT[e] = TOT[e] + ACC[e];                                                                            \
                ACC[e] = 0.0f;                                                                                       \
            }                                                                                                        \
        }                                                                                                            \
    } while (0)

#define GX_F16_DOTS(D, roff, bb)                                                                                     \
    do {                                                                                                             \
        if (t < M) {                                                                                                 \
            for (int e = 0; e < 16; e++) {                                                                           \
                const int n = n0 + (roff) + 8 * (e >> 2) + 4 * g + (e & 3);                                          \
                if (n >= row_start && n < row_end)                                                                   \
                    dots[((size_t)t * nrows + (n - row_start)) * B + (bb)] = (int32_t)D[e];                          \
            }                                                                                                        \
        }                                                                                                            \
    } while (0)

#define GX_F16_STAGE(P0, P1, DS, h)                                                                                  \
    do {                                                                                                             \
        const int buf = (h) & 1;                                                                                     \
        const int nb = min(kFStage, B - (h) * kFStage);                                                              \
        for (int j = 0; j < kFStage; j++) {                                                                          \
            if (j < nb) {                                                                                            \
                const int b = (h) * kFStage + j;                                                                     \
                const v4h Bs = k0_operand(float_to_half_bits(DS[j]), g == 0);                                        \
                {                                                                                                    \
                    const v8h A00 = *(const v8h *)&wl[buf][j][li][8 * g];                                            \
                    const v8h A01 = *(const v8h *)&wl[buf][j][li][16 + 8 * g];                                       \
                    D0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A00, P0[j], zero_f, 0, 0, 0);                         \
                    D0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A01, P1[j], D0, 0, 0, 0);                            \
                    if (!DOTS)                                                                                       \
                        S0 = __builtin_amdgcn_mfma_f32_32x32x8f16(k0_operand(dwl[buf][j][li], g == 0), Bs, zero_f,  \
                                                                  0, 0, 0);                                          \
                }                                                                                                    \
                if (!DOTS && pend >= 0)                                                                              \
                    GX_F16_FMA(D1, S1, acc1, tot1, pend);                                                            \
                {                                                                                                    \
                    const v8h A10 = *(const v8h *)&wl[buf][j][32 + li][8 * g];                                       \
                    const v8h A11 = *(const v8h *)&wl[buf][j][32 + li][16 + 8 * g];                                  \
                    D1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A10, P0[j], zero_f, 0, 0, 0);                         \
                    D1 = __builtin_amdgcn_mfma_f32_32x32x16_f16(A11, P1[j], D1, 0, 0, 0);                            \
                    if (!DOTS)                                                                                       \
                        S1 = __builtin_amdgcn_mfma_f32_32x32x8f16(k0_operand(dwl[buf][j][32 + li], g == 0), Bs,     \
                                                                  zero_f, 0, 0, 0);                                  \
                }                                                                                                    \
                if (DOTS) {                                                                                          \
                    GX_F16_DOTS(D0, 0, b);                                                                           \
                    GX_F16_DOTS(D1, 32, b);                                                                          \
                } else {                                                                                             \
                    GX_F16_FMA(D0, S0, acc0, tot0, b);                                                               \
                }                                                                                                    \
                pend = b;                                                                                            \
            }                                                                                                        \
        }                                                                                                            \
    } while (0)

    v16f D0 = zero_f, D1 = zero_f, S0 = zero_f, S1 = zero_f;
    int pend = -1;
    fetch_w(0, raw, sraw);
    GX_F16_LOAD_SET(PA0, PA1, dA, 0);
    commit_w(0, raw, sraw);
    __syncthreads();
    for (int h = 0; h < S; h += 2) {  // set A holds stage h
        if (h + 1 < S) {  // in flight during this stage's arithmetic
            fetch_w(h + 1, raw, sraw);
            GX_F16_LOAD_SET(PB0, PB1, dB, h + 1);
        }
        GX_F16_STAGE(PA0, PA1, dA, h);
        if (h + 1 >= S)
            break;
        commit_w((h + 1) & 1, raw, sraw);
        __syncthreads();
        if (h + 2 < S) {
            fetch_w(h + 2, raw, sraw);
            GX_F16_LOAD_SET(PA0, PA1, dA, h + 2);
        }
        GX_F16_STAGE(PB0, PB1, dB, h + 1);
        if (h + 2 < S) {
            commit_w(h & 1, raw, sraw);
            __syncthreads();
        }
    }
    if (!DOTS && pend >= 0)  // the last block's tile-1 fmas
        GX_F16_FMA(D1, S1, acc1, tot1, pend);
#undef GX_F16_LOAD_SET
#undef GX_F16_STAGE
#undef GX_F16_FMA
#undef GX_F16_DOTS
    if (DOTS || t >= M)
        return;
#pragma unroll
    for (int e = 0; e < 16; e++) {
        const int r = 8 * (e >> 2) + 4 * g + (e & 3);
        const int na = n0 + r, nb2 = n0 + 32 + r;
        if (na >= row_start && na < row_end)
            y[(size_t)t * ldy + na] = bias ? tot0[e] + bias[na] : tot0[e];
        if (nb2 >= row_start && nb2 < row_end)
            y[(size_t)t * ldy + nb2] = bias ? tot1[e] + bias[nb2] : tot1[e];
    }
}


// ---- the int8 product, loads straight into LDS -------------------------
//
// The kernel for the Q4_0 x Q8_0 product of a batch.  Every stage's operands
// come in by direct global-to-LDS loads (global_load_lds_dwordx4 / _dword):
// no registers stage them, and the stages live in an LDS ring of kRing slots,
// all but one in flight while one is multiplied.  Per stage (4 blocks) each
// wavefront issues exactly kLoads loads, so `s_waitcnt vmcnt((kRing - 2)
// kLoads)` before the stage's barrier means "this stage has landed" for every
// wavefront; the barrier is the bare s_barrier (the fence of __syncthreads
// would wait for every load in flight).  A stage's loads go out one or two a
// tile, and a block's operands are read from LDS a block ahead, across
// stages.
//
// What bounds it: a tile and block take three MFMAs (96 cycles of the matrix
// core) and about 23 vector instructions, which mostly add up; under that
// load the clock is 2.1 GHz.  Taken out of a copy, the loads changed 126 us
// to 122 and the stores to 114 (9728 x 2560 at 2048 tokens).  With a token a
// lane in the activation's loads, the subtraction on the vector ALU and one
// 32x32 tile a wavefront throughout the same product took 175 us (0.117 of
// the int8 rate; now 0.162), 49 at 500 tokens (now 38), 2560 x 9728 at 500 64
// (now 51), a mixture layer of 128 experts at 256 positions 175 (159).
//
// The integer products are taken as floats without a conversion.  The weights
// enter the MFMA as 16 * (n - 8) (the nibble in a byte's high half, its top
// bit flipped) and its addend is the bits of 0.1875, the middle of the binade
// [1/8, 1/4): a block's 16 * isum is at most 16 * 32 * 8 * 128 = 2^19 in
// magnitude, 2^3 less than the 2^22 ulps to either end, so the output read as
// fp32 is 0.1875 + 16 * isum * 2^-26 exactly, and no block waits for the one
// before it.  A second MFMA (1 * -0.1875 added to that output) leaves
// isum * 2^-22 exactly: a sixteen-instruction subtraction taken off the
// vector ALU, whose instructions, not the matrix core's, bound the product
// (the two units' times add up on a SIMD; 57 -> 52 ns a tile and block).  The
// scale outer product is 2 d_w d_a (k04_operand), so a stretch's sums, and
// the total, are golem's times 2^-21, rounded where golem's are (a power of
// two moves no rounding; the least term that is not zero is 2^-69): the total
// is multiplied by 2^21 once, exactly.
constexpr int kIntBias = 0x3E400000;     // 0.1875
constexpr float kUnscale = 2097152.0f;   // 2^21

// One block's operands from LDS (a row's nibble chunk, a token's 16 bytes),
// issued without a wait.  Written out so that the compiler sees no LDS load:
// it would otherwise make each one wait for every load-to-LDS in flight, the
// next stages' included.  The caller waits (lgkmcnt) before it uses them.
template <int OFF>
__device__ __forceinline__ void lds_read_b128(uint32_t at, v4u &r) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=&v"(r) : "v"(at), "i"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read_b32(uint32_t at, uint32_t &r) {
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=&v"(r) : "v"(at), "i"(OFF));
}
template <int OFF>
__device__ __forceinline__ void lds_read_u16(uint32_t at, uint32_t &r) {
    asm volatile("ds_read_u16 %0, %1 offset:%2" : "=&v"(r) : "v"(at), "i"(OFF));
}

template <int J, int N, typename F>
__device__ __forceinline__ void unroll(F &&f) {  // f(integral_constant<int, J>) for J in [J, N)
    if constexpr (J < N) {
        f(std::integral_constant<int, J>{});
        unroll<J + 1, N>(f);
    }
}

// A tile shape of the product: WR x WT wavefronts of 32 rows x 32 * TT tokens.
// Slot bytes of a stage:
//   [0, kAct)             nibbles  [block 4][row kRows][16]
//   [kAct, kActScale)     int8     [token kTok][16-byte piece 8], piece p of
//                         token t in place p ^ (t & 7)
//   [kActScale, kWScale)  act. scales (fp32) [token kTok][block 4]
//   [kWScale, kDummy)     weight scales (fp16) [row kRows][block 4]
//   [kDummy, + 256)       where loads go that only keep the count even
// The activation comes in eight tokens' whole 128-byte stage rows a load
// (eight lines; a token a lane touched 64, and its scales, a dword a lane, 64
// more: the CU's address path, one line a clock, then set the product's
// time), and the places' exclusive-or spreads eight tokens' same piece over
// all banks when it is read.
template <int TT, int WR, int WT, int RING, int OCC>
struct GemmShape {
    static constexpr int kTT = TT, kWR = WR, kWT = WT, kRing = RING, kOcc = OCC;
    static constexpr int kRows = 32 * WR, kTok = 32 * TT * WT, kWaves = WR * WT, kThreads = 64 * kWaves;
    static constexpr int kWLoads = kRows / 16 / kWaves, kALoads = kTok / 8 / kWaves;
    static constexpr int kSLoads = (kTok / 16 + kWaves - 1) / kWaves, kDLoads = (kRows / 32 + kWaves - 1) / kWaves;
    static constexpr int kLoads = kWLoads + kALoads + kSLoads + kDLoads;
    static constexpr int kAct = kRows * 64, kActScale = kAct + kTok * 128, kWScale = kActScale + kTok * 16,
                         kDummy = kWScale + kRows * 8;
    static constexpr bool kPad = kSLoads * kWaves > kTok / 16 || kDLoads * kWaves > kRows / 32;
    static constexpr int kSlot = kDummy + (kPad ? 256 : 0);
    static_assert(kRows % 64 == 0 && kWLoads * kWaves * 16 == kRows && kALoads * kWaves * 8 == kTok, "whole loads");
    static_assert((RING - 1) * kSlot + (3 * kRows * 16 > TT * 4096 ? 3 * kRows * 16 : TT * 4096) < 65536, "a read's slot and block are its immediate offset");
    static_assert(RING * kSlot <= 160 * 1024, "the ring fits the LDS");
};

// EPI 2's epilogue (see the kernel): 4 wavefronts, wavefront rg holding
// rows 32 rg .. of the workgroup's 128 for tokens first + li.  Element e of
// a rotated head: pair j = e % half, a = re c - im s (e < half), b = re s +
// im c, re = x_j sc g_j, im = x_{j+half} sc g_{j+half} (RoPETable.Apply,
// nn/rope.go:62-73; qwen/attention.go:57-84, qwen/cache.go:52-60).
constexpr int kQkvStride = 129;  // a token's staged row: a lane a token reads down a column without conflicts

__device__ __forceinline__ void qkv_rope_epilogue(const v16f &tot, uint8_t *lds, const QkvRopeArgs &qr, int T0,
                                                  int rg, int li, int g, int first, int count) {
    const int tid = threadIdx.x;
    const int hd = qr.hd, half = hd >> 1, P = hd >> 3, hpw = 128 / hd;  // pieces a head; heads a workgroup
    const int nheads = qr.heads + 2 * qr.kv_heads;
    const int h0 = T0 * kTileRows / hd;  // the workgroup's first head
    float *hs = (float *)lds;                       // [32 tokens][kQkvStride]
    float *gs = hs + 32 * kQkvStride;               // [128]: each row's gain
    float *scs = gs + 128;                          // [2][32] norm scales
    int *pos_s = (int *)(scs + 64), *place_s = pos_s + 32, *slot_s = place_s + 32;
    __syncthreads();  // every wavefront is past its last operand reads
#pragma unroll
    for (int e = 0; e < 16; e++)
        hs[li * kQkvStride + 32 * rg + 8 * (e >> 2) + 4 * g + (e & 3)] = tot[e];
    // section of head k of the workgroup: 0 query, 1 key, 2 value, 3 none
    auto section = [&](int k) -> int {
        const int hg = h0 + k;
        return hg < qr.heads ? 0 : hg < qr.heads + qr.kv_heads ? 1 : hg < nheads ? 2 : 3;
    };
    if (tid < 32) {
        int pl = -1, pos = 0, sl = 0;
        if (tid < count) {
            const int t = first + tid;
            pos = qr.positions[t];
            sl = qr.slots ? qr.slots[t] : 0;
            pl = pos >= 0 && pos < qr.context && (!qr.slots || (sl >= 0 && sl < qr.nslots)) ? 1 : 0;
        }
        pos_s[tid] = pos;
        place_s[tid] = pl;
        slot_s[tid] = sl;
    } else if (tid >= 64 && tid < 192) {
        const int r = tid - 64, sec = section(r / hd);
        gs[r] = sec == 0 ? qr.q_norm[r % hd] : sec == 1 ? qr.k_norm[r % hd] : 0.0f;
    }
    __syncthreads();
    // (head, token, piece) items of the query and key heads, two a thread:
    // a query's pieces fastest (contiguous in qh), a key's tokens fastest
    // (a piece's positions are contiguous in the cache).  Their rotation
    // tables go out now, while the norms' sums run.
    float4 c0[2], c1[2], s0[2], s1[2];
    int ik[2], itk[2], ipc[2], isec[2];
#pragma unroll
    for (int it = 0; it < 2; it++) {
        const int idx = tid + 256 * it, k = idx / (32 * P), rem = idx - k * 32 * P;
        const int sec = section(k);
        const int tk = sec == 0 ? rem / P : rem & 31, pc = sec == 0 ? rem % P : rem >> 5;
        ik[it] = k, itk[it] = tk, ipc[it] = pc, isec[it] = sec;
        if (sec <= 1 && place_s[tk] > 0) {
            const int pos = pos_s[tk];
            const int j0 = 8 * pc < half ? 8 * pc : 8 * pc - half;
            c0[it] = *(const float4 *)(qr.rope_cos + (size_t)pos * half + j0);
            c1[it] = *(const float4 *)(qr.rope_cos + (size_t)pos * half + j0 + 4);
            s0[it] = *(const float4 *)(qr.rope_sin + (size_t)pos * half + j0);
            s1[it] = *(const float4 *)(qr.rope_sin + (size_t)pos * half + j0 + 4);
        }
    }
    if (tid < 32 * hpw) {
        // head_norm_scale's sum, left to right, sixteen values read ahead
        const int k = tid >> 5, tk = tid & 31;
        if (section(k) <= 1 && tk < count) {
            const float *hr = hs + tk * kQkvStride + k * hd;
            double acc = 0.0;
            for (int i0 = 0; i0 < hd; i0 += 16) {
                float v[16];
#pragma unroll
                for (int i = 0; i < 16; i++)
                    v[i] = hr[i0 + i];
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float sq = v[i] * v[i];
                    acc += (double)sq;
                }
            }
            const float mean = (float)(acc / (double)hd);
            scs[tid] = (float)(1.0 / sqrt((double)(mean + qr.eps)));
        }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < 2; it++) {
        const int k = ik[it], tk = itk[it], pc = ipc[it], sec = isec[it];
        const int pl = place_s[tk];
        if (sec > 1 || pl < 0)
            continue;
        const int pos = pos_s[tk], hg = h0 + k;
        uint32_t w[4] = {0x7E007E00u, 0x7E007E00u, 0x7E007E00u, 0x7E007E00u};  // no place: a NaN query
        if (pl) {
            const bool lo = 8 * pc < half;
            const int j0 = lo ? 8 * pc : 8 * pc - half;
            const float cs[8] = {c0[it].x, c0[it].y, c0[it].z, c0[it].w, c1[it].x, c1[it].y, c1[it].z, c1[it].w};
            const float sn[8] = {s0[it].x, s0[it].y, s0[it].z, s0[it].w, s1[it].x, s1[it].y, s1[it].z, s1[it].w};
            const float sc = scs[k * 32 + tk];
            const float *hr = hs + tk * kQkvStride + k * hd;
            const float *gr = gs + k * hd;
            uint32_t hb[8];
#pragma unroll
            for (int kk = 0; kk < 8; kk++) {
                const int j = j0 + kk;
                const float re = (hr[j] * sc) * gr[j], im = (hr[j + half] * sc) * gr[j + half];
                const float v = lo ? re * cs[kk] - im * sn[kk] : re * sn[kk] + im * cs[kk];
                hb[kk] = float_to_half_bits(v);
            }
#pragma unroll
            for (int kk = 0; kk < 4; kk++)
                w[kk] = hb[2 * kk] | (hb[2 * kk + 1] << 16);
        }
        const v4u_stream o = {w[0], w[1], w[2], w[3]};
        if (sec == 0) {
            *(v4u_stream *)(qr.qh + (size_t)(first + tk) * qr.heads * hd + (size_t)hg * hd + 8 * pc) = o;
        } else if (pl) {
            uint16_t *kt = qr.kcache + (size_t)slot_s[tk] * qr.kv_heads * hd * qr.context +
                           (size_t)(hg - qr.heads) * hd * qr.context;
            *(v4u_stream *)(kt + ((size_t)pc * qr.context + pos) * 8) = o;
        }
    }
    // the value heads: a lane a token down each element row
    for (int k = 0; k < hpw; k++) {
        if (section(k) != 2)
            continue;
        const int kvh = h0 + k - qr.heads - qr.kv_heads;
        for (int idx = tid; idx < 32 * hd; idx += 256) {
            const int tk = idx & 31, d = idx >> 5;
            if (place_s[tk] > 0) {
                uint16_t *vt = qr.vcache + (size_t)slot_s[tk] * qr.kv_heads * hd * qr.context +
                               (size_t)kvh * hd * qr.context;
                vt[(size_t)d * qr.context + pos_s[tk]] = (uint16_t)float_to_half_bits(hs[tk * kQkvStride + k * hd + d]);
            }
        }
    }
}

// GROUPED: blockIdx.y is an item of the expert work list (grp.work[item] =
// {expert, first, count <= kTok, 0}; count 0 past the last item): the item's
// tokens are units sorted[first ..], token t reading activation row
// sorted[first + t] / act_div and writing output row sorted[first + t], all
// against expert grp.work[item].x of the stack (matrices matrix_bytes
// apart).  Otherwise tokens kTok * blockIdx.y .. of the batch.
//
// DOTS: the same kernel, also writing every block's integer (x below) to
// dots[out row][n - row_start][b]; the scales are then not needed, and their
// loads read the activation instead (in bounds).
//
// EPI 1 (dense, whole matrix): the rows are gate and up interleaved by 32 (a
// tile's rows 0..31 gate, 32..63 up, for the same 32 outputs), and the
// product ends in silu(gate) * up and its Q8_0 (qwen_swiglu_quant_kernel's
// arithmetic, element for element) into mq / ms / mqs [M][rows / 2]: the
// wavefront of a tile's up rows passes its sums through LDS to the
// wavefront of the gate rows, whose lane pair (l, l + 32) holds one token's
// 32 outputs, one Q8_0 block.
//
// EPI 2 (dense, whole matrix, four wavefronts of rows): the rows are the
// query, key and value heads stacked (hd = 64 or 128 rows a head, so a
// workgroup's 128 rows are whole heads), and the product ends in
// qwen_qk_rope_tile_kernel's work for its heads, 32 tokens at a time, bit for
// bit: the sums staged in LDS by token, a query or key head's RMSNormPlain
// (float64, left to right, a lane a token), RoPE with golem's tables, fp16,
// the query into qr.qh and the key and value into the caches -- without the
// [M][rows] float round trip.
template <typename Sh, bool GROUPED, bool DOTS, int EPI>
__global__ __launch_bounds__(Sh::kThreads, DOTS ? 1 : Sh::kOcc) void q4_0_gemm_kernel(
    const uint8_t *__restrict__ W, size_t plane0_bytes, int B, int DC, const int8_t *__restrict__ q,
    const float *__restrict__ scales, int K, int M, int tiles, int tile0, int row_start, int row_end,
    const float *__restrict__ bias, float *__restrict__ y, int ldy, int32_t *__restrict__ dots, Groups grp,
    int xcd_cols, int8_t *__restrict__ mq, float *__restrict__ ms, int32_t *__restrict__ mqs, QkvRopeArgs qr) {
    constexpr int kSlotB = Sh::kSlot, kRing = Sh::kRing, TT = Sh::kTT, kWaves = Sh::kWaves, kTok = Sh::kTok;
    constexpr int kTilesWg = Sh::kRows / kTileRows;
    constexpr int kA0 = Sh::kWLoads, kS0 = kA0 + Sh::kALoads, kD0 = kS0 + Sh::kSLoads, kLoads = Sh::kLoads;
    __shared__ __align__(16) uint8_t ring_lds[kRing * kSlotB];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // The workgroup's row group bx and token group by.  With xcd_cols > 0 the
    // grid is one-dimensional in the dispatcher's XCD order (workgroup i runs
    // on XCD i % 8): XCD x takes row groups [x P / 8, (x + 1) P / 8) of the P
    // and every token group, token group by token group, so that its L2
    // holds its rows' weights while the tokens stream past once.  (A 2-D
    // grid deals every XCD all row groups: each L2 refetches the whole matrix
    // many times over.)
    int bx = blockIdx.x, by = blockIdx.y;
    if (!GROUPED && xcd_cols > 0) {
        const int x = blockIdx.x & 7, local = blockIdx.x >> 3;
        const int lo = x * xcd_cols / 8, n = (x + 1) * xcd_cols / 8 - lo;
        if (local >= n * ((M + kTok - 1) / kTok))
            return;  // this XCD's share is done: the whole workgroup
        by = local / n;
        bx = lo + (local - by * n);
    }
    const int T0 = tile0 + kTilesWg * bx;                 // the workgroup's first R64 tile
    const int rg = wv % Sh::kWR, tg = wv / Sh::kWR;       // this wavefront's 32 rows and 32 * TT tokens
    const int li = lane & 31, g = lane >> 5;
    int first, count;
    if (GROUPED) {
        const int4 item = ((const int4 *)grp.work)[by];
        count = item.z;
        if (count <= 0)
            return;  // past the last item: the whole workgroup
        W += (size_t)item.x * grp.matrix_bytes;
        first = item.y;
    } else {
        first = by * kTok;
        count = min(kTok, M - first);
    }
    // token t's activation row and output row
    auto arow = [&](int t) -> int { return GROUPED ? grp.sorted[first + t] / grp.act_div : first + t; };
    auto orow = [&](int t) -> int { return GROUPED ? grp.sorted[first + t] : first + t; };
    // Stages, two to a stretch.  An odd count gets one more stage: the second
    // half of the last stretch, all of whose blocks lie past the row, with
    // weight scales 0 from the plane's padding.
    const int Hp = ((B + kStage - 1) / kStage + 1) & ~1;

    // This lane's sources, fixed for the product.  Loads past the matrix, the
    // batch or the second tile read in-bounds neighbours; their values are
    // never used (weight scale 0, or not stored).
    // A dense product's are 32-bit offsets from its first token (a register
    // and no address arithmetic a load), a grouped one's whole addresses.
    using Src = std::conditional_t<GROUPED, size_t, uint32_t>;
    const uint8_t *abase = (const uint8_t *)q + (GROUPED ? 0 : (size_t)first * K);
    const uint8_t *sbase = DOTS ? abase : (const uint8_t *)scales + (GROUPED ? 0 : (size_t)first * B * 4);
    Src asrc[Sh::kALoads], ssrc[Sh::kSLoads];
    // load i of the activation: tokens 8 (wv + kWaves i) + lane / 8; of its
    // scales: tokens 16 (wv + kWaves i) + lane / 4, block lane % 4
#pragma unroll
    for (int i = 0; i < Sh::kALoads; i++) {
        const int t = min(8 * (wv + kWaves * i) + (lane >> 3), count - 1);
        asrc[i] = (Src)(GROUPED ? arow(t) : t) * (Src)K;
    }
#pragma unroll
    for (int i = 0; i < Sh::kSLoads; i++) {
        const int t = min(16 * (wv + kWaves * i) + (lane >> 2), count - 1);
        ssrc[i] = (Src)(GROUPED ? arow(t) : t) * (Src)(DOTS ? K : 4 * B);
    }
    const int apiece = 16 * ((lane & 7) ^ ((lane >> 3) & 7)), sblock = lane & 3;

    // load i of this wavefront's kLoads of a stage: nibbles, then activations, then their scales, then the weights'
    auto issue_one = [&](auto slot_tag, auto i_tag, int h) __attribute__((always_inline)) {
        constexpr int i = decltype(i_tag)::value;
        h = min(h, Hp - 1);  // past the last stage: the last stage again, into the free slot
        uint8_t *slot = ring_lds + decltype(slot_tag)::value * kSlotB;
        const int b0 = h * kStage;
        // A uniform address (opaque, so that it stays one) plus a lane's 32-bit
        // offset: the load takes both as they are.
        if constexpr (i < kA0) {  // block idx % 4 of the workgroup's tile idx / 4
            const int idx = wv + kWaves * i, blk = idx & 3, tl = idx >> 2;
            const uint8_t *src = W + ((size_t)min(T0 + tl, tiles - 1) * B + min(b0 + blk, B - 1)) * (kTileRows * kChunk);
            asm("" : "+s"(src));
            src += (uint32_t)(lane * kChunk);
            __builtin_amdgcn_global_load_lds(src, (lds_ptr)(slot + (blk * Sh::kRows + kTileRows * tl) * kChunk), 16, 0, 0);
        } else if constexpr (i < kS0) {
            const uint8_t *src = abase + (Src)(asrc[i - kA0] + (uint32_t)min(b0 * kQ4Block + apiece, K - 16));
            __builtin_amdgcn_global_load_lds(src, (lds_ptr)(slot + Sh::kAct + (wv + kWaves * (i - kA0)) * 1024), 16, 0, 0);
        } else if constexpr (i < kD0) {
            const int idx = wv + kWaves * (i - kS0);
            const uint8_t *src = sbase + (Src)(ssrc[i - kS0] + (uint32_t)(4 * min(b0 + sblock, B - 1)));
            __builtin_amdgcn_global_load_lds(src, (lds_ptr)(slot + (idx < kTok / 16 ? Sh::kActScale + idx * 256 : Sh::kDummy)),
                                             4, 0, 0);
        } else {  // rows 32 idx + lane / 2, blocks 2 (lane % 2) ..
            const int idx = wv + kWaves * (i - kD0), rw = min(32 * idx, Sh::kRows - 32);
            const uint8_t *src = W + plane0_bytes +
                                 (((size_t)min(T0 + (rw >> 6), tiles - 1) * DC + (b0 >> 3)) * kTileRows + (rw & 63)) * kChunk +
                                 8 * ((b0 >> 2) & 1);
            asm("" : "+s"(src));
            src += (uint32_t)((lane >> 1) * kChunk + 4 * (lane & 1));
            __builtin_amdgcn_global_load_lds(
                src, (lds_ptr)(slot + (idx < Sh::kRows / 32 ? Sh::kWScale + idx * 256 : Sh::kDummy)), 4, 0, 0);
        }
    };

    // The loads of a stage spread over its 4 TT steps, kPer a step: those of step `piece`.
    constexpr int kPer = (kLoads + kStage * TT - 1) / (kStage * TT);
    static_assert(kPer * kStage * TT >= kLoads && kPer * TT <= kLoads, "every load has its step");
    auto issue_step = [&](auto slot_tag, auto piece_tag, int h) __attribute__((always_inline)) {
        constexpr int p = decltype(piece_tag)::value * kPer;
        unroll<p, (p + kPer < kLoads ? p + kPer : kLoads)>(
            [&](auto i_tag) __attribute__((always_inline)) { issue_one(slot_tag, i_tag, h); });
    };

    v16f acc[TT], tot[TT];
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++)
            tot[t][e] = 0.0f;
    v16i bias_i;
#pragma unroll
    for (int e = 0; e < 16; e++)
        bias_i[e] = kIntBias;
    const v16f zero_f = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    // This lane's LDS read addresses in slot 0 (the slot and block go in the
    // reads' immediate offsets).  A block's MFMA slot k of lane half g is
    // input 16 g + k: the low nibbles of the row's chunk for g = 0, the high
    // ones for g = 1, against the token's piece 2 j + g of the stage.
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr)ring_lds;
    const uint32_t lds_w = lds_base + (32 * rg + li) * kChunk;
    const uint32_t lds_dw = lds_base + Sh::kWScale + (32 * rg + li) * 8;
    const uint32_t lds_da = lds_base + Sh::kActScale + (32 * TT * tg + li) * 16;
    uint32_t lds_a[kStage];
#pragma unroll
    for (int j = 0; j < kStage; j++)
        lds_a[j] = lds_base + Sh::kAct + (32 * TT * tg + li) * 128 + 16 * ((2 * j + g) ^ (li & 7));
    const int up = g ? 0 : 4;  // brings the lane's nibble of a byte into its high half

    const v4h one = k0_operand(0x3C00u, g == 0), minus = k0_operand(0xB200u, g == 0);  // 1, -0.1875

    // What the next block multiplies, read one block ahead.
    uint32_t dw_n, da_n[TT];
    v4u wq_n, bq_n[TT];
    auto read = [&](auto slot_tag, auto j_tag) __attribute__((always_inline)) {
        constexpr int so = decltype(slot_tag)::value * kSlotB, j = decltype(j_tag)::value;
        lds_read_b128<so + j * Sh::kRows * kChunk>(lds_w, wq_n);
        lds_read_u16<so + 2 * j>(lds_dw, dw_n);
        unroll<0, TT>([&](auto t_tag) __attribute__((always_inline)) {
            constexpr int t = decltype(t_tag)::value;
            lds_read_b128<so + t * 4096>(lds_a[j], bq_n[t]);
            lds_read_b32<so + t * 512 + 4 * j>(lds_da, da_n[t]);
        });
    };

    // The reads land; their registers pass through the wait so that nothing
    // touches them before it.
    auto landed = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(wq_n), "+v"(dw_n));
#pragma unroll
        for (int t = 0; t < TT; t++)
            asm volatile("" : "+v"(bq_n[t]), "+v"(da_n[t]));
    };

    // One stage: four blocks.  kFirst marks a stretch's first stage.  At its
    // fourth block this wavefront holds all it needs of the stage; the next
    // stage has landed, for every wavefront past the barrier, and this
    // stage's slot is free: the loads of stage h + kRing go into it, spread
    // from here to the next stage's third block.
    auto stage = [&](auto slot_tag, auto first_tag, int h) __attribute__((always_inline)) {
        constexpr int kSlot = decltype(slot_tag)::value, kPrev = (kSlot + kRing - 1) % kRing, kNext = (kSlot + 1) % kRing;
        constexpr bool kFirst = decltype(first_tag)::value;
        unroll<0, kStage>([&](auto j_tag) __attribute__((always_inline)) {
            constexpr int j = decltype(j_tag)::value;
            // the previous block's work stays above this block's wait
            __builtin_amdgcn_sched_barrier(0);
            landed();
            if constexpr (j == kStage - 1) {
                wait_vmcnt<(kRing - 2) * kLoads>();
                __builtin_amdgcn_s_barrier();
            }
            const v4h dwop = k04_operand(dw_n);
            v4i A;  // 16 (n - 8) in every byte
#pragma unroll
            for (int i = 0; i < 4; i++)
                A[i] = (int)(((wq_n[i] << up) & 0xF0F0F0F0u) ^ 0x80808080u);
            v4u bq[TT];
            uint32_t dah[TT];
#pragma unroll
            for (int t = 0; t < TT; t++) {
                bq[t] = bq_n[t];
                dah[t] = half2_bits_rtz(__uint_as_float(da_n[t]));
            }
            if constexpr (j + 1 < kStage)
                read(slot_tag, std::integral_constant<int, j + 1>{});
            else
                read(std::integral_constant<int, kNext>{}, std::integral_constant<int, 0>{});
            unroll<0, TT>([&](auto t_tag) __attribute__((always_inline)) {
                constexpr int t = decltype(t_tag)::value;
                // a block past the row has weight scale 0 (the padding is zero):
                // fma(x, 0, acc) == acc
                const v16i D = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, __builtin_bit_cast(v4i, bq[t]), bias_i, 0, 0, 0);
                const v16f S = __builtin_amdgcn_mfma_f32_32x32x8f16(dwop, k04_operand(dah[t]), zero_f, 0, 0, 0);
                const v16f X =
                    __builtin_amdgcn_mfma_f32_32x32x8f16(one, minus, __builtin_bit_cast(v16f, D), 0, 0, 0);  // isum * 2^-22
                constexpr int piece = ((j + 1) % kStage) * TT + t;  // of the stage being loaded
                if constexpr (j == kStage - 1)
                    issue_step(slot_tag, std::integral_constant<int, piece>{}, h + kRing);
                else
                    issue_step(std::integral_constant<int, kPrev>{}, std::integral_constant<int, piece>{}, h - 1 + kRing);
                __builtin_amdgcn_sched_barrier(0);
                // a stretch's first block takes the product for the sum (x *
                // s == fma(x, s, 0) but for the sign of a zero, which the
                // total's 0 + P cannot show); its eighth adds it to the total
#pragma unroll
                for (int e = 0; e < 16; e++)
                    acc[t][e] = kFirst && j == 0 ? X[e] * S[e] : fmaf(X[e], S[e], acc[t][e]);
                if constexpr (!kFirst && j == kStage - 1) {
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        tot[t][e] = tot[t][e] + acc[t][e];
                }
                // the sums are complete here, not sunk past the next barrier
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    if constexpr (!kFirst && j == kStage - 1)
                        asm volatile("" : "+v"(tot[t][e]));
                    else
                        asm volatile("" : "+v"(acc[t][e]));
                }
                if constexpr (DOTS) {
                    const int tt = 32 * (TT * tg + t) + li, b = h * kStage + j;
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int n = T0 * kTileRows + 32 * rg + 8 * (e >> 2) + 4 * g + (e & 3);
                        if (b < B && tt < count && n >= row_start && n < row_end)
                            dots[((size_t)orow(tt) * (row_end - row_start) + (n - row_start)) * B + b] =
                                (int)(X[e] * 4194304.0f);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    };

    // Stages 0 .. kRing - 2 whole, and the pieces of stage kRing - 1 that
    // come before a stage's first block (the rest follow in stage 0).
    unroll<0, kRing - 1>([&](auto n_tag) __attribute__((always_inline)) {
        unroll<0, kLoads>([&](auto i_tag) __attribute__((always_inline)) { issue_one(n_tag, i_tag, decltype(n_tag)::value); });
    });
    unroll<0, TT>([&](auto t_tag) __attribute__((always_inline)) {
        issue_step(std::integral_constant<int, kRing - 1>{}, t_tag, kRing - 1);
    });
    wait_vmcnt<(kRing - 2) * kLoads + kPer * TT>();  // stage 0 has landed
    __builtin_amdgcn_s_barrier();
    read(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
    using F = std::true_type;
    using N = std::false_type;
    if constexpr (kRing == 2) {
        for (int h = 0; h < Hp; h += 2) {
            stage(std::integral_constant<int, 0>{}, F{}, h);
            stage(std::integral_constant<int, 1>{}, N{}, h + 1);
        }
    } else if constexpr (kRing == 3) {
        for (int h = 0;; h += 6) {  // three stretches: the ring comes round to slot 0
            stage(std::integral_constant<int, 0>{}, F{}, h);
            stage(std::integral_constant<int, 1>{}, N{}, h + 1);
            if (h + 2 >= Hp)
                break;
            stage(std::integral_constant<int, 2>{}, F{}, h + 2);
            stage(std::integral_constant<int, 0>{}, N{}, h + 3);
            if (h + 4 >= Hp)
                break;
            stage(std::integral_constant<int, 1>{}, F{}, h + 4);
            stage(std::integral_constant<int, 2>{}, N{}, h + 5);
            if (h + 6 >= Hp)
                break;
        }
    } else {
        static_assert(kRing == 4, "rings of two to four slots");
        for (int h = 0;; h += 4) {  // two stretches: the ring comes round to slot 0
            stage(std::integral_constant<int, 0>{}, F{}, h);
            stage(std::integral_constant<int, 1>{}, N{}, h + 1);
            if (h + 2 >= Hp)
                break;
            stage(std::integral_constant<int, 2>{}, F{}, h + 2);
            stage(std::integral_constant<int, 3>{}, N{}, h + 3);
            if (h + 4 >= Hp)
                break;
        }
    }
    landed();         // the last block's reads ahead: into registers that are free from here
    wait_vmcnt<0>();  // the trailing loads land before the workgroup ends
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++)
            tot[t][e] = tot[t][e] * kUnscale;
    // the lane again, so that no register holds it through the loop
    const int elane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)), eli = elane & 31, eg = elane >> 5;
    if constexpr (EPI == 1) {
        __syncthreads();  // every wavefront is past its last operand reads
        float *xch = (float *)ring_lds;  // [wavefront pair][token tile][lane][17]
        const int pair = wv >> 1;
        if (rg & 1) {
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    xch[((pair * TT + tt) * 64 + 32 * eg + eli) * 17 + e] = tot[tt][e];
        }
        __syncthreads();
        const int tile = T0 + (rg >> 1);
        if (!(rg & 1) && tile * kTileRows < row_end) {
            const int F2 = row_end >> 1;  // outputs a token
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                const int t = 32 * (TT * tg + tt) + eli;
                float v[16];
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const float gt = tot[tt][e], u = xch[((pair * TT + tt) * 64 + 32 * eg + eli) * 17 + e];
                    const float ex = ggml_expf(-gt);
                    const float den = 1.0f + ex;
                    const float sl = gt / den;
                    v[e] = sl * u;
                }
                float peak = fabsf(v[0]);
#pragma unroll
                for (int e = 1; e < 16; e++)
                    peak = fmaxf(peak, fabsf(v[e]));
                peak = fmaxf(peak, __shfl_xor(peak, 32, 64));  // the token's other 16 outputs
                int32_t n[16];
                float stored = 0.0f;
                if (peak == 0.0f) {
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        n[e] = 0;
                } else {
                    const float scale = __fdiv_rn(peak, 127.0f);
                    const float inverse = __fdiv_rn(127.0f, peak);
                    stored = half_bits_to_float(float_to_half_bits(scale));
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int32_t k = nearest_int(v[e] * inverse);
                        n[e] = k > 127 ? 127 : (k < -128 ? -128 : k);
                    }
                }
                int32_t sum = 0;
#pragma unroll
                for (int e = 0; e < 16; e++)
                    sum += n[e];
                sum += __shfl_xor(sum, 32, 64);
                if (t < count) {
                    const int row = orow(t);
                    // element e is output 8 (e / 4) + 4 eg + e % 4 of the tile's 32
#pragma unroll
                    for (int e4 = 0; e4 < 4; e4++) {
                        const uint32_t w = (uint32_t)(n[4 * e4] & 0xFF) | ((uint32_t)(n[4 * e4 + 1] & 0xFF) << 8) |
                                           ((uint32_t)(n[4 * e4 + 2] & 0xFF) << 16) |
                                           ((uint32_t)(n[4 * e4 + 3] & 0xFF) << 24);
                        *(uint32_t *)(mq + (size_t)row * F2 + tile * 32 + 8 * e4 + 4 * eg) = w;
                    }
                    if (eg == 0) {
                        ms[(size_t)row * (F2 >> 5) + tile] = stored;
                        mqs[(size_t)row * (F2 >> 5) + tile] = sum;
                    }
                }
            }
        }
    } else if constexpr (EPI == 2) {
        static_assert(Sh::kWR == 4 && Sh::kWT == 1 && !GROUPED && !DOTS, "the Q|K|V epilogue: 128 rows, 256 threads");
#pragma unroll
        for (int tt = 0; tt < TT; tt++)
            if (32 * tt < count)
                qkv_rope_epilogue(tot[tt], ring_lds, qr, T0, rg, li, g, first + 32 * tt, min(32, count - 32 * tt));
    } else if constexpr (!DOTS) {
        const int nb = T0 * kTileRows + 32 * rg;  // the wavefront's first row
        // four rows a store where the output takes 16-byte stores
        const bool wide = (ldy & 3) == 0 && ((uintptr_t)y & 15) == 0;
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
            const int t = 32 * (TT * tg + tt) + eli;
            if (t >= count)
                continue;
            float *yr = y + (size_t)orow(t) * ldy;
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const int n0 = nb + 8 * e4 + 4 * eg;
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++)
                    v[e] = tot[tt][4 * e4 + e];
                if (n0 >= row_start && n0 + 4 <= row_end) {
                    if (bias) {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            v[e] = v[e] + bias[n0 + e];
                    }
                    if (wide) {
                        *(float4 *)(yr + n0) = make_float4(v[0], v[1], v[2], v[3]);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            yr[n0 + e] = v[e];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int n = n0 + e;
                        if (n >= row_start && n < row_end)
                            yr[n] = bias ? v[e] + bias[n] : v[e];
                    }
                }
            }
        }
    }
}

}  // namespace

namespace {
// Three wavefronts a SIMD each (twelve a CU, in three to six workgroups).  128
// x 64: two token tiles a wavefront share its widened weights; 168 registers
// and a ring of two.  64 x 64 and 128 x 32: one tile a wavefront.
using Shape128x64 = GemmShape<2, 4, 1, 2, 3>;
using Shape64x64 = GemmShape<1, 2, 2, 2, 3>;
using Shape128x32 = GemmShape<1, 4, 1, 3, 3>;

template <typename Sh, bool DD, int EPI>
int launch_shape(gx_ctx *ctx, const gx_weight *w, const uint8_t *mat, const int8_t *q, const float *scales, int M,
                 int row_start, int row_end, const float *bias, float *y, int ldy, int32_t *dots, int8_t *mq,
                 float *ms, int32_t *mqs, const QkvRopeArgs &qr) {
    constexpr int kTiles = Sh::kRows / kTileRows;
    // the widened weights are signed: no recentring term, so no qsum
    const int tile0 = row_start / kTileRows;
    const int tiles = (row_end + kTileRows - 1) / kTileRows - tile0;
    const Groups none{nullptr, nullptr, 1, 0};
    const int cols = (tiles + kTiles - 1) / kTiles;
    const int groups = (M + Sh::kTok - 1) / Sh::kTok;
    // XCD order for matrices of at least eight row groups (every XCD some).
    const int xc = cols >= 8 ? cols : 0;
    const dim3 grid = xc ? dim3((unsigned)(8 * ((cols + 7) / 8) * groups)) : dim3((unsigned)cols, (unsigned)groups);
    q4_0_gemm_kernel<Sh, false, DD, EPI><<<grid, Sh::kThreads, 0, ctx->stream>>>(
        mat, w->plane0_bytes, w->blocks, w->dchunks, q, scales, w->cols, M, w->tiles, tile0, row_start, row_end, bias,
        y, ldy, dots, none, xc, mq, ms, mqs, qr);
    return check_launch("q4_0_gemm");
}

// The shape of a dense product.  Its time goes by the most workgroups any CU
// takes (in turn or three at once: the matrix core's time a workgroup is the
// same), so by whole rounds of the CUs: a few tokens or rows more that start a
// round cost all of it, and which shape needs the fewer, smaller rounds changes
// from size to size.  A shape's time is taken as a + b rounds, in tenths of a
// us at 2560 inputs, fitted to 18 matrices of 512 to 32000 rows and 512 to
// 9728 inputs at 35 token counts from 24 to 2,048: no size takes 3 % more than
// under the rules before (a count of the workgroups alone) and all 0.7 % more
// than the fastest shape on average (1.7 % before).  128 x 64 in less than
// three rounds only with the SwiGLU epilogue: the product's own outputs are
// four to eight times as many bytes, and three whole tiles a CU then end
// together.  us 128 x 64 / 64 x 64 / 128 x 32: 19456 x 2560 with SwiGLU at 65
// tokens 31.2 / 26.3 / 20.5, at 129 34.8 / 35.0 / 29.7, at 257 49.2 / 52.3 /
// 54.0; 10240 x 2560 with SwiGLU at 560 48.7 / 51.7 / 53.3, at 584 62.6 / 57.8 /
// 54.3; 9728 x 2560 at 584 56.0 / 48.9 / 50.0, at 2048 126 / 137; 2560 x 4096 at
// 1500 55.8 / 46.6.  Up to 32 tokens half of a 64-token tile would be empty:
// 128 x 32 (19456 x 2560 with SwiGLU at 32: 15.0 against 17.9).  The Q|K|V
// epilogue's heads need 128 rows.
struct ShapeCost {
    int rows, tokens, a, b;
    size_t workgroups(int tiles, int M) const {
        const int per = rows / kTileRows;
        return (size_t)((tiles + per - 1) / per) * (size_t)((M + tokens - 1) / tokens);
    }
    size_t operator()(gx_ctx *ctx, int tiles, int M) const {
        return a + b * ((workgroups(tiles, M) + ctx->cu_count - 1) / ctx->cu_count);
    }
};
constexpr ShapeCost kCost128x64{128, 64, 90, 120}, kCost64x64{64, 64, 30, 74}, kCost128x32{128, 32, 60, 78};

template <int EPI>
int launch_dense(gx_ctx *ctx, const gx_weight *w, const uint8_t *mat, const int8_t *q, const float *scales, int M,
                 int row_start, int row_end, const float *bias, float *y, int ldy, int32_t *dots, int8_t *mq,
                 float *ms, int32_t *mqs, const QkvRopeArgs &qr) {
    const int tiles = (row_end + kTileRows - 1) / kTileRows - row_start / kTileRows;
#define GX_SHAPE(SH)                                                                                                 \
    do {                                                                                                             \
        if (EPI == 0 && dots)                                                                                        \
            return launch_shape<SH, EPI == 0, EPI>(ctx, w, mat, q, scales, M, row_start, row_end, bias, y, ldy,     \
                                                   dots, mq, ms, mqs, qr);                                          \
        return launch_shape<SH, false, EPI>(ctx, w, mat, q, scales, M, row_start, row_end, bias, y, ldy, nullptr,   \
                                            mq, ms, mqs, qr);                                                       \
    } while (0)
    const size_t wide = kCost128x64(ctx, tiles, M), narrow = kCost128x32(ctx, tiles, M);
    const bool whole = EPI == 1 || kCost128x64.workgroups(tiles, M) >= 3 * (size_t)ctx->cu_count;
    if constexpr (EPI != 2) {
        if (M > 32 && kCost64x64(ctx, tiles, M) < (whole ? std::min(wide, narrow) : narrow))
            GX_SHAPE(Shape64x64);
    }
    if (whole && wide < narrow)
        GX_SHAPE(Shape128x64);
    GX_SHAPE(Shape128x32);
#undef GX_SHAPE
}
}  // namespace

int launch_q4_0_gemm(gx_ctx *ctx, const gx_weight *w, const uint8_t *mat, const int8_t *q, const float *scales,
                     int M, int row_start, int row_end, const float *bias, float *y, int ldy, int32_t *dots) {
    return launch_dense<0>(ctx, w, mat, q, scales, M, row_start, row_end, bias, y, ldy, dots, nullptr, nullptr,
                           nullptr, QkvRopeArgs{});
}

int launch_q4_0_gemm_swiglu(gx_ctx *ctx, const gx_weight *w, const int8_t *q, const float *scales, int M,
                            int8_t *mq, float *ms, int32_t *mqs) {
    return launch_dense<1>(ctx, w, w->dev, q, scales, M, 0, w->rows, nullptr, nullptr, 0, nullptr, mq, ms, mqs,
                           QkvRopeArgs{});
}

int launch_q4_0_gemm_qkv_rope(gx_ctx *ctx, const gx_weight *w, const int8_t *q, const float *scales, int M,
                              const QkvRopeArgs &a) {
    return launch_dense<2>(ctx, w, w->dev, q, scales, M, 0, w->rows, nullptr, nullptr, 0, nullptr, nullptr, nullptr,
                           nullptr, a);
}

int launch_q4_0_gemm_grouped(gx_ctx *ctx, const gx_weight *w, const int32_t *work, int max_items,
                             const int32_t *sorted, int act_div, const int8_t *q, const float *scales, float *y,
                             int ldy, int32_t *dots) {
    // Items of at most kGroupTok units (the sort's tile), 32 tokens a workgroup.
    const dim3 grid((unsigned)((w->tiles + 1) / 2), (unsigned)max_items);
    const Groups grp{work, sorted, act_div, w->matrix_bytes};
    if (dots)
        q4_0_gemm_kernel<Shape128x32, true, true, 0><<<grid, Shape128x32::kThreads, 0, ctx->stream>>>(
            w->dev, w->plane0_bytes, w->blocks, w->dchunks, q, scales, w->cols, 0, w->tiles, 0, 0, w->rows, nullptr,
            y, ldy, dots, grp, 0, nullptr, nullptr, nullptr, QkvRopeArgs{});
    else
        q4_0_gemm_kernel<Shape128x32, true, false, 0><<<grid, Shape128x32::kThreads, 0, ctx->stream>>>(
            w->dev, w->plane0_bytes, w->blocks, w->dchunks, q, scales, w->cols, 0, w->tiles, 0, 0, w->rows, nullptr,
            y, ldy, nullptr, grp, 0, nullptr, nullptr, nullptr, QkvRopeArgs{});
    return check_launch("q4_0_gemm_grouped");
}
}  // namespace gx

namespace gx {

int launch_q4_0_gemm_f16(gx_ctx *ctx, const gx_weight *w, const uint8_t *mat, const uint16_t *q16,
                         const float *scales, int M, int row_start, int row_end, const float *bias, float *y, int ldy,
                         int32_t *dots) {
    const int tile0 = row_start / kTileRows;
    const unsigned tiles = (unsigned)((row_end + kTileRows - 1) / kTileRows - tile0);
    const int groups = (M + 31) / 32;
    // Token groups per workgroup: wider workgroups share the widening of the
    // weights among more tokens; narrower ones keep more workgroups in flight.
    const int nwt = groups <= 32 ? 2 : 4;
    const dim3 grid(tiles, (unsigned)((groups + nwt - 1) / nwt));
#define GX_F16_LAUNCH(N)                                                                                             \
    do {                                                                                                             \
        if (dots)                                                                                                    \
            q4_0_gemm_f16_kernel<N, true><<<grid, 64 * N, 0, ctx->stream>>>(                                         \
                mat, w->plane0_bytes, w->blocks, w->dchunks, q16, scales, M, tile0, row_start, row_end, bias, y, ldy, \
                dots);                                                                                               \
        else                                                                                                         \
            q4_0_gemm_f16_kernel<N, false><<<grid, 64 * N, 0, ctx->stream>>>(                                        \
                mat, w->plane0_bytes, w->blocks, w->dchunks, q16, scales, M, tile0, row_start, row_end, bias, y, ldy, \
                dots);                                                                                               \
    } while (0)
    if (nwt == 2)
        GX_F16_LAUNCH(2);
    else
        GX_F16_LAUNCH(4);
#undef GX_F16_LAUNCH
    return check_launch("q4_0_gemm_f16");
}

}  // namespace gx
