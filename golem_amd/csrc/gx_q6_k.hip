// gx_q6_k.hip - the Q6_K x Q8_K matrix-vector product (the logit head).
//
// golem's matVecQ6_KRows / dotQ6_KGo (nn/dot_q6_k.go:19-54, :77-103), bit for
// bit: per superblock the exact integer sum - 32*shift, then
//   t_b   = (float(isum_b) * d_b) * kscale_b       two fp32 products
//   total = ((0 + t_0) + t_1) + ...                 in superblock order
// (-ffp-contract=off keeps the products and sums unfused, as Go's amd64
// compiler leaves them).  Up to eight activation columns share one read of
// the weights, the role of dotQ6_Kx2 (nn/dot_q6_k_x2_amd64.s:64-154), and
// give each column exactly its one-column result.
//
// One column (and inputs the second kernel does not take) runs on the vector
// ALU, two to sixteen at a time on the matrix cores (below).
// Decomposition as the Q4_0 kernel: a workgroup owns one 64-row tile, each
// wavefront whole superblocks, a lane one row.  The activation of a
// superblock is uniform across the wavefront and is read into SGPRs with
// scalar loads; the superblock terms meet in LDS and one wavefront adds them
// in order.
#include "gx_device.hpp"
#include "gx_internal.hpp"

namespace gx {
namespace {

template <int NC>
__global__ __launch_bounds__(1024) void q6_k_matvec_kernel(
    const uint8_t *__restrict__ W, size_t plane0_bytes, int B, int DC, const int8_t *__restrict__ q,
    const float *__restrict__ kscales, const int16_t *__restrict__ bsums, int K, int tile0, int row_start,
    int row_end, const float *__restrict__ bias, float *__restrict__ y, int ldy, int32_t *__restrict__ dots) {
    extern __shared__ float part[];  // [B][NC][64]
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nwaves = blockDim.x >> 6;
    const int tile = tile0 + blockIdx.x;
    const int row = tile * kTileRows + lane;
    const uint8_t *d_row = W + plane0_bytes + ((size_t)tile * DC * kTileRows + lane) * kChunk;

    for (int s = wave; s < B; s += nwaves) {
        const uint8_t *base = W + (((size_t)tile * B + s) * kQ6Chunks * kTileRows + lane) * kChunk;
        uint32_t ql[32], qh[16];
#pragma unroll
        for (int c = 0; c < 8; c++) {
            const uint4 v = load_stream(base + (size_t)c * kTileRows * kChunk);
            ql[4 * c] = v.x, ql[4 * c + 1] = v.y, ql[4 * c + 2] = v.z, ql[4 * c + 3] = v.w;
        }
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint4 v = load_stream(base + (size_t)(8 + c) * kTileRows * kChunk);
            qh[4 * c] = v.x, qh[4 * c + 1] = v.y, qh[4 * c + 2] = v.z, qh[4 * c + 3] = v.w;
        }
        const uint4 sc = load_stream(base + (size_t)12 * kTileRows * kChunk);
        const float d = half_bits_to_float(*(const uint16_t *)(d_row + (size_t)(s >> 3) * kTileRows * kChunk +
                                                              (size_t)(s & 7) * 2));
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const uint32_t *a = (const uint32_t *)(q + (size_t)c * K + (size_t)s * kSuper);
            const uint32_t *bs = (const uint32_t *)(bsums + (size_t)c * (K / 16) + (size_t)s * 16);
            const int32_t isum = q6_k_block_isum(ql, qh, sc, a, bs);
            if (dots) {
                if (row >= row_start && row < row_end)
                    dots[((size_t)c * (row_end - row_start) + (row - row_start)) * B + s] = isum;
            } else {
                const float t0 = (float)isum * d;
                part[(s * NC + c) * kTileRows + lane] = t0 * kscales[(size_t)c * B + s];
            }
        }
    }
    if (dots)
        return;
    __syncthreads();
    if (wave == 0 && row >= row_start && row < row_end) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            float total = 0.0f;
            for (int s = 0; s < B; s++)
                total = total + part[(s * NC + c) * kTileRows + lane];
            if (bias)
                total = total + bias[row];
            y[(size_t)c * ldy + row] = total;
        }
    }
}

constexpr size_t kMatvecLds = 64 * 1024;

template <int NC>
int launch_nc(gx_ctx *ctx, const gx_weight *w, const int8_t *q, const float *kscales, const int16_t *bsums,
              int row_start, int row_end, const float *bias, float *y, int ldy, int32_t *dots) {
    const int B = w->blocks;
    const int waves = min(B, 16);
    const size_t lds = dots ? 0 : (size_t)B * NC * kTileRows * sizeof(float);
    GX_CHECK(lds <= kMatvecLds, "gx: a %d-input Q6_K row is wider than this kernel's LDS", w->cols);
    const int tile0 = row_start / kTileRows;
    const int grid = (row_end + kTileRows - 1) / kTileRows - tile0;
    q6_k_matvec_kernel<NC><<<grid, 64 * waves, lds, ctx->stream>>>(w->dev, w->plane0_bytes, B, w->dchunks, q,
                                                                   kscales, bsums, w->cols, tile0, row_start,
                                                                   row_end, bias, y, ldy, dots);
    return check_launch("q6_k_matvec");
}

// ---- 2 to 16 columns on the matrix cores ------------------------------------
//
// v_mfma_i32_16x16x64_i8 takes 64 inputs of 16 rows against 16 columns, a
// lane the 16 inputs of one of the row's four scale groups: the group's scale
// is that lane's own, so it goes into the weights, (q - 32) * scale, at most
// 32 * 128 in magnitude, as 256 * h + l with h in [-16, 16] and l in [-128,
// 127], two int8 operands.  A superblock's integer sum - 32*shift is then 256
// * (the h products) + (the l products), exactly, for every column at once;
// the rest is the one-column kernel's arithmetic in its order: (float(isum) *
// d) * kscale, added superblock by superblock, in the lane that holds the
// output.
//
// A workgroup owns 128 rows (two R64 tiles), a wavefront 16 of them and all
// their superblocks, the next one's loads in flight under this one's
// arithmetic.  A lane loads its row's chunk of its own group, so a load's 64
// lanes cover four 256-byte runs.  The columns' inputs sit in LDS, rows K +
// 16 bytes apart (no bank conflicts), with their scales and the rows' d.
//
// What bounds it: HBM (the bytes take 47 us at 151936 x 2560), beside the
// widening (240 vector instructions per 16 rows and superblock).  2 / 4 / 6 /
// 8 / 16 columns there: 60 / 61 / 61 / 62 / 67 us, where the vector kernel
// above, its columns in turn, takes 61 / 72 / 132 / 115 / 225 (102 registers,
// so one workgroup a CU, and scalar loads of the activation a column).  Four
// wavefronts a workgroup: 60 / 62 / 79 us at 2 / 6 / 16; sixteen 67 / 69 / 75;
// two superblocks ahead 63 / 65 / 71.
constexpr int kColsWaves = 8, kColsRows = 16 * kColsWaves, kColsMax = 16;

typedef short v2s __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));

// Four 6-bit weights q (one a byte) times the scale, (q - 32) * scale = 256 h +
// l: m = q * scale + (128 - 32 * scale) is 256 h + l + 128, so h is m's high
// byte and l its low one with the top bit flipped.
__device__ __forceinline__ void q6_scaled(uint32_t q, uint32_t sc2, uint32_t add2, int &h, int &l) {
    const uint32_t e = __builtin_amdgcn_perm(0u, q, 0x0c020c00u), o = __builtin_amdgcn_perm(0u, q, 0x0c030c01u);
    uint32_t me, mo;
    asm("v_pk_mad_i16 %0, %1, %2, %3" : "=v"(me) : "v"(e), "v"(sc2), "v"(add2));
    asm("v_pk_mad_i16 %0, %1, %2, %3" : "=v"(mo) : "v"(o), "v"(sc2), "v"(add2));
    h = (int)__builtin_amdgcn_perm(mo, me, 0x07030501u);
    l = (int)(__builtin_amdgcn_perm(mo, me, 0x06020400u) ^ 0x80808080u);
}

// The workgroup's LDS: the inputs [M][K + 16], the column scales [M][B] and
// the rows' d [DC * 8][128], each part from a multiple of 16 bytes (d is read
// eight bytes at a time, whatever M and B).
__host__ __device__ constexpr size_t q6_cols_scales(int M, int K) { return (size_t)M * (K + 16); }
__host__ __device__ constexpr size_t q6_cols_d(int M, int K, int B) {
    return q6_cols_scales(M, K) + ((size_t)M * B * 4 + 15) / 16 * 16;
}
__host__ __device__ constexpr size_t q6_cols_lds(int M, int K, int B, int DC) {
    return q6_cols_d(M, K, B) + (size_t)DC * 8 * kColsRows * 2;
}
constexpr bool q6_cols_aligned() {
    for (int M = 1; M <= kColsMax; M++)
        for (int B = 1; B <= 64; B++)
            if (q6_cols_scales(M, 256 * B) % 16 != 0 || q6_cols_d(M, 256 * B, B) % 16 != 0)
                return false;
    return true;
}
static_assert(q6_cols_aligned(), "every part of the LDS can be read at its access width");

template <bool DOTS>
__global__ __launch_bounds__(64 * kColsWaves, 4) void q6_k_mfma_cols_kernel(
    const uint8_t *__restrict__ W, size_t plane0_bytes, int B, int DC, const int8_t *__restrict__ q,
    const float *__restrict__ kscales, int K, int M, int tiles, int tile0, int row_start, int row_end,
    const float *__restrict__ bias, float *__restrict__ y, int ldy, int32_t *__restrict__ dots) {
    extern __shared__ __align__(16) uint8_t lds[];  // inputs [M][K + 16], kscales [M][B], d [DC * 8][128]
    float *ks = (float *)(lds + q6_cols_scales(M, K));
    uint16_t *dl = (uint16_t *)(lds + q6_cols_d(M, K, B));
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 15, g = lane >> 4;
    const int T0 = tile0 + kColsRows / kTileRows * blockIdx.x, tile = min(T0 + (wave >> 2), tiles - 1);
    const uint8_t *base = W + (size_t)tile * B * kQ6Chunks * kTileRows * kChunk;
    const uint32_t row_off = (uint32_t)(16 * (wave & 3) + li) * kChunk;
    uint32_t o_ql[2], o_qh[2];
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
        o_ql[hh] = (uint32_t)(4 * hh + g) * kTileRows * kChunk + row_off;
        o_qh[hh] = (uint32_t)(8 + 2 * hh + (g & 1)) * kTileRows * kChunk + row_off;
    }
    const uint32_t o_sc = 12u * kTileRows * kChunk + row_off;
    struct Super {
        uint4 ql[2], qh[2], sc;
    };
    auto load = [&](Super &w, int s) __attribute__((always_inline)) {
        const uint8_t *p = base + (size_t)s * kQ6Chunks * kTileRows * kChunk;
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            w.ql[hh] = load_stream(p + o_ql[hh]);
            w.qh[hh] = load_stream(p + o_qh[hh]);
        }
        w.sc = load_stream(p + o_sc);
    };
    Super wa, wb;
    load(wa, 0);

    // the columns and scales into LDS
    const int pieces = M * (K / 16);
    for (int i = tid; i < pieces; i += 64 * kColsWaves) {
        const int c = i / (K / 16), p = i - c * (K / 16);
        *(v4u_stream *)(lds + (size_t)c * (K + 16) + 16 * p) = *(const v4u_stream *)(q + (size_t)c * K + 16 * p);
    }
    for (int i = tid; i < M * B; i += 64 * kColsWaves)
        ks[i] = DOTS ? 0.0f : kscales[i];
    for (int i = tid; i < kColsRows * DC; i += 64 * kColsWaves) {
        const int r = i & (kColsRows - 1), c = i / kColsRows;
        const v4u_stream v = *(const v4u_stream *)(W + plane0_bytes +
                                                   (((size_t)min(T0 + (r >> 6), tiles - 1) * DC + c) * kTileRows + (r & 63)) *
                                                       kChunk);
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 8; j++)
            dl[(8 * c + j) * kColsRows + r] = (uint16_t)(w[j >> 1] >> (16 * (j & 1)));
    }
    __syncthreads();

    const int col = min(li, M - 1);  // a lane past the columns repeats the last: never stored
    const uint8_t *act = lds + (size_t)col * (K + 16) + 16 * g;
    const uint32_t sl = g < 2 ? 4 : 2, sh = g < 2 ? 0 : 2;
    float total[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int row0 = T0 * kTileRows + 16 * wave + 4 * g;  // this lane's four outputs
    auto step = [&](const Super &w, int s) __attribute__((always_inline)) {
        const uint32_t scw[4] = {w.sc.x, w.sc.y, w.sc.z, w.sc.w};
        v4i Dh = {0, 0, 0, 0}, Dl = {0, 0, 0, 0};
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            const uint32_t L[4] = {w.ql[hh].x, w.ql[hh].y, w.ql[hh].z, w.ql[hh].w};
            const uint32_t H[4] = {w.qh[hh].x, w.qh[hh].y, w.qh[hh].z, w.qh[hh].w};
#pragma unroll
            for (int hi = 0; hi < 2; hi++) {  // groups 8 hh + 4 hi + g: the low nibbles, then the high ones
                const v4i bv = *(const v4i *)(act + (size_t)s * kSuper + 128 * hh + 64 * hi);
                const int sc = (int)(scw[2 * hh + hi] << (24 - 8 * g)) >> 24;
                const uint32_t sc2 = __builtin_amdgcn_perm(0u, (uint32_t)sc, 0x01000100u);
                const v2s a2 = {(short)(128 - 32 * sc), (short)(128 - 32 * sc)};
                const uint32_t add2 = __builtin_bit_cast(uint32_t, a2);
                v4i h, l;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t q6 = hi ? ((L[k] >> 4) & 0x0F0F0F0Fu) | ((H[k] >> sh) & 0x30303030u)
                                           : (L[k] & 0x0F0F0F0Fu) | ((H[k] << sl) & 0x30303030u);
                    int hk, lk;
                    q6_scaled(q6, sc2, add2, hk, lk);
                    h[k] = hk;
                    l[k] = lk;
                }
                Dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(h, bv, Dh, 0, 0, 0);
                Dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(l, bv, Dl, 0, 0, 0);
            }
        }
        const uint2 dw = *(const uint2 *)(dl + s * kColsRows + 16 * wave + 4 * g);
        const float kc = ks[col * B + s];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int32_t isum = (Dh[i] << 8) + Dl[i];
            if constexpr (DOTS) {
                const int r = row0 + i;
                if (li < M && r >= row_start && r < row_end)
                    dots[((size_t)li * (row_end - row_start) + (r - row_start)) * B + s] = isum;
            } else {
                const uint32_t dh = (i < 2 ? dw.x : dw.y) >> (16 * (i & 1));
                const float t0 = (float)isum * half_bits_to_float(dh & 0xFFFFu);
                const float t = t0 * kc;
                total[i] = total[i] + t;
            }
        }
    };
    for (int s = 0; s < B; s += 2) {
        load(wb, min(s + 1, B - 1));
        step(wa, s);
        if (s + 1 < B) {
            load(wa, min(s + 2, B - 1));
            step(wb, s + 1);
        }
    }
    if (DOTS || li >= M)
        return;
    float *yr = y + (size_t)li * ldy;
    if (bias) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            total[i] = total[i] + bias[min(row0 + i, row_end - 1)];
    }
    if (row0 >= row_start && row0 + 4 <= row_end && (ldy & 3) == 0 && ((uintptr_t)y & 15) == 0) {
        *(float4 *)(yr + row0) = make_float4(total[0], total[1], total[2], total[3]);
    } else {
#pragma unroll
        for (int i = 0; i < 4; i++)
            if (row0 + i >= row_start && row0 + i < row_end)
                yr[row0 + i] = total[i];
    }
}

int launch_cols(gx_ctx *ctx, const gx_weight *w, const int8_t *q, const float *kscales, int M, int row_start,
                int row_end, const float *bias, float *y, int ldy, int32_t *dots) {
    const int tile0 = row_start / kTileRows;
    const int grid = (row_end - tile0 * kTileRows + kColsRows - 1) / kColsRows;
    const size_t lds = q6_cols_lds(M, w->cols, w->blocks, w->dchunks);
#define GX_Q6_COLS(DD)                                                                                               \
    q6_k_mfma_cols_kernel<DD><<<grid, 64 * kColsWaves, lds, ctx->stream>>>(                                          \
        w->dev, w->plane0_bytes, w->blocks, w->dchunks, q, kscales, w->cols, M, w->tiles, tile0, row_start, row_end,  \
        bias, y, ldy, dots)
    if (dots)
        GX_Q6_COLS(true);
    else
        GX_Q6_COLS(false);
#undef GX_Q6_COLS
    return check_launch("q6_k_mfma_cols");
}

// How many of `left` columns the matrix cores take in one launch, 0 for none:
// as many as leave the LDS to two workgroups a CU (sixteen of up to 4,608
// inputs, fourteen of 5,120), where the inputs can be read 16 bytes at a time.
// A workgroup's superblocks are a serial chain (2.5 us and 1.15 more each,
// however few the rows), where the vector kernel spreads them over its
// wavefronts but reads the weights again for its next power of two of
// columns.  So nine columns and more always go here; of the others those the
// vector kernel takes in several reads (7 in three; 3, 5 and 6 in two) where a
// row has few superblocks or the workgroups reach a small part of the CUs (7),
// half of them (5, 6) or three quarters (3); and those it takes in one read
// (2, 4, 8) from the counts at which its registers cost it more than the
// chain.  us vector / matrix cores over weights not in the caches, rows x
// inputs: two columns 4096 x 2560 6.6 / 14.7, 98304 x 2560 38.5 / 38.6, 151936
// x 2560 59.7 / 58.2; three 8192 x 2560 12.7 / 15.0, 24576 x 2560 24.5 / 17.5,
// 256 x 1024 7.3 / 7.1; four 16384 x 2560 10.8 / 16.0, 65536 x 2816 33.6 /
// 29.1, 151936 x 1024 23.2 / 27.3; five 16384 x 2560 17.8 / 15.6; six 4096 x
// 4096 17.3 / 21.9, 16384 x 4096 23.3 / 22.4; seven 512 x 5120 23.7 / 26.0,
// 1024 x 4096 22.4 / 21.7; eight 16384 x 4096 17.9 / 22.7, 24576 x 4096 31.1 /
// 23.3, 4096 x 1024 9.9 / 7.8.
int cols_on_mfma(gx_ctx *ctx, const gx_weight *w, int left, bool aligned, int row_start, int row_end) {
    const int cus = ctx->cu_count, few_supers = 4;
    const int groups = (row_end - row_start / kTileRows * kTileRows + kColsRows - 1) / kColsRows;
    int n = min(left, kColsMax);
    while (n > 1 && q6_cols_lds(n, w->cols, w->blocks, w->dchunks) > 80 * 1024)
        n--;
    if (n < 2 || !aligned)
        return 0;
    const bool few = w->blocks <= few_supers;
    const bool pays = n >= 9             ? true
                    : n == 7             ? w->blocks <= 3 * few_supers || groups >= cus / 32
                    : n == 2             ? !few && groups >= 4 * cus
                    : n == 4             ? !few && groups >= 2 * cus
                    : n == 3 || n == 8   ? few || groups >= 3 * cus / 4
                                         : few || groups >= cus / 2;
    return pays ? n : 0;
}

}  // namespace

int launch_q6_k_matvec(gx_ctx *ctx, const gx_weight *w, const int8_t *q, const float *kscales,
                       const int16_t *bsums, int M, int row_start, int row_end, const float *bias, float *y,
                       int ldy, int32_t *dots) {
    const int K = w->cols, B = w->blocks;
    const size_t nrows = (size_t)(row_end - row_start);
    // the vector kernel's LDS holds nc columns' terms (it stores integers directly)
    auto fits = [&](int nc) { return dots || (size_t)B * nc * kTileRows * sizeof(float) <= kMatvecLds; };
    int c = 0;
    while (c < M) {
        const int left = M - c;
        const int8_t *qc = q + (size_t)c * K;
        const float *kc = kscales ? kscales + (size_t)c * B : nullptr;
        const int16_t *bc = bsums + (size_t)c * (K / 16);
        float *yc = y ? y + (size_t)c * ldy : nullptr;
        int32_t *dc = dots ? dots + (size_t)c * nrows * B : nullptr;
        int rc;
        const int n = cols_on_mfma(ctx, w, left, (uintptr_t)q % 16 == 0, row_start, row_end);
        if (n) {
            rc = launch_cols(ctx, w, qc, kc, n, row_start, row_end, bias, yc, ldy, dc);
            c += n;
        } else if (left >= 8 && fits(8)) {
            rc = launch_nc<8>(ctx, w, qc, kc, bc, row_start, row_end, bias, yc, ldy, dc);
            c += 8;
        } else if (left >= 4 && fits(4)) {
            rc = launch_nc<4>(ctx, w, qc, kc, bc, row_start, row_end, bias, yc, ldy, dc);
            c += 4;
        } else if (left >= 2 && fits(2)) {
            rc = launch_nc<2>(ctx, w, qc, kc, bc, row_start, row_end, bias, yc, ldy, dc);
            c += 2;
        } else {
            rc = launch_nc<1>(ctx, w, qc, kc, bc, row_start, row_end, bias, yc, ldy, dc);
            c += 1;
        }
        if (rc)
            return rc;
    }
    return GX_OK;
}

}  // namespace gx
