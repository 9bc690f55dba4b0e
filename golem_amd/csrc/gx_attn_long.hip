// gx_attn_long.hip - the parallel-order attention past the prefixes that one
// workgroup holds (gx_qwen.hip): a decode step's positions spread over the
// chip, or a workgroup a token and a few of its heads; and a prompt's attention
// on the matrix cores with nothing but the block sums kept between its sweeps.
//
// All compute what the short forms compute (qwen/attention.go:96-124,
// nn/ops.go:59-73): the scores, their maximum, the float64 exponential of the
// float difference rounded to float (exp_neg), the total as 64-position blocks
// summed pairwise and the blocks added in order, the probabilities divided
// and rounded through fp16, the value sums.
#include <algorithm>
#include <type_traits>

#include "gx_device.hpp"
#include "gx_internal.hpp"

namespace gx {
namespace {

// lo/hi(a) * lo/hi(b) + c for fp16 pairs a and b, as one v_fma_mix.
__device__ __forceinline__ float fma_mix_lo(uint32_t a, uint32_t b, float c) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ float fma_mix_hi(uint32_t a, uint32_t b, float c) {
    float r;
    asm("v_fma_mix_f32 %0, %1, %2, %3 op_sel:[1,1,0] op_sel_hi:[1,1,0]" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

constexpr int kOne = 1024;          // positions a prompt's LDS form takes (gx_qwen.hip)
constexpr int kSplitTokens = 16;    // tokens the split form takes
constexpr int kSplitWaves = 16384;  // wavefronts a launch of it (split_share)
constexpr int kBlock = 64;  // positions a block of the softmax total
constexpr int kRun = 32;    // positions a run of the value sums

// ---- one position at a time (M <= 4, or one per conversation) ---------------
//
// Four launches, each spread over the prefix: the scores (a wavefront a head
// and 64 positions) with each block's maximum; the exponentials with each
// block's sum; the probabilities and the runs' value chains; the runs in order
// with the Q8_0.  The order of every sum is attn_par_kernel's, whatever the
// extent.  The grids' slowest dimension is the prefix, so that the workgroups
// with positions come first and on different CUs: with the tokens slowest, the
// empty ones between put every token's first block on the same few (sixteen
// conversations at position 20, launched for 1,024: 24.7 us, now 15.0).
// What bounds it: the launches (about 2 us each) and their load latencies;
// then the bytes and two serial sums that every workgroup or lane repeats, a
// prefix's blocks and its runs.  One position of 32 heads of 128 at 20 / 1,000
// / 3,000 / 16,000 / 32,000: 14 / 15 / 20 / 43 / 80 us, where the serial
// passes take 14 / 40 / 102 / 485 / 937.

// grid (kv_heads, tokens, blocks' share), 64 threads a query head of the group:
// blocks blockIdx.z, blockIdx.z + share, ..
template <int HD>
__global__ __launch_bounds__(512) void attn_split_scores_kernel(
    const uint16_t *__restrict__ qh, int heads, int kv_heads, const int32_t *__restrict__ positions, int limit,
    const uint16_t *__restrict__ kcache, int context, float scale, int S, float *__restrict__ sc,
    float *__restrict__ mx, const int32_t *__restrict__ slots, int nslots, int share) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kvh = blockIdx.x, t = blockIdx.y;
    const int h = kvh * (heads / kv_heads) + wave;
    const int n = min(positions[t] + 1, limit);
    if (slots)
        kcache += (size_t)min(max(slots[t], 0), nslots - 1) * kv_heads * HD * context;
    // the query is one address for the wavefront
    const v4u_stream *qv = (const v4u_stream *)(qh + ((size_t)t * heads + h) * HD);
    const size_t row = (size_t)t * heads + h;
    for (int b = blockIdx.z; b * kBlock < n; b += share) {
        const int p = b * kBlock + lane;
        const v4u_stream *kr = (const v4u_stream *)(kcache + (size_t)kvh * HD * context) + min(p, n - 1);
        v4u_stream k[HD / 8];
#pragma unroll
        for (int i = 0; i < HD / 8; i++)
            k[i] = kr[(size_t)i * context];
        float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
#pragma unroll
        for (int i = 0; i < HD / 8; i++) {
            const v4u_stream qq = qv[i], kk = k[i];
            s0 = fma_mix_lo(qq.x, kk.x, s0);
            s1 = fma_mix_hi(qq.x, kk.x, s1);
            s2 = fma_mix_lo(qq.y, kk.y, s2);
            s3 = fma_mix_hi(qq.y, kk.y, s3);
            s0 = fma_mix_lo(qq.z, kk.z, s0);
            s1 = fma_mix_hi(qq.z, kk.z, s1);
            s2 = fma_mix_lo(qq.w, kk.w, s2);
            s3 = fma_mix_hi(qq.w, kk.w, s3);
        }
        const float v = scale * ((s0 + s1) + (s2 + s3));
        if (p < n)
            sc[row * S + p] = v;
        const float m = wave_max(p < n ? v : -INFINITY);
        if (lane == 0)
            mx[row * (S / kBlock) + b] = m;
    }
}

// grid (heads, tokens, blocks' share), four wavefronts, each with every fourth
// of the workgroup's blocks: exponentials in place.
__global__ __launch_bounds__(256) void attn_split_exp_kernel(int heads, int kv_heads,
                                                             const int32_t *__restrict__ positions, int limit, int S,
                                                             float *__restrict__ sc, const float *__restrict__ mx,
                                                             float *__restrict__ bs, int share) {
    const int lane = threadIdx.x & 63, b0 = blockIdx.z * 4 + (threadIdx.x >> 6);
    const int t = blockIdx.y;
    const int n = min(positions[t] + 1, limit), nb = n > 0 ? (n + kBlock - 1) / kBlock : 0;
    if (b0 >= nb)
        return;
    // key-value heads fastest: on the XCD that wrote the scores, where there are eight
    const int h = (int)blockIdx.x % kv_heads * (heads / kv_heads) + (int)blockIdx.x / kv_heads;
    const size_t row = (size_t)t * heads + h;
    float *s = sc + row * S;
    float v = s[min(b0 * kBlock + lane, n - 1)];
    const float *mr = mx + row * (S / kBlock);
    float m = -INFINITY;
    for (int i = lane; i < nb; i += 64)
        m = fmaxf(m, mr[i]);
    m = wave_max(m);
    for (int b = b0;;) {
        const int p = b * kBlock + lane;
        const float e = p < n ? exp_neg(v - m) : 0.0f;
        s[p] = e;  // S is a whole number of blocks
        const float sum = wave_pairwise_sum(e);
        if (lane == 0)
            bs[row * (S / kBlock) + b] = sum;
        b += 4 * share;
        if (b >= nb)
            break;
        v = s[min(b * kBlock + lane, n - 1)];
    }
}

// grid (heads / G, tokens, the positions' share), RW * HD threads: run r of RW,
// element d; G heads of a key-value head share the thread's 32 values.  (Eight
// query heads a key-value head go four a workgroup: with a run's eight chains
// in turn the step took 16.6 us at a prefix of 20, now 14.2.)
template <int HD, int G>
__global__ __launch_bounds__(256) void attn_split_values_kernel(
    int heads, int kv_heads, const int32_t *__restrict__ positions, int limit, const uint16_t *__restrict__ vcache,
    int context, int S, const float *__restrict__ sc, const float *__restrict__ bs, float *__restrict__ runs,
    const int32_t *__restrict__ slots, int nslots, int share) {
    constexpr int RW = 256 / HD, NT = RW * HD, kPos = RW * kRun;
    __shared__ float bl[G][256];
    __shared__ float tot[G];
    __shared__ __align__(16) uint16_t ps[G][kPos];
    const int tid = threadIdx.x;
    const int h0 = blockIdx.x * G, kvh = h0 / (heads / kv_heads), t = blockIdx.y, step = share * kPos;
    const int n = min(positions[t] + 1, limit), nb = (n + kBlock - 1) / kBlock;
    if ((int)blockIdx.z * kPos >= n)
        return;
    if (slots)
        vcache += (size_t)min(max(slots[t], 0), nslots - 1) * kv_heads * HD * context;
    const size_t row0 = (size_t)t * heads + h0;
    const int d = tid % HD, r = tid / HD;
    const uint16_t *vrow = vcache + ((size_t)kvh * HD + d) * context;
    v4u_stream v[4];
    auto vload = [&](int pr) __attribute__((always_inline)) {  // the run from position pr
#pragma unroll
        for (int u = 0; u < 4; u++)  // context is a multiple of 8; pieces past the prefix are read and not used
            v[u] = *(const v4u_stream *)(vrow + min(pr + 8 * u, context - 8));
    };
    vload(blockIdx.z * kPos + r * kRun);
    // the heads' totals, blocks in order, 256 blocks at a time
    float total = 0.0f;  // thread g < G: head g's
    for (int c0 = 0; c0 < nb; c0 += 256) {
        const int cn = min(256, nb - c0);
        __syncthreads();
        for (int i = tid; i < G * cn; i += NT) {
            const int g = i / cn, c = i - g * cn;
            bl[g][c] = bs[(row0 + g) * (S / kBlock) + c0 + c];
        }
        __syncthreads();
        if (tid < G) {
            int c = 0;
            for (; c + 8 <= cn; c += 8) {
                float w[8];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    w[u] = bl[tid][c + u];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    total = total + w[u];
            }
            for (; c < cn; c++)
                total = total + bl[tid][c];
        }
    }
    if (tid < G)
        tot[tid] = total;
    for (int p0 = blockIdx.z * kPos; p0 < n; p0 += step) {
        __syncthreads();  // the totals are there; the probabilities before are spent
        for (int i = tid; i < G * kPos; i += NT) {
            const int g = i / kPos, p = i - g * kPos;
            ps[g][p] = p0 + p < n
                           ? (uint16_t)float_to_half_bits(__fdiv_rn(sc[(row0 + g) * S + p0 + p], tot[g]))
                           : (uint16_t)0;
        }
        __syncthreads();
        const int pr = p0 + r * kRun, live = min(kRun, n - pr);  // the thread's run and its positions
        if (live > 0) {
            float acc[G];
#pragma unroll
            for (int g = 0; g < G; g++)
                acc[g] = 0.0f;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t vw[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int g = 0; g < G; g++) {
                    const v4u_stream pp = *(const v4u_stream *)(&ps[g][r * kRun + 8 * u]);
                    const uint32_t pw[4] = {pp.x, pp.y, pp.z, pp.w};
#pragma unroll
                    for (int c = 0; c < 8; c++)
                        if (8 * u + c < live)  // nothing past the prefix enters a sum
                            acc[g] = (c & 1) ? fma_mix_hi(pw[c >> 1], vw[c >> 1], acc[g])
                                             : fma_mix_lo(pw[c >> 1], vw[c >> 1], acc[g]);
                }
            }
#pragma unroll
            for (int g = 0; g < G; g++)
                runs[((row0 + g) * (S / kRun) + pr / kRun) * HD + d] = acc[g];
        }
        if (p0 + step < n)
            vload(pr + step);
    }
}

// grid (heads * HD / 64, tokens), 64 threads: an element's runs in order, a
// 32-lane group a Q8_0 block.
__global__ __launch_bounds__(64) void attn_split_finish_kernel(int heads, int hd, const int32_t *__restrict__ positions,
                                                               int limit, int S, const float *__restrict__ runs,
                                                               int8_t *__restrict__ q, float *__restrict__ scales,
                                                               int32_t *__restrict__ qsum) {
    const int lane = threadIdx.x, t = blockIdx.y;
    const int col = blockIdx.x * 64 + lane, width = heads * hd;
    const int n = min(positions[t] + 1, limit), nr = n > 0 ? (n + kRun - 1) / kRun : 0;
    const int h = min(col, width - 1) / hd, d = min(col, width - 1) - h * hd;
    const float *rr = runs + ((size_t)t * heads + h) * (S / kRun) * hd + d;
    float o = 0.0f;
    int r = 0;
    for (; r + 32 <= nr; r += 32) {  // thirty-two loads in flight
        float w[32];
#pragma unroll
        for (int u = 0; u < 32; u++)
            w[u] = rr[(size_t)(r + u) * hd];
#pragma unroll
        for (int u = 0; u < 32; u++)
            o = o + w[u];
    }
    for (; r < nr; r += 8) {
        float w[8];
#pragma unroll
        for (int u = 0; u < 8; u++)
            w[u] = rr[(size_t)min(r + u, nr - 1) * hd];
#pragma unroll
        for (int u = 0; u < 8; u++)
            o = r + u < nr ? o + w[u] : o;
    }
    float stored;
    int32_t sm;
    const int32_t nq = q8_0_lane(o, &stored, &sm);
    if (col < width) {
        q[(size_t)t * width + col] = (int8_t)nq;
        if ((lane & 31) == 0) {
            scales[(size_t)t * (width >> 5) + (col >> 5)] = stored;
            qsum[(size_t)t * (width >> 5) + (col >> 5)] = sm;
        }
    }
}

// ---- a workgroup a token and a few of its heads ------------------------------
//
// grid (heads / GH * HD / VD, tokens), 512 threads: the four steps above in one
// launch, for GH heads of a key-value head and VD of their elements, over the
// token's own prefix alone: the scores (a wavefront a block of 64 positions),
// the exponentials and block sums, the total, then the runs RW at a time,
// added in order as they come.  Every sum is the split form's, so the two give
// the same bits.  Scores and exponentials stay in LDS (SLDS) while GH rows of
// them take at most kRowsLds, else in the caller's rows (which one workgroup
// writes: VD is HD then).
// What bounds it: few tokens, one workgroup's chain of steps (about 1 us a 100
// positions, 0.5 with VD of 32, whose chunks are four times as long); many,
// the keys and values read once a GH heads.
constexpr int kRowsThreads = 512;
constexpr size_t kRowsLds = 32 * 1024;

template <int HD, int GH, int VD, bool SLDS>
__global__ __launch_bounds__(kRowsThreads) void attn_rows_kernel(
    const uint16_t *__restrict__ qh, int heads, int kv_heads, const int32_t *__restrict__ positions, int limit,
    const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, int context, float scale, int S,
    int8_t *__restrict__ q, float *__restrict__ scales, int32_t *__restrict__ qsum, float *sc, float *bs,
    const int32_t *__restrict__ slots, int nslots, int least) {
    constexpr int NT = kRowsThreads, NW = NT / 64, kPieces = HD / 8;
    constexpr int RW = NT / VD, kPos = RW * kRun;  // runs and positions a chunk
    static_assert(SLDS || VD == HD, "the caller's rows have one writer");
    extern __shared__ __align__(16) float dyn[];  // SLDS: [GH][S] scores, then exponentials; [GH][S / 64] block sums
    __shared__ __align__(16) v4u_stream qs[GH][kPieces];
    __shared__ float mw[NW][GH], tot[GH];
    __shared__ __align__(16) uint16_t ps[2][GH][kPos];
    __shared__ float rs[2][RW][GH][VD];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h0 = blockIdx.x / (HD / VD) * GH, d0 = blockIdx.x % (HD / VD) * VD;
    const int kvh = h0 / (heads / kv_heads), t = blockIdx.y;
    const int n = max(min(positions[t] + 1, limit), least);
    const int nb = n > 0 ? (n + kBlock - 1) / kBlock : 0, chunks = n > 0 ? (n + kPos - 1) / kPos : 0;
    if (slots) {  // reads stay inside the caches
        const size_t at = (size_t)min(max(slots[t], 0), nslots - 1) * kv_heads * HD * context;
        kcache += at;
        vcache += at;
    }
    const size_t row0 = (size_t)t * heads + h0;
    float *s = SLDS ? dyn : sc + row0 * S;
    float *bsum = SLDS ? dyn + (size_t)GH * S : bs + row0 * (S / kBlock);
    const int d = tid % VD, r = tid / VD;  // this thread's element and run of a chunk (none past RW)
    const uint16_t *vrow = vcache + ((size_t)kvh * HD + d0 + d) * context;
    auto vload = [&](v4u_stream *v, int pr) __attribute__((always_inline)) {  // the run from position pr
        if (pr < n) {
#pragma unroll
            for (int u = 0; u < 4; u++)  // context is a multiple of 8; pieces past the prefix are not used
                v[u] = *(const v4u_stream *)(vrow + min(pr + 8 * u, context - 8));
        }
    };
    v4u_stream v[4] = {};
    vload(v, r * kRun);
    if (tid < GH * kPieces)
        (&qs[0][0])[tid] = ((const v4u_stream *)(qh + row0 * HD))[tid];
    __syncthreads();

    // the scores and their maximum
    float m[GH];
#pragma unroll
    for (int g = 0; g < GH; g++)
        m[g] = -INFINITY;
    for (int b = wave; b < nb; b += NW) {
        const int p = b * kBlock + lane;
        const v4u_stream *kr = (const v4u_stream *)(kcache + (size_t)kvh * HD * context) + min(p, n - 1);
        v4u_stream k[kPieces];
#pragma unroll
        for (int i = 0; i < kPieces; i++)
            k[i] = kr[(size_t)i * context];
        asm volatile("" ::: "memory");  // the queries are read here, not kept across the loop (GH of 4: 256 registers)
#pragma unroll
        for (int g = 0; g < GH; g++) {
            float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
#pragma unroll
            for (int i = 0; i < kPieces; i++) {
                const v4u_stream qq = qs[g][i], kk = k[i];
                s0 = fma_mix_lo(qq.x, kk.x, s0);
                s1 = fma_mix_hi(qq.x, kk.x, s1);
                s2 = fma_mix_lo(qq.y, kk.y, s2);
                s3 = fma_mix_hi(qq.y, kk.y, s3);
                s0 = fma_mix_lo(qq.z, kk.z, s0);
                s1 = fma_mix_hi(qq.z, kk.z, s1);
                s2 = fma_mix_lo(qq.w, kk.w, s2);
                s3 = fma_mix_hi(qq.w, kk.w, s3);
            }
            const float x = scale * ((s0 + s1) + (s2 + s3));
            if (p < n) {
                s[(size_t)g * S + p] = x;
                m[g] = fmaxf(m[g], x);
            }
        }
    }
#pragma unroll
    for (int g = 0; g < GH; g++) {
        m[g] = wave_max(m[g]);
        if (lane == 0)
            mw[wave][g] = m[g];
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < GH; g++)
#pragma unroll
        for (int w = 0; w < NW; w++)
            m[g] = fmaxf(m[g], mw[w][g]);

    // the exponentials in place (a lane's own scores) and the block sums
    for (int b = wave; b < nb; b += NW) {
        const int p = b * kBlock + lane;
        float df[GH], e[GH];
#pragma unroll
        for (int g = 0; g < GH; g++)
            df[g] = (p < n ? s[(size_t)g * S + p] : m[g]) - m[g];
        exp_neg_n<GH>(df, e);
#pragma unroll
        for (int g = 0; g < GH; g++) {
            e[g] = p < n ? e[g] : 0.0f;
            if (p < n)
                s[(size_t)g * S + p] = e[g];
            const float sum = wave_pairwise_sum(e[g]);
            if (lane == 0)
                bsum[g * (S / kBlock) + b] = sum;
        }
    }
    __syncthreads();
    // the totals, blocks in order: wavefront g head g's
    if (wave < GH) {
        float total = 0.0f;
        for (int c0 = 0; c0 < nb; c0 += 64) {
            const float w = bsum[wave * (S / kBlock) + min(c0 + lane, nb - 1)];
            const int cn = min(64, nb - c0);
            for (int i = 0; i < cn; i++)
                total = total + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), i));
        }
        if (lane == 0)
            tot[wave] = total;
    }
    __syncthreads();

    // the value sums: a chunk's probabilities, then its runs, added to the
    // outputs while the next chunk's are taken
    float o = 0.0f;  // thread g * VD + d: head g's element d
    const int og = tid / VD;
    for (int c = 0; c < chunks; c++) {
        const int buf = c & 1, p0 = c * kPos, pr = p0 + r * kRun;
        for (int i = tid; i < GH * kPos; i += NT) {
            const int g = i / kPos, p = i - g * kPos;
            ps[buf][g][p] = p0 + p < n ? (uint16_t)float_to_half_bits(__fdiv_rn(s[(size_t)g * S + p0 + p], tot[g]))
                                       : (uint16_t)0;
        }
        v4u_stream vn[4] = {};
        vload(vn, pr + kPos);
        __syncthreads();
        if (c > 0 && tid < GH * VD) {
#pragma unroll
            for (int i = 0; i < RW; i++)
                o = o + rs[buf ^ 1][i][og][d];
        }
        const int live = r < RW ? min(kRun, n - pr) : 0;  // the run's positions
        if (live > 0) {
            float acc[GH];
#pragma unroll
            for (int g = 0; g < GH; g++)
                acc[g] = 0.0f;
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const uint32_t vw[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                for (int g = 0; g < GH; g++) {
                    const v4u_stream pp = *(const v4u_stream *)(&ps[buf][g][r * kRun + 8 * u]);
                    const uint32_t pw[4] = {pp.x, pp.y, pp.z, pp.w};
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (8 * u + e < live)  // nothing past the prefix enters a sum
                            acc[g] = (e & 1) ? fma_mix_hi(pw[e >> 1], vw[e >> 1], acc[g])
                                             : fma_mix_lo(pw[e >> 1], vw[e >> 1], acc[g]);
                }
            }
#pragma unroll
            for (int g = 0; g < GH; g++)
                rs[buf][r][g][d] = acc[g];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
            v[u] = vn[u];
    }
    __syncthreads();
    if (tid < GH * VD) {
        const int last = chunks - 1, runs = (n - last * kPos + kRun - 1) / kRun;  // of the last chunk
        if (chunks > 0) {
#pragma unroll
            for (int i = 0; i < RW; i++)
                o = i < runs ? o + rs[last & 1][i][og][d] : o;
        }
        // whole 32-lane groups, a Q8_0 block each
        const int width = heads * HD, col = (h0 + og) * HD + d0 + d;
        float stored;
        int32_t sm;
        const int32_t nq = q8_0_lane(o, &stored, &sm);
        q[(size_t)t * width + col] = (int8_t)nq;
        if ((lane & 31) == 0) {
            scales[(size_t)t * (width >> 5) + (col >> 5)] = stored;
            qsum[(size_t)t * (width >> 5) + (col >> 5)] = sm;
        }
    }
}

// ---- a prompt ---------------------------------------------------------------
//
// grid (heads, ceil(M / 32)), a workgroup per (query head, 32-token tile), NW
// wavefronts, each with its own 64-position blocks of the prefix (block b:
// wavefront b % NW; of the last sweep's values, the groups b % 8 that leave the
// wavefront's number when divided by NW).  The scores are taken transposed, positions by tokens
// (v_mfma_f32_32x32x16_f16, the keys as the row operand): a lane then holds
// sixteen positions of one token, so that
//   - the token's maximum and the pairwise block sums are sums over the lane's
//     own registers and one exchange with lane ^ 32 (positions 4 .. 7 of every
//     eight), no tree across the wavefront;
//   - the probabilities are, as they stand, the column operand of the value
//     product (elements by tokens): k-slot (g, j) of a step is position 4 g + j
//     (j < 4) or 8 + 4 g + j - 4 of its sixteen, and the values are read in
//     that order.  Nothing passes through LDS and no barrier stands between a
//     block's steps.
// A probability needs its token's total before it can be rounded, and a total
// its maximum, so the prefix is swept three times (maximum; block sums;
// probabilities and values), the scores and exponentials computed again each
// time: both cost less than writing them out and reading them back (1,500
// tokens of 32 heads: 144 MB).  The keys, 32 KB a wavefront's block, come
// from the L2.  The value sums of the eight groups of blocks (b % 8) are added
// pairwise at the end (c + 4, then c + 2, c + 1).
// What bounds it: the exponentials (float64, twice) and the MFMAs, about 900
// and 300 cycles a 32 x 32 tile and sweep.  1,500 tokens of 32 heads: 154 us in
// a replayed graph, where the serial passes took 679 (scores 226, softmax 132,
// values 321).
typedef _Float16 pl_v8h __attribute__((ext_vector_type(8)));
typedef float pl_v16f __attribute__((ext_vector_type(16)));
typedef uint32_t pl_v2u __attribute__((ext_vector_type(2)));

constexpr int kPlTok = 32;
constexpr int kPlGroups = 8;  // blocks b with the same b % 8 make one value sum

template <int HD, int NW>
__global__ __launch_bounds__(64 * NW, HD <= 64 ? 4 : 2) void attn_prompt_long_kernel(
    const uint16_t *__restrict__ qh, int M, int heads, int kv_heads, const int32_t *__restrict__ positions,
    int limit, const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, int context, float scale,
    int8_t *__restrict__ q, float *__restrict__ scales, int32_t *__restrict__ qsum, float *__restrict__ heads_f) {
    constexpr int KS = HD / 16, DB = HD / 32;
    using Own = std::integral_constant<int, NW>;
    using Group = std::integral_constant<int, kPlGroups>;
    extern __shared__ __align__(16) float sl[];  // block sums [blocks][32]; then the value sums and the output tile
    __shared__ float mw[NW][kPlTok];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, g = lane >> 5;
    // a key-value head's query heads one XCD apart in the grid's order (they
    // read the same keys), the longest prefixes first
    const int kvh = blockIdx.x % kv_heads, h = kvh * (heads / kv_heads) + blockIdx.x / kv_heads;
    const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * kPlTok, t = t0 + li;
    // this lane's token's positions (a negative position: as the LDS form to
    // 1024 positions, one; as the serial passes past them, none)
    const int n = t < M ? max(min(positions[t] + 1, limit), limit <= kOne ? 1 : 0) : 0;
    int nmax = n, nmin = t < M ? n : limit;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
        nmax = max(nmax, __shfl_xor(nmax, off, 64));
        nmin = min(nmin, __shfl_xor(nmin, off, 64));
    }
    nmax = __builtin_amdgcn_readfirstlane(nmax);
    nmin = __builtin_amdgcn_readfirstlane(nmin);
    const int nb = (nmax + kBlock - 1) / kBlock;

    pl_v8h qf[KS];  // the token's query: elements 16 s + 8 g ..
    {
        const uint16_t *qr = qh + ((size_t)min(t, M - 1) * heads + h) * HD + 8 * g;
#pragma unroll
        for (int s = 0; s < KS; s++)
            qf[s] = *(const pl_v8h *)(qr + 16 * s);
    }
    const char *kb = (const char *)(kcache + (size_t)kvh * HD * context);
    auto kload = [&](int p0, pl_v8h *k) __attribute__((always_inline)) {  // key rows p0 + li (past the prefix: its last)
        const int p = min(p0 + li, nmax - 1);
#pragma unroll
        for (int s = 0; s < KS; s++)
            k[s] = *(const pl_v8h *)(kb + ((uint32_t)((2 * s + g) * context + p) * 16u));
    };
    // scores of positions p0 + 8 (e / 4) + 4 g + e % 4 for this lane's token
    auto score = [&](const pl_v8h *k, float *s) __attribute__((always_inline)) {
        pl_v16f acc = {};
#pragma unroll
        for (int i = 0; i < KS; i++)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(k[i], qf[i], acc, 0, 0, 0);
#pragma unroll
        for (int e = 0; e < 16; e++)
            s[e] = scale * acc[e];
    };
    // the lane's e-th position of a tile is 8 (e / 4) + 4 g + e % 4 in: below `own` = left(first position, end) or not
    auto left = [&](int p0, int end) __attribute__((always_inline)) { return end - p0 - 4 * g; };
    auto in = [](int own, int e) __attribute__((always_inline)) { return 8 * (e >> 2) + (e & 3) < own; };
    // every tile of blocks b0, b0 + step, ..: f(first position, scores), the
    // next tile's keys on their way
    auto sweep = [&](int b0, auto step_tag, auto &&f) __attribute__((always_inline)) {
        constexpr int step = decltype(step_tag)::value;
        pl_v8h k[KS];
        if (b0 < nb)
            kload(b0 * kBlock, k);
        for (int b = b0; b < nb; b += step) {
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                const int p0 = b * kBlock + 32 * hf;
                float s[16];
                score(k, s);
                kload(hf ? (b + step < nb ? (b + step) * kBlock : p0) : p0 + 32, k);
                f(p0, s, hf);
            }
        }
    };

    // the maximum
    float m = -INFINITY;
    sweep(wave, Own{}, [&](int p0, const float *s, int) __attribute__((always_inline)) {
        if (p0 + 32 <= nmin) {
#pragma unroll
            for (int e = 0; e < 16; e++)
                m = fmaxf(m, s[e]);
        } else {
            const int own = left(p0, n);
#pragma unroll
            for (int e = 0; e < 16; e++)
                m = in(own, e) ? fmaxf(m, s[e]) : m;
        }
    });
    m = fmaxf(m, __shfl_xor(m, 32, 64));
    if (g == 0)
        mw[wave][li] = m;
    __syncthreads();
    m = mw[0][li];
#pragma unroll
    for (int w = 1; w < NW; w++)
        m = fmaxf(m, mw[w][li]);

    // a tile's exponentials, +0 past the token's own positions
    auto exps = [&](int p0, const float *s, float *e16) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            float d[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                d[e] = s[4 * c + e] - m;
            exp_neg_n<4>(d, e16 + 4 * c);
            __builtin_amdgcn_sched_barrier(0);  // four chains side by side: more would spill
        }
        if (p0 + 32 > nmin) {
            const int own = left(p0, n);
#pragma unroll
            for (int e = 0; e < 16; e++)
                e16[e] = in(own, e) ? e16[e] : 0.0f;
        }
    };

    // the block sums, pairwise in position order: two and four within the
    // lane, eight with lane ^ 32, sixteen and thirty-two within the lane, the
    // block's two tiles
    float half_sum = 0.0f;
    sweep(wave, Own{}, [&](int p0, const float *s, int hf) __attribute__((always_inline)) {
        float e16[16], c4[4];
        exps(p0, s, e16);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            c4[c] = (e16[4 * c] + e16[4 * c + 1]) + (e16[4 * c + 2] + e16[4 * c + 3]);
            c4[c] = c4[c] + __shfl_xor(c4[c], 32, 64);
        }
        const float tile = (c4[0] + c4[1]) + (c4[2] + c4[3]);
        if (hf == 0)
            half_sum = tile;
        else if (g == 0)
            sl[(p0 / kBlock) * kPlTok + li] = half_sum + tile;
    });
    __syncthreads();
    float total = 0.0f;  // the blocks in order
    {
        const int own = (n + kBlock - 1) / kBlock;
        int b = 0;
        for (; b + 8 <= nb; b += 8) {
            float w[8];
#pragma unroll
            for (int u = 0; u < 8; u++)
                w[u] = sl[(b + u) * kPlTok + li];
#pragma unroll
            for (int u = 0; u < 8; u++)
                total = b + u < own ? total + w[u] : total;
        }
        for (; b < nb; b++)
            total = b < own ? total + sl[b * kPlTok + li] : total;
    }

    // the probabilities and the value sums
    pl_v16f acc[DB];
#pragma unroll
    for (int db = 0; db < DB; db++)
        acc[db] = pl_v16f{};
    const char *vb = (const char *)(vcache + (size_t)kvh * HD * context);  // 32-bit offsets, as the keys'
    // a tile's probabilities, fp16 pairs
    auto probs = [&](int p0, const float *s, uint32_t *ph) __attribute__((always_inline)) {
        float e16[16];
        exps(p0, s, e16);
#pragma unroll
        for (int e = 0; e < 16; e += 2) {
            ph[e >> 1] = float_to_half_bits(__fdiv_rn(e16[e], total)) |
                         (float_to_half_bits(__fdiv_rn(e16[e + 1], total)) << 16);
            __builtin_amdgcn_sched_barrier(0);
        }
        if (p0 + 32 > nmin) {  // past the token's own positions +0 (0 / total is NaN where no position is visible)
            const int own = left(p0, n);
#pragma unroll
            for (int e = 0; e < 16; e += 2)
                ph[e >> 1] &= (in(own, e) ? 0x0000FFFFu : 0u) | (in(own, e + 1) ? 0xFFFF0000u : 0u);
        }
    };
    auto vload = [&](int p0, int db, int st, int u) __attribute__((always_inline)) {
        return *(const pl_v2u *)(vb + ((uint32_t)((32 * db + li) * context +
                                                  min(p0 + 16 * st + 8 * u + 4 * g, context - 4)) *
                                       2u));
    };
    // A later token's infinite or NaN value must not reach an earlier one as
    // 0 * inf: the wavefront's tiles from the first with such a value past
    // some token's own positions wait.  (Looked for ahead of the sweep: in it,
    // where the values are at hand, it spilled, 172 -> 186 us.)
    //
    // The value sums go by eight groups of blocks whatever the wavefronts, so
    // that a token's bits do not depend on the batch it came in: of four
    // wavefronts each takes its upper group first and leaves that sum in LDS.
    float *upper = sl + (size_t)wave * DB * 16 * 64 + lane;
    __syncthreads();  // the block sums are spent
#pragma unroll 1
    for (int group = wave + kPlGroups - NW; group >= 0; group -= NW) {
        int late = nmax;
        int b0 = group;
        while (b0 < nb && (b0 + 1) * kBlock <= nmin)
            b0 += kPlGroups;
#pragma unroll 1
        for (int p0 = b0 * kBlock; p0 < late; p0 += (p0 & 32) ? kPlGroups * kBlock - 32 : 32) {
            const int own = left(p0, nmax);
            uint32_t any = 0;
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int w = 0; w < 8; w++) {
                    const int e = 2 * w;
                    const uint32_t keep = (in(own, e) ? 0x7FFFu : 0u) | (in(own, e + 1) ? 0x7FFF0000u : 0u);
                    // an exponent of all ones carries into the half's sign place
                    any |= ((vload(p0, db, w >> 2, (w >> 1) & 1)[w & 1] & keep) + 0x04000400u) & 0x80008000u;
                }
            if (p0 + 32 > nmin && __ballot(any != 0) != 0)
                late = p0;
        }
        late = __builtin_amdgcn_readfirstlane(late);
        sweep(group, Group{}, [&](int p0, const float *s, int) __attribute__((always_inline)) {
            if (p0 >= late)
                return;
            pl_v2u v[DB][2][2];  // [element block][k-step][positions 4 g .., 8 + 4 g ..]
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int st = 0; st < 2; st++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        v[db][st][u] = vload(p0, db, st, u);
            uint32_t ph[8];
            probs(p0, s, ph);
            if (p0 + 32 > nmax) {  // values past the tile's last position may be unwritten: zeros
                const int own = left(p0, nmax);
#pragma unroll
                for (int st = 0; st < 2; st++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
#pragma unroll
                        for (int c = 0; c < 2; c++) {
                            const int e = 8 * st + 4 * u + 2 * c;
                            const uint32_t keep = (in(own, e) ? 0x0000FFFFu : 0u) | (in(own, e + 1) ? 0xFFFF0000u : 0u);
#pragma unroll
                            for (int db = 0; db < DB; db++)
                                v[db][st][u][c] &= keep;
                        }
            }
#pragma unroll
            for (int st = 0; st < 2; st++) {
                const uint4 pb = make_uint4(ph[4 * st], ph[4 * st + 1], ph[4 * st + 2], ph[4 * st + 3]);
#pragma unroll
                for (int db = 0; db < DB; db++) {
                    const uint4 va = make_uint4(v[db][st][0].x, v[db][st][0].y, v[db][st][1].x, v[db][st][1].y);
                    acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pl_v8h, va),
                                                                     __builtin_bit_cast(pl_v8h, pb), acc[db], 0, 0, 0);
                }
            }
        });

        // the tiles that waited, a token at a time with the values past it zeroed
#pragma unroll 1
        for (int p0 = late; p0 < nmax; p0 += (p0 & 32) ? kPlGroups * kBlock - 32 : 32) {
            uint32_t ph[8];
            {
                pl_v8h k[KS];
                float s[16];
                kload(p0, k);
                score(k, s);
                probs(p0, s, ph);
            }
#pragma unroll 1
            for (int tt = 0; tt < kPlTok; tt++) {
                const int own = left(p0, __builtin_amdgcn_readlane(n, tt));
#pragma unroll
                for (int db = 0; db < DB; db++) {
                    pl_v16f one = acc[db];
#pragma unroll
                    for (int st = 0; st < 2; st++) {
                        uint32_t vm[4];
#pragma unroll
                        for (int u = 0; u < 2; u++) {
                            const pl_v2u x = vload(p0, db, st, u);
#pragma unroll
                            for (int c = 0; c < 2; c++) {
                                const int e = 8 * st + 4 * u + 2 * c;
                                vm[2 * u + c] =
                                    x[c] & ((in(own, e) ? 0x0000FFFFu : 0u) | (in(own, e + 1) ? 0xFFFF0000u : 0u));
                            }
                        }
                        const uint4 pb = make_uint4(ph[4 * st], ph[4 * st + 1], ph[4 * st + 2], ph[4 * st + 3]);
                        const uint4 va = make_uint4(vm[0], vm[1], vm[2], vm[3]);
                        one = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pl_v8h, va),
                                                                     __builtin_bit_cast(pl_v8h, pb), one, 0, 0, 0);
                    }
#pragma unroll
                    for (int e = 0; e < 16; e++)
                        acc[db][e] = li == tt ? one[e] : acc[db][e];
                }
            }
        }
        if (NW < kPlGroups && group >= NW) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    upper[(db * 16 + e) * 64] = acc[db][e];
                    acc[db][e] = 0.0f;
                }
        }
    }
    if (NW < kPlGroups) {
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int e = 0; e < 16; e++)
                acc[db][e] = acc[db][e] + upper[(db * 16 + e) * 64];
        __syncthreads();  // the upper groups' sums are spent
    }

    // the wavefronts' sums: the upper half's added to the lower half's
#pragma unroll
    for (int half = NW / 2; half > 0; half >>= 1) {
        float *part = sl + (size_t)(wave & (half - 1)) * DB * 16 * 64 + lane;
        if (wave >= half && wave < 2 * half) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    part[(db * 16 + e) * 64] = acc[db][e];
        }
        __syncthreads();
        if (wave < half) {
#pragma unroll
            for (int db = 0; db < DB; db++)
#pragma unroll
                for (int e = 0; e < 16; e++)
                    acc[db][e] = acc[db][e] + part[(db * 16 + e) * 64];
        }
        __syncthreads();
    }
    // the head floats token by token, then four values a thread, eight lanes a
    // Q8_0 block
    constexpr int OS = HD + 4;
    if (wave == 0) {
#pragma unroll
        for (int db = 0; db < DB; db++)
#pragma unroll
            for (int c = 0; c < 4; c++)
                *(float4 *)(sl + li * OS + 32 * db + 8 * c + 4 * g) =
                    make_float4(acc[db][4 * c], acc[db][4 * c + 1], acc[db][4 * c + 2], acc[db][4 * c + 3]);
    }
    __syncthreads();
    const int width = heads * HD;
    for (int i4 = tid; i4 < kPlTok * (HD / 4); i4 += 64 * NW) {
        const int tk = i4 / (HD / 4), c4 = i4 - tk * (HD / 4);
        const float4 o = *(const float4 *)(sl + tk * OS + 4 * c4);
        const float v[4] = {o.x, o.y, o.z, o.w};
        float stored;
        int32_t sm;
        const uint32_t packed = q8_0_quad(v, &stored, &sm);
        if (t0 + tk < M) {
            const int col = h * HD + 4 * c4;
            if (heads_f)
                *(float4 *)(heads_f + (size_t)(t0 + tk) * width + col) = o;
            if (q) {
                *(uint32_t *)(q + (size_t)(t0 + tk) * width + col) = packed;
                if ((c4 & 7) != 0)
                    continue;
                scales[(size_t)(t0 + tk) * (width >> 5) + (col >> 5)] = stored;
                qsum[(size_t)(t0 + tk) * (width >> 5) + (col >> 5)] = sm;
            }
        }
    }
}

size_t prompt_long_lds(int hd, int limit) {
    const size_t sums = (size_t)((limit + kBlock - 1) / kBlock) * kPlTok;
    const size_t parts = (size_t)(kPlGroups / 2) * (hd / 32) * 16 * 64, tile = (size_t)kPlTok * (hd + 4);
    return sizeof(float) * std::max(sums, std::max(parts, tile));
}

}  // namespace

// The block sums have to fit the LDS, a key-value head's cache a 32-bit offset.
bool attn_prompt_long_fits(int hd, int limit, int context) {
    return prompt_long_lds(hd, limit) <= 150 * 1024 && (uint64_t)hd * context * sizeof(uint16_t) <= 1u << 31;
}

// Wavefronts a workgroup: eight to two workgroups a CU, four past that (us 8 /
// 4 at 1,100 positions: 32 heads of 128 256 tokens 48 / 57, 500 74 / 69, 544 95
// / 85, 1,000 113 / 102; 16 heads of 128 768 tokens 59 / 62; 32 of 64 512
// tokens 50 / 55, 1,000 69 / 70; the same bits).
int launch_attn_prompt_long(gx_ctx *ctx, const uint16_t *qh, int M, int heads, int kv_heads, int hd, int limit,
                            const int32_t *positions, const uint16_t *kcache, const uint16_t *vcache, int context,
                            float scale, int8_t *q, float *scales, int32_t *qsum, float *heads_f) {
    const dim3 grid((unsigned)heads, (unsigned)((M + kPlTok - 1) / kPlTok));
    const bool wide = (size_t)grid.x * grid.y <= 2 * (size_t)ctx->cu_count;
    const size_t lds = prompt_long_lds(hd, limit);
#define GX_PL(HH, WW)                                                                                                \
    attn_prompt_long_kernel<HH, WW><<<grid, 64 * WW, lds, ctx->stream>>>(qh, M, heads, kv_heads, positions, limit,   \
                                                                         kcache, vcache, context, scale, q, scales,  \
                                                                         qsum, heads_f)
#define GX_PL_W(HH)                                                                                                  \
    do {                                                                                                             \
        if (wide)                                                                                                    \
            GX_PL(HH, 8);                                                                                            \
        else                                                                                                         \
            GX_PL(HH, 4);                                                                                            \
    } while (0)
    if (hd == 32)
        GX_PL_W(32);
    else if (hd == 64)
        GX_PL_W(64);
    else if (hd == 96)
        GX_PL_W(96);
    else
        GX_PL_W(128);
#undef GX_PL_W
#undef GX_PL
    return check_launch("qwen_attention long prompt");
}

static size_t rows_lds(int gh, int S) { return (size_t)gh * (S + S / kBlock) * sizeof(float); }

// Whether a head's elements go 32 a workgroup: while the CUs hold them all.
static bool rows_sliced(gx_ctx *ctx, int M, int heads, int hd, int S) {
    return (size_t)M * heads * (hd / 32) <= 2 * (size_t)ctx->cu_count && rows_lds(1, S) <= kRowsLds;
}

// Which form a call past the one-kernel form's prefixes takes: a workgroup a
// token's heads, or the positions spread over the chip in four launches.  The
// launch covers `limit` positions; the tokens may be anywhere below (a step
// replayed from a graph).  The rows form is the faster for a lone
// conversation's tokens to 1,024 positions and for many tokens, the split form
// for few tokens far in.  32 heads of 128, us rows / split at positions 20 /
// 600 / 1023: one token 7.2 / 14.2, 10.3 / 15.6, 12.4 / 15.2; conversations:
// eight 7.0 / 14.7, 20.5 / 21.6, 28.7 / 23.5, twelve 7.9 / 14.9, 21 / 24, 29.6
// / 28.1, 32 10.6 / 28.4, 31 / 51, 44 / 62.  Far in: one token at 4,095 33 /
// 20, conversations at 2,999 sixteen 83 / 67, 24 131 / 135, 128 420 / 690.
// (The forms before them: one token in a cache of 1,024 9.2 at 20 and 23 at
// 1,023; the serial passes 16 and 44 for eight conversations, and 119, 166 and
// 565 at 2,999 for sixteen, 24 and 128.)
bool attn_rows_form(gx_ctx *ctx, int M, int heads, int limit, bool slots) {
    if (M > kSplitTokens)
        return true;
    return limit <= kOne && (!slots || (size_t)M * heads > (size_t)ctx->cu_count);
}

// sc: [M][heads][S] floats, bs: [M][heads][S / 64] floats (used past kRowsLds).
// Heads a workgroup: as many of a key-value head's as leave the CUs busy (us
// 1 / 2 / 4 heads, 32 of 128 at 1,024 positions: 16 tokens 45 / 32 / 38, 32
// tokens 82 / 48 / 44, 128 298 / 169 / 120).
int launch_attn_rows(gx_ctx *ctx, const uint16_t *qh, int M, int heads, int kv_heads, int hd, int limit, int S,
                     const int32_t *positions, const uint16_t *kcache, const uint16_t *vcache, int context,
                     float scale, int8_t *q, float *scales, int32_t *qsum, float *sc, float *bs, const int32_t *slots,
                     int nslots) {
    int gh = std::min(heads / kv_heads, 4);
    while (gh > 1 && (size_t)M * heads <= (gh == 4 ? 3 : 1) * (size_t)ctx->cu_count)
        gh /= 2;
    const size_t lds = rows_lds(gh, S);
    const bool sliced = gh == 1 && rows_sliced(ctx, M, heads, hd, S);
    // A negative position sees one position in a lone conversation's calls to
    // 1,024 positions, as a prompt's does there, and none in the others.
    const int least = !slots && limit <= kOne ? 1 : 0;
#define GX_ROWS(HH, GG, VV, LL)                                                                                      \
    attn_rows_kernel<HH, GG, VV, LL>                                                                                 \
        <<<dim3((unsigned)(heads / GG * (HH / VV)), (unsigned)M), kRowsThreads, LL ? lds : 0, ctx->stream>>>(        \
            qh, heads, kv_heads, positions, limit, kcache, vcache, context, scale, S, q, scales, qsum, sc, bs,       \
            slots, nslots, least)
#define GX_ROWS_G(HH, GG)                                                                                            \
    do {                                                                                                             \
        if (lds <= kRowsLds)                                                                                         \
            GX_ROWS(HH, GG, HH, true);                                                                               \
        else                                                                                                         \
            GX_ROWS(HH, GG, HH, false);                                                                              \
    } while (0)
#define GX_ROWS_H(HH)                                                                                                \
    do {                                                                                                             \
        if (sliced)                                                                                                  \
            GX_ROWS(HH, 1, 32, true);                                                                                \
        else if (gh == 1)                                                                                            \
            GX_ROWS_G(HH, 1);                                                                                        \
        else if (gh == 2)                                                                                            \
            GX_ROWS_G(HH, 2);                                                                                        \
        else                                                                                                         \
            GX_ROWS_G(HH, 4);                                                                                        \
    } while (0)
    if (hd == 32)
        GX_ROWS_H(32);
    else if (hd == 64)
        GX_ROWS_H(64);
    else if (hd == 96)
        GX_ROWS_H(96);
    else
        GX_ROWS_H(128);
#undef GX_ROWS_H
#undef GX_ROWS_G
#undef GX_ROWS
    return check_launch("qwen_attention rows");
}

// The runs' floats, past the scores' workspace.
size_t attn_split_workspace(int M, int heads, int S) {
    return (size_t)std::min(M, kSplitTokens) * heads * (S / kRun) * 128 * sizeof(float);
}

// A step's workgroups along the prefix: one a piece while their wavefronts
// (`others` a piece) number at most kSplitWaves, past that each takes several.
// So a step replayed for a long context does not pay for its empty workgroups:
// eight conversations of 32 heads at position 100, launched for 16,384, 31 ->
// 16 us, at position 16,383 231 -> 223.
static int split_share(int pieces, int others) { return std::min(pieces, std::max(1, kSplitWaves / others)); }

// M <= kSplitTokens.  sc: [M][heads][S] floats; small: as many halves (the
// block maxima and sums take an eighth of a half a position); runs:
// attn_split_workspace bytes.
int launch_attn_split(gx_ctx *ctx, const uint16_t *qh, int M, int heads, int kv_heads, int hd, int limit, int S,
                      const int32_t *positions, const uint16_t *kcache, const uint16_t *vcache, int context,
                      float scale, int8_t *q, float *scales, int32_t *qsum, float *sc, float *small, float *runs,
                      const int32_t *slots, int nslots) {
    const int G = heads / kv_heads, width = heads * hd;
    float *mx = small, *bs = small + (size_t)M * heads * (S / kBlock);
    const int nblocks = (limit + kBlock - 1) / kBlock, pw = 256 / hd * kRun, vx = heads / std::min(G, 4);
    const dim3 sgrid((unsigned)kv_heads, (unsigned)M, (unsigned)split_share(nblocks, heads * M));
    const dim3 egrid((unsigned)heads, (unsigned)M, (unsigned)split_share((nblocks + 3) / 4, 4 * heads * M));
    const dim3 vgrid((unsigned)vx, (unsigned)M, (unsigned)split_share((limit + pw - 1) / pw, 4 * vx * M));
#define GX_SPLIT_V(HH, GG)                                                                                           \
    attn_split_values_kernel<HH, GG><<<vgrid, (256 / HH) * HH, 0, ctx->stream>>>(                                    \
        heads, kv_heads, positions, limit, vcache, context, S, sc, bs, runs, slots, nslots, (int)vgrid.z)
#define GX_SPLIT(HH)                                                                                                 \
    do {                                                                                                             \
        attn_split_scores_kernel<HH><<<sgrid, 64 * G, 0, ctx->stream>>>(qh, heads, kv_heads, positions, limit,       \
                                                                        kcache, context, scale, S, sc, mx, slots,    \
                                                                        nslots, (int)sgrid.z);                       \
        attn_split_exp_kernel<<<egrid, 256, 0, ctx->stream>>>(heads, kv_heads, positions, limit, S, sc, mx, bs,      \
                                                              (int)egrid.z);                                         \
        if (G == 1)                                                                                                  \
            GX_SPLIT_V(HH, 1);                                                                                       \
        else if (G == 2)                                                                                             \
            GX_SPLIT_V(HH, 2);                                                                                       \
        else                                                                                                         \
            GX_SPLIT_V(HH, 4);                                                                                       \
    } while (0)
    if (hd == 32)
        GX_SPLIT(32);
    else if (hd == 64)
        GX_SPLIT(64);
    else if (hd == 96)
        GX_SPLIT(96);
    else
        GX_SPLIT(128);
#undef GX_SPLIT
#undef GX_SPLIT_V
    attn_split_finish_kernel<<<dim3((unsigned)((width + 63) / 64), (unsigned)M), 64, 0, ctx->stream>>>(
        heads, hd, positions, limit, S, runs, q, scales, qsum);
    return check_launch("qwen_attention split");
}

}  // namespace gx
