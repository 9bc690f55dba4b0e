// gx_attn_long.hip - the parallel-order attention past the prefixes that one
// workgroup holds (gx_qwen.hip): a decode step's positions spread over the
// chip, and a prompt's attention on the matrix cores with nothing but the
// block sums kept between its sweeps.
//
// Both compute what the short forms compute (qwen/attention.go:96-124,
// nn/ops.go:59-73): the scores, their maximum, the float64 exponential of the
// float difference rounded to float (exp_neg), the total as 64-position blocks
// summed pairwise and the blocks added in order, the probabilities divided
// and rounded through fp16, the value sums.
#include <algorithm>

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

constexpr int kBlock = 64;  // positions a block of the softmax total
constexpr int kRun = 32;    // positions a run of the value sums

// ---- one position at a time (M <= 4, or one per conversation) ---------------
//
// Four launches, each spread over the prefix, so that the step's time does not
// grow with it until the chip is full: the scores (a wavefront a head and 64
// positions) with each block's maximum; the exponentials with each block's
// sum; the probabilities and the runs' value chains; the runs in order with
// the Q8_0.  The order of every sum is attn_par_kernel's, whatever the
// extent.  What bounds it: the launches (about 2 us each) and their load
// latencies; the bytes of 3,000 positions (12 MB) take 2 us.  The serial
// passes it replaces took 104 us there (one lane's 3,000-step softmax total
// 59, the value chains 38); these take 4.8 + 2.8 + 7.7 + 4.6.

// grid (kv_heads, S / 64, tokens), 64 threads a query head of the group.
template <int HD>
__global__ __launch_bounds__(512) void attn_split_scores_kernel(
    const uint16_t *__restrict__ qh, int heads, int kv_heads, const int32_t *__restrict__ positions, int limit,
    const uint16_t *__restrict__ kcache, int context, float scale, int S, float *__restrict__ sc,
    float *__restrict__ mx, const int32_t *__restrict__ slots, int nslots) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kvh = blockIdx.x, b = blockIdx.y, t = blockIdx.z;
    const int h = kvh * (heads / kv_heads) + wave;
    const int n = min(positions[t] + 1, limit);
    if (b * kBlock >= n)
        return;
    if (slots)
        kcache += (size_t)min(max(slots[t], 0), nslots - 1) * kv_heads * HD * context;
    const int p = b * kBlock + lane;
    const v4u_stream *kr = (const v4u_stream *)(kcache + (size_t)kvh * HD * context) + min(p, n - 1);
    v4u_stream k[HD / 8];
#pragma unroll
    for (int i = 0; i < HD / 8; i++)
        k[i] = kr[(size_t)i * context];
    // the query is one address for the wavefront
    const v4u_stream *qv = (const v4u_stream *)(qh + ((size_t)t * heads + h) * HD);
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
    const size_t row = (size_t)t * heads + h;
    if (p < n)
        sc[row * S + p] = v;
    const float m = wave_max(p < n ? v : -INFINITY);
    if (lane == 0)
        mx[row * (S / kBlock) + b] = m;
}

// grid (S / 256, heads, tokens), a wavefront a block: exponentials in place.
__global__ __launch_bounds__(256) void attn_split_exp_kernel(int heads, const int32_t *__restrict__ positions,
                                                             int limit, int S, float *__restrict__ sc,
                                                             const float *__restrict__ mx, float *__restrict__ bs) {
    const int lane = threadIdx.x & 63, b = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int t = blockIdx.z;
    const int n = min(positions[t] + 1, limit), nb = (n + kBlock - 1) / kBlock;
    if (b >= nb)
        return;
    const size_t row = (size_t)t * heads + blockIdx.y;
    const int p = b * kBlock + lane;
    float *s = sc + row * S;
    const float v = s[min(p, n - 1)];
    const float *mr = mx + row * (S / kBlock);
    float m = -INFINITY;
    for (int i = lane; i < nb; i += 64)
        m = fmaxf(m, mr[i]);
    m = wave_max(m);
    const float e = p < n ? exp_neg(v - m) : 0.0f;
    s[p] = e;  // S is a whole number of blocks
    const float sum = wave_pairwise_sum(e);
    if (lane == 0)
        bs[row * (S / kBlock) + b] = sum;
}

// grid (kv_heads, S / (32 RW), tokens), RW * HD threads: run r of RW, element
// d; the group's heads share the thread's 32 values.
template <int HD, int G>
__global__ __launch_bounds__(256) void attn_split_values_kernel(
    int heads, int kv_heads, const int32_t *__restrict__ positions, int limit, const uint16_t *__restrict__ vcache,
    int context, int S, const float *__restrict__ sc, const float *__restrict__ bs, float *__restrict__ runs,
    const int32_t *__restrict__ slots, int nslots) {
    constexpr int RW = 256 / HD, NT = RW * HD, kPos = RW * kRun;
    __shared__ float bl[G][256];
    __shared__ float tot[G];
    __shared__ __align__(16) uint16_t ps[G][kPos];
    const int tid = threadIdx.x;
    const int kvh = blockIdx.x, p0 = blockIdx.y * kPos, t = blockIdx.z;
    const int n = min(positions[t] + 1, limit), nb = (n + kBlock - 1) / kBlock;
    if (p0 >= n)
        return;
    if (slots)
        vcache += (size_t)min(max(slots[t], 0), nslots - 1) * kv_heads * HD * context;
    const size_t row0 = (size_t)t * heads + kvh * G;
    const int d = tid % HD, r = tid / HD;
    const int pr = p0 + r * kRun;  // the thread's run
    const uint16_t *vrow = vcache + ((size_t)kvh * HD + d) * context;
    v4u_stream v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)  // context is a multiple of 8; pieces past the prefix are read and not used
        v[u] = *(const v4u_stream *)(vrow + min(pr + 8 * u, context - 8));
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
    __syncthreads();
    for (int i = tid; i < G * kPos; i += NT) {
        const int g = i / kPos, p = i - g * kPos;
        ps[g][p] = p0 + p < n
                       ? (uint16_t)float_to_half_bits(__fdiv_rn(sc[(row0 + g) * S + p0 + p], tot[g]))
                       : (uint16_t)0;
    }
    __syncthreads();
    const int live = min(kRun, n - pr);  // the run's positions
    if (live <= 0)
        return;
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
                    acc[g] = (c & 1) ? fma_mix_hi(pw[c >> 1], vw[c >> 1], acc[g]) : fma_mix_lo(pw[c >> 1], vw[c >> 1], acc[g]);
        }
    }
#pragma unroll
    for (int g = 0; g < G; g++)
        runs[((row0 + g) * (S / kRun) + pr / kRun) * HD + d] = acc[g];
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

// ---- a prompt ---------------------------------------------------------------
//
// grid (heads, ceil(M / 32)), a workgroup per (query head, 32-token tile), NW
// wavefronts, each with its own 64-position blocks of the prefix (block b:
// wavefront b % NW).  The scores are taken transposed, positions by tokens
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
// from the L2.  The wavefronts' value sums are added pairwise at the end
// (w + NW/2, then w + NW/4, ...).
// What bounds it: the exponentials (float64, twice) and the MFMAs, about 900
// and 300 cycles a 32 x 32 tile and sweep.  1,500 tokens of 32 heads: 172 us,
// where the serial passes took 679 (scores 226, softmax 132, values 321).
typedef _Float16 pl_v8h __attribute__((ext_vector_type(8)));
typedef float pl_v16f __attribute__((ext_vector_type(16)));
typedef uint32_t pl_v2u __attribute__((ext_vector_type(2)));

constexpr int kPlTok = 32;
constexpr int kPlOne = 1024;  // positions the LDS form takes

template <int HD, int NW>
__global__ __launch_bounds__(64 * NW, 2) void attn_prompt_long_kernel(
    const uint16_t *__restrict__ qh, int M, int heads, int kv_heads, const int32_t *__restrict__ positions,
    int limit, const uint16_t *__restrict__ kcache, const uint16_t *__restrict__ vcache, int context, float scale,
    int8_t *__restrict__ q, float *__restrict__ scales, int32_t *__restrict__ qsum, float *__restrict__ heads_f) {
    constexpr int KS = HD / 16, DB = HD / 32;
    extern __shared__ __align__(16) float sl[];  // block sums [blocks][32]; at the end the value sums and the output tile
    __shared__ float mw[NW][kPlTok];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, g = lane >> 5;
    // a key-value head's query heads one XCD apart in the grid's order (they
    // read the same keys), the longest prefixes first
    const int kvh = blockIdx.x % kv_heads, h = kvh * (heads / kv_heads) + blockIdx.x / kv_heads;
    const int t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * kPlTok, t = t0 + li;
    // this lane's token's positions (a negative position: as the LDS form to
    // 1024 positions, one; as the serial passes past them, none)
    const int n = t < M ? max(min(positions[t] + 1, limit), limit <= kPlOne ? 1 : 0) : 0;
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
    // every tile of this wavefront's blocks: f(first position, scores), the
    // next tile's keys on their way
    auto sweep = [&](auto &&f) __attribute__((always_inline)) {
        pl_v8h k[KS];
        if (wave < nb)
            kload(wave * kBlock, k);
        for (int b = wave; b < nb; b += NW) {
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                const int p0 = b * kBlock + 32 * hf;
                float s[16];
                score(k, s);
                kload(hf ? (b + NW < nb ? (b + NW) * kBlock : p0) : p0 + 32, k);
                f(p0, s, hf);
            }
        }
    };

    // the maximum
    float m = -INFINITY;
    sweep([&](int p0, const float *s, int) __attribute__((always_inline)) {
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
    sweep([&](int p0, const float *s, int hf) __attribute__((always_inline)) {
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
    int late = nmax;
    int b0 = wave;
    while (b0 < nb && (b0 + 1) * kBlock <= nmin)
        b0 += NW;
#pragma unroll 1
    for (int p0 = b0 * kBlock; p0 < late; p0 += (p0 & 32) ? NW * kBlock - 32 : 32) {
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
    sweep([&](int p0, const float *s, int) __attribute__((always_inline)) {
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
    for (int p0 = late; p0 < nmax; p0 += (p0 & 32) ? NW * kBlock - 32 : 32) {
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

    // the wavefronts' sums: the upper half's added to the lower half's
    __syncthreads();  // the block sums are spent
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

size_t prompt_long_lds(int hd, int nw, int limit) {
    const size_t sums = (size_t)((limit + kBlock - 1) / kBlock) * kPlTok;
    const size_t parts = (size_t)(nw / 2) * (hd / 32) * 16 * 64, tile = (size_t)kPlTok * (hd + 4);
    return sizeof(float) * std::max(sums, std::max(parts, tile));
}

}  // namespace

// The block sums have to fit the LDS, a key-value head's cache a 32-bit offset.
bool attn_prompt_long_fits(int hd, int limit, int context) {
    return prompt_long_lds(hd, 8, limit) <= 150 * 1024 && (uint64_t)hd * context * sizeof(uint16_t) <= 1u << 31;
}

// Wavefronts a workgroup: eight while the tiles would leave CUs without one,
// four (two workgroups a CU) otherwise.
int launch_attn_prompt_long(gx_ctx *ctx, const uint16_t *qh, int M, int heads, int kv_heads, int hd, int limit,
                            const int32_t *positions, const uint16_t *kcache, const uint16_t *vcache, int context,
                            float scale, int8_t *q, float *scales, int32_t *qsum, float *heads_f) {
    const dim3 grid((unsigned)heads, (unsigned)((M + kPlTok - 1) / kPlTok));
    const bool wide = (size_t)grid.x * grid.y <= 2 * (size_t)ctx->cu_count;
    const int nw = wide ? 8 : 4;
    const size_t lds = prompt_long_lds(hd, nw, limit);
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

// The runs' floats of up to kSplitTokens tokens, past the scores' workspace.
constexpr int kSplitTokens = 16;
size_t attn_split_workspace(int M, int heads, int S) {
    return (size_t)std::min(M, kSplitTokens) * heads * (S / kRun) * 128 * sizeof(float);
}

// sc: [M][heads][S] floats; small: as many halves (the block maxima and sums
// take an eighth of a half a position); runs: attn_split_workspace bytes.
int launch_attn_split(gx_ctx *ctx, const uint16_t *qh, int M, int heads, int kv_heads, int hd, int limit, int S,
                      const int32_t *positions, const uint16_t *kcache, const uint16_t *vcache, int context,
                      float scale, int8_t *q, float *scales, int32_t *qsum, float *sc, float *small, float *runs,
                      const int32_t *slots, int nslots) {
    const int G = heads / kv_heads, width = heads * hd;
    float *mx = small, *bs = small + (size_t)std::min(M, kSplitTokens) * heads * (S / kBlock);
    const int nblocks = (limit + kBlock - 1) / kBlock;
    for (int t0 = 0; t0 < M; t0 += kSplitTokens) {
        const unsigned tn = (unsigned)std::min(kSplitTokens, M - t0);
        const uint16_t *qt = qh + (size_t)t0 * width;
        const int32_t *pos = positions + t0, *sl = slots ? slots + t0 : nullptr;
        const int rw = 256 / hd, pw = rw * kRun;
        const dim3 vgrid((unsigned)kv_heads, (unsigned)((limit + pw - 1) / pw), tn);
#define GX_SPLIT_V(HH, GG)                                                                                           \
    attn_split_values_kernel<HH, GG><<<vgrid, (256 / HH) * HH, 0, ctx->stream>>>(                                    \
        heads, kv_heads, pos, limit, vcache, context, S, sc, bs, runs, sl, nslots)
#define GX_SPLIT(HH)                                                                                                 \
    do {                                                                                                             \
        attn_split_scores_kernel<HH><<<dim3((unsigned)kv_heads, (unsigned)nblocks, tn), 64 * G, 0, ctx->stream>>>(   \
            qt, heads, kv_heads, pos, limit, kcache, context, scale, S, sc, mx, sl, nslots);                         \
        attn_split_exp_kernel<<<dim3((unsigned)((nblocks + 3) / 4), (unsigned)heads, tn), 256, 0, ctx->stream>>>(    \
            heads, pos, limit, S, sc, mx, bs);                                                                       \
        if (G == 1)                                                                                                  \
            GX_SPLIT_V(HH, 1);                                                                                       \
        else if (G == 2)                                                                                             \
            GX_SPLIT_V(HH, 2);                                                                                       \
        else if (G == 4)                                                                                             \
            GX_SPLIT_V(HH, 4);                                                                                       \
        else                                                                                                         \
            GX_SPLIT_V(HH, 8);                                                                                       \
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
        attn_split_finish_kernel<<<dim3((unsigned)((width + 63) / 64), tn), 64, 0, ctx->stream>>>(
            heads, hd, pos, limit, S, runs, q + (size_t)t0 * width, scales + (size_t)t0 * (width >> 5),
            qsum + (size_t)t0 * (width >> 5));
        if (int rc = check_launch("qwen_attention split"))
            return rc;
    }
    return GX_OK;
}

}  // namespace gx
