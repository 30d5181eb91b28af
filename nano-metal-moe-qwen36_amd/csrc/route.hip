/*
 * route.hip -- router logits and bit-exact softmax / top-k / renormalise.
 *
 * Reference behaviour (file:line relative to the reference root):
 *   logits : metal/kernels.metal:472-513 (q4 router rows of
 *            nmoe_route_shared_q4); the benchmark configs use a dense bf16
 *            router [256][2048] instead.
 *   routing: src/runtime.m:1498-1511 runs, on the host,
 *            math.m:67-93  softmax  (max; expf(v-max); long double sum;
 *                                    multiply by 1/(float)sum)
 *            math.m:95-132 top-k    (k arg-max passes; a tie goes to the
 *                                    lower index)
 *            math.m:134-153 renormalise (fp32 sum; multiply by 1/sum).
 *
 * Here the whole routing runs in one wavefront per token.  The selected
 * indices depend on exact probability ties, so every step reproduces the
 * host arithmetic bit for bit: expf is glibc's algorithm restated in double
 * (nmoe_exact.h), and the long double running sum is either proven exact
 * (every term >= 2^-32, summed as integers in units of 2^-55) or replayed
 * sequentially with an emulated 64-bit-significand adder in lane 0.
 *
 * Logits use a fixed reduction order (lane L accumulates its 16-byte chunks
 * L, L+64, ... with fma; the 64 lane partials are combined by the balanced
 * pairwise tree over lanes in order), so identical inputs give identical
 * logits on every run, in both the standalone and the fused kernels.
 */
#include <type_traits>

#include "nmoe_device.h"

#pragma clang fp contract(off)

static __constant__ uint64_t nmoe_exp2_tab[32] = NMOE_EXP2_TAB32;

/* ------------------------------------------------------------- logits */

/* One wavefront per (row, token block): logits[t][e] for t in [t0, t1). */
template <typename XT>
__global__ void __launch_bounds__(64) nmoe_router_bf16_kernel(const uint16_t *__restrict__ w, const XT *__restrict__ x,
                                                              int ntok, int num_experts, int tok_per_block,
                                                              float *__restrict__ logits) {
    const int e = blockIdx.x;
    const int lane = threadIdx.x;
    const uint4 *row = (const uint4 *)(w + (size_t)e * NMOE_HIDDEN);
    uint4 wv[4];
#pragma unroll
    for (int j = 0; j < 4; j++) wv[j] = row[lane + 64 * j];
    int t0 = blockIdx.y * tok_per_block;
    int t1 = min(ntok, t0 + tok_per_block);
    for (int t = t0; t < t1; t++) {
        const XT *xt = x + (size_t)t * NMOE_HIDDEN;
        float xs[32];
#pragma unroll
        for (int j = 0; j < 4; j++) nmoe_load_cols<XT>(xt, (lane + 64 * j) * 8, 8, xs + 8 * j);
        float logit = nmoe_router_row_bf16(wv, xs);
        if (lane == 0) logits[(size_t)t * num_experts + e] = logit;
    }
}

/* q4 router row (the reference model's router, kernels.metal:472-513):
 * 256 words; lane L owns words L, L+64, L+128, L+192 and accumulates
 * acc + fma(q, s*x, b*x) per column (kernels.metal:500-508); lane partials
 * combined by the pairwise tree. */
template <typename XT>
__global__ void __launch_bounds__(64) nmoe_router_q4_kernel(const uint32_t *__restrict__ w,
                                                            const uint16_t *__restrict__ sc,
                                                            const uint16_t *__restrict__ bi, const XT *__restrict__ x,
                                                            int ntok, int num_experts, int tok_per_block,
                                                            float *__restrict__ logits) {
    const int e = blockIdx.x;
    const int lane = threadIdx.x;
    uint32_t wv[4];
    float s[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        int c = lane + 64 * j;
        wv[j] = w[(size_t)e * (NMOE_HIDDEN / 8) + c];
        s[j] = nmoe_bf16f(sc[(size_t)e * (NMOE_HIDDEN / NMOE_GROUP) + c / 8]);
        b[j] = nmoe_bf16f(bi[(size_t)e * (NMOE_HIDDEN / NMOE_GROUP) + c / 8]);
    }
    int t0 = blockIdx.y * tok_per_block;
    int t1 = min(ntok, t0 + tok_per_block);
    for (int t = t0; t < t1; t++) {
        const XT *xt = x + (size_t)t * NMOE_HIDDEN;
        float acc = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float xv[8];
            nmoe_load_cols<XT>(xt, (lane + 64 * j) * 8, 8, xv);
#pragma unroll
            for (int i = 0; i < 8; i++) acc = nmoe_router_q4_term(acc, (wv[j] >> (4 * i)) & 0xFu, s[j], b[j], xv[i]);
        }
        acc = nmoe_wave_sum_tree(acc);
        if (lane == 0) logits[(size_t)t * num_experts + e] = acc;
    }
}

/* ------------------------------------------------ logits of many tokens */

/* The same logits, bit for bit, on the fp32 matrix instructions.  A K-deep
 * fp32 MFMA is K fused multiply-adds one after the other, each rounded
 * (v_mfma_f32_16x16x4_f32 in k order; checked on the device against fmaf,
 * subnormals included), so a lane's chain of 32 fmas (nmoe_router_row_bf16)
 * becomes eight MFMAs of a 16-token x 16-expert tile, and the tree over the
 * 64 lanes' chains is added tile by tile: wavefront w of the block owns
 * chains 8 w .. 8 w + 7 and adds them as the tree does, the eight
 * wavefronts' sums meet in LDS and the last three levels follow.
 *
 * The q4 router's term acc + fma(q, s x, b x) rounds each term before it is
 * added, so it needs products of their own: v_mfma_f32_16x16x1_f32 (four
 * independent 16 x 16 products of one k each) gives b x and s x for four
 * columns at once.  bf16 x: s x is exact (16 significant bits) unless it is
 * subnormal or overflows, so fma(q, s x, b x) = fma(q s, x, b x) is a second
 * MFMA on top of b x, and only the add is left to the vector ALU.  fp32 x,
 * and a bf16 chain that holds an x or s so small or so large that s x or q s
 * may be subnormal or overflow: s x and b x by MFMA, fma and add by the
 * vector ALU.
 *
 * Operands: lane l (row r = l % 16, kb = l / 16) loads columns 8 L .. 8 L + 7
 * of segment kb (512 columns a segment) of its row for chain L; a 4 x 4
 * transpose over the wavefront's four rows of lanes (v_permlane32_swap,
 * v_permlane16_swap) turns four elements of four segments into the operand
 * of each segment, lane kb holding element kb. */

typedef __attribute__((ext_vector_type(4))) float nmoe_rt_f32x4;
typedef __attribute__((ext_vector_type(16))) float nmoe_rt_f32x16;
typedef __attribute__((ext_vector_type(2))) uint16_t nmoe_rt_u16x2;

/* Registers v[0..3] (elements) over the lane rows 0..3 (segments) become
 * registers (segments) over lane rows (elements). */
__device__ __forceinline__ void nmoe_rt_transpose4(float v[4]) {
    uint32_t a[4];
#pragma unroll
    for (int i = 0; i < 4; i++) a[i] = __float_as_uint(v[i]);
    auto p = __builtin_amdgcn_permlane32_swap(a[0], a[2], false, false);
    auto q = __builtin_amdgcn_permlane32_swap(a[1], a[3], false, false);
    auto r = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
    auto s = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
    v[0] = __uint_as_float(r[0]);
    v[1] = __uint_as_float(r[1]);
    v[2] = __uint_as_float(s[0]);
    v[3] = __uint_as_float(s[1]);
}

/* A 16-row block's raw loads of one chain, and the eight operands made of
 * them: o[h][j] = element 4 h + kb of segment j. */
template <typename T>
struct nmoe_rt_raw {
    uint4 v[sizeof(T) / 2];
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t L) {
#pragma unroll
        for (int i = 0; i < (int)sizeof(T) / 2; i++)
            v[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff + 16 * i, (int)(8 * sizeof(T) * L), 0));
    }
    __device__ __forceinline__ void operands(float o[2][4]) const {
        float f[8];
        if constexpr (sizeof(T) == 2) {
            nmoe_unpack_bf16x8(v[0], f);
        } else {
            const uint32_t w[8] = {v[0].x, v[0].y, v[0].z, v[0].w, v[1].x, v[1].y, v[1].z, v[1].w};
#pragma unroll
            for (int i = 0; i < 8; i++) f[i] = __uint_as_float(w[i]);
        }
#pragma unroll
        for (int h = 0; h < 2; h++) {
#pragma unroll
            for (int e = 0; e < 4; e++) o[h][e] = f[4 * h + e];
            nmoe_rt_transpose4(o[h]);
        }
    }
};

/* MT x NT tiles of 16 tokens x 16 experts a block of eight wavefronts.
 * Bound: bf16 router, the fp32 MFMA rate (128 fmas a clock a CU: 28 us for
 * 4,096 tokens, matrix cores busy 41 % of the launch with fp32 x, 46 % with
 * bf16 x) and the lines of w and x (a lane reads 32 or 64 bytes of a row at a
 * time; one chain at a time, 16 or 32, took 63 against 51 us; each die reads
 * all of x, 328 MB of 34 in all with fp32 x); q4 router, fp32 MFMAs and vector
 * instructions, which do not overlap on this part (the counter of cycles with
 * both is 0; together they take 96 % of the launch's cycles with fp32 x, 93 %
 * with bf16 x; 2 MFMAs and 16 fma + 16 add a four-column step with fp32 x:
 * 192 clocks of the 220 measured).  4,096 tokens, one-row-a-wavefront kernels
 * against this (us): bf16 router 292 -> 61 (fp32 x), 166 -> 51 (bf16 x); q4
 * router 301 -> 202, 227 -> 145. */
template <bool Q4, typename XT, int MT, int NT>
__global__ void __launch_bounds__(512) nmoe_router_mm_kernel(const void *__restrict__ w, const uint16_t *__restrict__ sc,
                                                             const uint16_t *__restrict__ bi, const XT *__restrict__ x,
                                                             int ntok, int num_experts, float *__restrict__ logits) {
    constexpr int GPR = NMOE_HIDDEN / NMOE_GROUP;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = lane & 15, kb = lane >> 4;
    const int t0 = 16 * MT * (int)blockIdx.y, e0 = 16 * NT * (int)blockIdx.x;
    const __amdgpu_buffer_rsrc_t xr = nmoe_buffer(x), wr = nmoe_buffer(w);
    uint32_t xoff[MT], woff[NT]; /* bytes; rows past the end read the last one and are not stored */
#pragma unroll
    for (int m = 0; m < MT; m++) xoff[m] = (uint32_t)(min(t0 + 16 * m + r, ntok - 1) * NMOE_HIDDEN + 512 * kb) * (uint32_t)sizeof(XT);
#pragma unroll
    for (int n = 0; n < NT; n++)
        woff[n] = (uint32_t)(min(e0 + 16 * n + r, num_experts - 1) * NMOE_HIDDEN + 512 * kb) * 2u / (Q4 ? 4u : 1u);
    float s[NT][4], b[NT][4]; /* q4: a wavefront's chains are one group of each segment */
    if constexpr (Q4) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int g = min(e0 + 16 * n + r, num_experts - 1) * GPR + 8 * j + wave;
                s[n][j] = nmoe_bf16f(sc[g]);
                b[n][j] = nmoe_bf16f(bi[g]);
            }
    }
    /* q4, bf16 x: whether the lane holds an s outside 2^-63 .. 1 (0 apart) */
    bool sout = false;
    if constexpr (Q4 && sizeof(XT) == 2) {
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t a = __float_as_uint(s[n][j]) & 0x7fffffffu;
                sout = sout || a - 1u < ((127u - 63u) << 23) - 1u || a > (127u << 23);
            }
    }
    /* the raw operands of two chains, loaded together (a row's 32 or 64
     * consecutive bytes) while the pair before them multiplies */
    nmoe_rt_raw<XT> xv[2][MT];
    nmoe_rt_raw<uint16_t> wv[2][NT];
    uint32_t wq[2][NT];
    auto load = [&](int L) {
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int c = 0; c < 2; c++) xv[c][m].load(xr, xoff[m], (uint32_t)(L + c));
#pragma unroll
        for (int n = 0; n < NT; n++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                if constexpr (Q4)
                    wq[c][n] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(wr, (int)woff[n], 4 * (L + c), 0);
                else
                    wv[c][n].load(wr, woff[n], (uint32_t)(L + c));
            }
    };
    nmoe_rt_f32x4 st[2][MT][NT], d[2][MT][NT];
    const nmoe_rt_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    load(8 * wave);
#pragma unroll 1
    for (int p = 0; p < 4; p++) {
#pragma unroll
        for (int c = 0; c < 2; c++) {
            float xo[MT][2][4];
#pragma unroll
            for (int m = 0; m < MT; m++) xv[c][m].operands(xo[m]);
#pragma unroll
            for (int m = 0; m < MT; m++)
#pragma unroll
                for (int n = 0; n < NT; n++) d[c][m][n] = zero;
            if constexpr (!Q4) {
                float wo[NT][2][4];
#pragma unroll
                for (int n = 0; n < NT; n++) wv[c][n].operands(wo[n]);
                if (c == 1) load(8 * wave + 2 * min(p + 1, 3));
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int h = 0; h < 2; h++)
#pragma unroll
                        for (int m = 0; m < MT; m++)
#pragma unroll
                            for (int n = 0; n < NT; n++)
                                d[c][m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(xo[m][h][j], wo[n][h][j], d[c][m][n], 0, 0, 0);
            } else {
                uint32_t wj[NT][4]; /* each segment's word in every lane row */
#pragma unroll
                for (int n = 0; n < NT; n++) {
                    auto v = __builtin_amdgcn_permlane32_swap(wq[c][n], wq[c][n], false, false);
                    auto q0 = __builtin_amdgcn_permlane16_swap(v[0], v[0], false, false);
                    auto q1 = __builtin_amdgcn_permlane16_swap(v[1], v[1], false, false);
                    wj[n][0] = q0[0];
                    wj[n][1] = q0[1];
                    wj[n][2] = q1[0];
                    wj[n][3] = q1[1];
                }
                /* s x and q s exact for every s and x of the chain: no nonzero |x|
                 * below 2^-70 and no nonzero |s| below 2^-63 (the lowest bit of
                 * s x is then 2^-147 or more, the subnormals' 2^-149), no |s|
                 * above 1 (no finite s x overflows) */
                bool exact = false;
                if constexpr (sizeof(XT) == 2) {
                    nmoe_rt_u16x2 xmin = {0xffff, 0xffff};
#pragma unroll
                    for (int m = 0; m < MT; m++) {
                        const uint32_t u[4] = {xv[c][m].v[0].x, xv[c][m].v[0].y, xv[c][m].v[0].z, xv[c][m].v[0].w};
#pragma unroll
                        for (int i = 0; i < 4; i++) {
                            const nmoe_rt_u16x2 one = {1, 1};
                            xmin = __builtin_elementwise_min(xmin, __builtin_bit_cast(nmoe_rt_u16x2, u[i] & 0x7fff7fffu) - one);
                        }
                    }
                    exact = __ballot(min(xmin.x, xmin.y) < ((127 - 70) << 7) - 1 || sout) == 0;
                }
                if (c == 1) load(8 * wave + 2 * min(p + 1, 3));
                const nmoe_rt_f32x16 z16 = {};
                auto steps = [&](auto exact_c) {
#pragma unroll
                    for (int j = 0; j < 4; j++)
#pragma unroll
                        for (int h = 0; h < 2; h++)
#pragma unroll
                            for (int n = 0; n < NT; n++) {
                                if constexpr (decltype(exact_c)::value) {
                                    const float qs = (float)((wj[n][j] >> (16 * h + 4 * kb)) & 15u) * s[n][j];
#pragma unroll
                                    for (int m = 0; m < MT; m++) {
                                        nmoe_rt_f32x16 t = __builtin_amdgcn_mfma_f32_16x16x1f32(xo[m][h][j], b[n][j], z16, 0, 0, 0);
                                        t = __builtin_amdgcn_mfma_f32_16x16x1f32(xo[m][h][j], qs, t, 0, 0, 0);
#pragma unroll
                                        for (int k = 0; k < 4; k++)
#pragma unroll
                                            for (int i = 0; i < 4; i++) d[c][m][n][i] = d[c][m][n][i] + t[4 * k + i];
                                    }
                                } else {
                                    const uint32_t lo = (wj[n][j] >> (16 * h)) & 0x0F0Fu, hi = (wj[n][j] >> (16 * h + 4)) & 0x0F0Fu;
                                    const float q[4] = {(float)(lo & 0xFFu), (float)(hi & 0xFFu), (float)(lo >> 8), (float)(hi >> 8)};
#pragma unroll
                                    for (int m = 0; m < MT; m++) {
                                        const nmoe_rt_f32x16 sx = __builtin_amdgcn_mfma_f32_16x16x1f32(xo[m][h][j], s[n][j], z16, 0, 0, 0);
                                        const nmoe_rt_f32x16 bx = __builtin_amdgcn_mfma_f32_16x16x1f32(xo[m][h][j], b[n][j], z16, 0, 0, 0);
#pragma unroll
                                        for (int k = 0; k < 4; k++)
#pragma unroll
                                            for (int i = 0; i < 4; i++)
                                                d[c][m][n][i] = d[c][m][n][i] + __builtin_fmaf(q[k], sx[4 * k + i], bx[4 * k + i]);
                                    }
                                }
                            }
                };
                if (exact)
                    steps(std::true_type{});
                else
                    steps(std::false_type{});
            }
        }
        /* the tree over the wavefront's chains: 0 + 1, 2 + 3, .. */
#pragma unroll
        for (int m = 0; m < MT; m++)
#pragma unroll
            for (int n = 0; n < NT; n++) {
                nmoe_rt_f32x4 v = d[0][m][n] + d[1][m][n];
                if (!(p & 1)) {
                    st[0][m][n] = v;
                } else {
                    v = st[0][m][n] + v;
                    if (p == 1)
                        st[1][m][n] = v;
                    else
                        d[0][m][n] = st[1][m][n] + v;
                }
            }
    }
    __shared__ nmoe_rt_f32x4 red[8 * MT * NT * 64];
#pragma unroll
    for (int m = 0; m < MT; m++)
#pragma unroll
        for (int n = 0; n < NT; n++) red[(wave * MT * NT + m * NT + n) * 64 + lane] = d[0][m][n];
    __syncthreads();
    for (int u = wave; u < MT * NT; u += 8) {
        nmoe_rt_f32x4 p[8];
#pragma unroll
        for (int i = 0; i < 8; i++) p[i] = red[(i * MT * NT + u) * 64 + lane];
        const nmoe_rt_f32x4 v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
        const int e = e0 + 16 * (u % NT) + r;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int t = t0 + 16 * (u / NT) + 4 * kb + i;
            if (t < ntok && e < num_experts) logits[(size_t)t * num_experts + e] = v[i];
        }
    }
}

template <bool Q4, typename XT, int MT, int NT>
static void nmoe_router_mm_launch(const nmoe_hip_router *router, const void *x, int ntok, float *logits, hipStream_t s) {
    const void *w = Q4 ? (const void *)router->w_q4 : (const void *)router->w_bf16;
    const int ne = router->num_experts;
    hipLaunchKernelGGL((nmoe_router_mm_kernel<Q4, XT, MT, NT>),
                       dim3((ne + 16 * NT - 1) / (16 * NT), (ntok + 16 * MT - 1) / (16 * MT)), dim3(512), 0, s, w,
                       router->scales, router->biases, (const XT *)x, ntok, ne, logits);
}

/* Whether the matrix form runs.  It takes the time of its rounds of 16 x 16
 * tiles over the 256 CUs, whatever they hold; the one-row-a-wavefront kernels
 * that of ntok (ne + c) terms, c for the loads of x.  256 experts, us, one row
 * a wavefront against the matrix form, either side of each line:
 *   bf16 router, fp32 x   8.3 / 8.1 at 88 tokens, 8.9 / 8.1 at 96
 *   bf16 router, bf16 x   5.9 / 6.2 at 96, 6.3 / 6.25 at 104; second round
 *                         12.6 / 10.4 at 257
 *   q4 router, fp32 x     17.4 / 17.6 at 200, 18.1 / 17.6 at 208; second
 *                         round 28.4 / 29.7 at 352, 30.7 / 29.7 at 384; third
 *                         42.0 / 41.5 at 513
 *   q4 router, bf16 x     12.5 / 13.0 at 192, 13.6 / 13.1 at 200; second
 *                         21.8 / 22.2 at 352, 22.7 / 22.3 at 368; third 30.0 /
 *                         30.4 at 513, 34.8 / 30.8 at 600
 * and fewer experts, from which c: 64 experts, fp32 x, 7.8 / 8.2 at 300 tokens
 * (bf16 router), 13.1 / 17.4 at 512 and 24.3 / 17.6 at 1,000 (q4); 16 experts,
 * 5.0 / 8.2 at 512 and 12.2 / 8.3 at 1,000, 12.6 / 17.4 at 1,000 and 23.0 /
 * 17.6 at 2,048; 2 experts, bf16 router, 4.0 / 7.4 at 2,048. */
static bool nmoe_router_mm_pays(bool q4, bool bf, int ntok, int ne) {
    if (ne < 4) return false;
    const int c = q4 ? (bf ? 11 : 20) : (bf ? 8 : 18);
    const long tokens = (long)ntok * (ne + c) / (NMOE_EXPERTS + c); /* of 256 experts */
    if (!q4) return tokens >= (bf ? 104 : 96);
    const long tiles = (long)((ne + 15) / 16) * ((ntok + 15) / 16);
    return tokens >= (tiles <= 256 ? (bf ? 200 : 208) : (bf ? 368 : 384));
}

template <typename XT>
static void nmoe_router_mm(const nmoe_hip_router *router, const void *x, int ntok, float *logits, hipStream_t s) {
    /* the smallest tile whose grid is one round of the 256 CUs (or, with
     * rows of x few enough, two): a larger tile reads each row of w and x less
     * often, a smaller one leaves no CU idle.  bf16 router, fp32 x, 256
     * experts, 16x16 / 32x32 / 32x64 tiles (us): 8.6 / 15 / 25 at 251 tokens,
     * 17.2 / 17.6 at 512, 20.8 / 17.7 at 513, 34 / 23 / 28 at 1,000, 125 / 80
     * / 61 at 4,096; bf16 x 12.0 / 14.0 at 272, 13.0 / 14.1 at 512; 128
     * experts 20.5 / 17.9 at 1,000; 64 experts, 32x32 / 32x64, 18.7 / 25.2 at
     * 2,048 and 31.3 / 27.3 at 4,096.  The q4 router is bound by its vector
     * instructions and keeps the smallest (the larger ones spill). */
    const int ne = router->num_experts;
    auto tiles = [&](int rows, int cols) { return (long)((ntok + rows - 1) / rows) * ((ne + cols - 1) / cols); };
    if (router->kind == NMOE_HIP_ROUTER_Q4)
        nmoe_router_mm_launch<true, XT, 1, 1>(router, x, ntok, logits, s);
    else if (ntok <= 512 || tiles(16, 16) <= 256)
        nmoe_router_mm_launch<false, XT, 1, 1>(router, x, ntok, logits, s);
    else if (ntok <= 2048 && tiles(32, 32) <= 256)
        nmoe_router_mm_launch<false, XT, 2, 2>(router, x, ntok, logits, s);
    else
        nmoe_router_mm_launch<false, XT, 2, 4>(router, x, ntok, logits, s);
}

/* ------------------------------------------------------------ routing */

__global__ void __launch_bounds__(64) nmoe_topk_kernel(const float *__restrict__ logits, int ntok, int num_experts,
                                                       int k, uint32_t *__restrict__ idx, float *__restrict__ w,
                                                       float *__restrict__ probs) {
    __shared__ float scratch[NMOE_EXPERTS];
    int t = blockIdx.x;
    if (t >= ntok) return;
    uint32_t si[NMOE_MAX_K];
    float sw[NMOE_MAX_K];
    nmoe_wave_route(logits + (size_t)t * num_experts, num_experts, k, scratch, nmoe_exp2_tab, si, sw,
                    probs != NULL ? probs + (size_t)t * num_experts : NULL);
    int lane = threadIdx.x;
    if (lane < NMOE_MAX_K) {
        uint32_t vi = 0;
        float vw = 0.0f;
#pragma unroll
        for (int s = 0; s < NMOE_MAX_K; s++)
            if (s == lane) {
                vi = si[s];
                vw = sw[s];
            }
        idx[(size_t)t * NMOE_MAX_K + lane] = vi;
        w[(size_t)t * NMOE_MAX_K + lane] = vw;
    }
}

/* ------------------------------------------------------- entry points */

int nmoe_check_router(nmoe_hip_ctx *ctx, const nmoe_hip_router *r) {
    if (r == NULL) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "NULL router");
    if (r->num_experts < 1 || r->num_experts > NMOE_EXPERTS)
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "num_experts %d outside 1..256", r->num_experts);
    if (r->kind == NMOE_HIP_ROUTER_BF16) {
        if (r->w_bf16 == NULL || !nmoe_aligned(r->w_bf16, 16))
            return nmoe_fail(ctx, NMOE_HIP_EINVAL, "bf16 router weights NULL or not 16-byte aligned");
    } else if (r->kind == NMOE_HIP_ROUTER_Q4) {
        if (r->w_q4 == NULL || r->scales == NULL || r->biases == NULL || !nmoe_aligned(r->w_q4, 4))
            return nmoe_fail(ctx, NMOE_HIP_EINVAL, "q4 router tensors NULL or misaligned");
    } else {
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "unknown router kind %d", r->kind);
    }
    return NMOE_HIP_OK;
}

int nmoe_check_x(nmoe_hip_ctx *ctx, const void *x, int x_dtype, int ntok) {
    if (x == NULL || !nmoe_aligned(x, 16)) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "x NULL or not 16-byte aligned");
    if (x_dtype != NMOE_HIP_F32 && x_dtype != NMOE_HIP_BF16)
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "x_dtype must be NMOE_HIP_F32 or NMOE_HIP_BF16");
    if (ntok < 1 || ntok > ctx->max_tokens)
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "ntok %d outside 1..%d (max_tokens at create)", ntok, ctx->max_tokens);
    return NMOE_HIP_OK;
}

/* The router launch with its arguments already checked. */
extern "C" hipError_t nmoe_router_logits_launch(const nmoe_hip_router *router, const void *x, int x_dtype, int ntok,
                                               float *logits, hipStream_t s) {
    if (nmoe_router_mm_pays(router->kind == NMOE_HIP_ROUTER_Q4, x_dtype == NMOE_HIP_BF16, ntok, router->num_experts)) {
        if (x_dtype == NMOE_HIP_BF16)
            nmoe_router_mm<uint16_t>(router, x, ntok, logits, s);
        else
            nmoe_router_mm<float>(router, x, ntok, logits, s);
        return hipGetLastError();
    }
    int tpb = ntok <= 4 ? ntok : 4;
    dim3 grid(router->num_experts, (ntok + tpb - 1) / tpb);
    if (router->kind == NMOE_HIP_ROUTER_BF16) {
        if (x_dtype == NMOE_HIP_BF16)
            hipLaunchKernelGGL(nmoe_router_bf16_kernel<uint16_t>, grid, dim3(64), 0, s, router->w_bf16,
                               (const uint16_t *)x, ntok, router->num_experts, tpb, logits);
        else
            hipLaunchKernelGGL(nmoe_router_bf16_kernel<float>, grid, dim3(64), 0, s, router->w_bf16,
                               (const float *)x, ntok, router->num_experts, tpb, logits);
    } else {
        if (x_dtype == NMOE_HIP_BF16)
            hipLaunchKernelGGL(nmoe_router_q4_kernel<uint16_t>, grid, dim3(64), 0, s, router->w_q4, router->scales,
                               router->biases, (const uint16_t *)x, ntok, router->num_experts, tpb, logits);
        else
            hipLaunchKernelGGL(nmoe_router_q4_kernel<float>, grid, dim3(64), 0, s, router->w_q4, router->scales,
                               router->biases, (const float *)x, ntok, router->num_experts, tpb, logits);
    }
    return hipGetLastError();
}

extern "C" hipError_t nmoe_topk_launch(const float *logits, int ntok, int num_experts, int k, uint32_t *idx, float *w,
                                      float *probs, hipStream_t s) {
    hipLaunchKernelGGL(nmoe_topk_kernel, dim3(ntok), dim3(64), 0, s, logits, ntok, num_experts, k, idx, w, probs);
    return hipGetLastError();
}

extern "C" int nmoe_moe_router_logits(nmoe_hip_ctx *ctx, const nmoe_hip_router *router, const void *x, int x_dtype,
                                      int ntok, float *logits, void *stream) {
    if (ctx == NULL) return NMOE_HIP_EINVAL;
    int rc = nmoe_check_router(ctx, router);
    if (rc == NMOE_HIP_OK) rc = nmoe_check_x(ctx, x, x_dtype, ntok);
    if (rc != NMOE_HIP_OK) return rc;
    if (logits == NULL) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "NULL logits");
    NMOE_HIP_TRY(ctx, nmoe_router_logits_launch(router, x, x_dtype, ntok, logits, nmoe_stream_of(ctx, stream)));
    return NMOE_HIP_OK;
}

extern "C" int nmoe_moe_topk(nmoe_hip_ctx *ctx, const float *logits, int ntok, int num_experts, int k, uint32_t *idx,
                             float *w, float *probs, void *stream) {
    if (ctx == NULL) return NMOE_HIP_EINVAL;
    if (logits == NULL || idx == NULL || w == NULL) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "NULL argument");
    if (k < 1 || k > NMOE_MAX_K) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "k=%d outside 1..8", k);
    if (num_experts < 1 || num_experts > NMOE_EXPERTS)
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "num_experts %d outside 1..256", num_experts);
    if (ntok < 1) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "ntok must be >= 1");
    NMOE_HIP_TRY(ctx, nmoe_topk_launch(logits, ntok, num_experts, k, idx, w, probs, nmoe_stream_of(ctx, stream)));
    return NMOE_HIP_OK;
}

extern "C" int nmoe_moe_route(nmoe_hip_ctx *ctx, const nmoe_hip_router *router, const void *x, int x_dtype, int ntok,
                              int k, uint32_t *idx, float *w, float *logits, void *stream) {
    if (ctx == NULL) return NMOE_HIP_EINVAL;
    if (k < 1 || k > NMOE_MAX_K) return nmoe_fail(ctx, NMOE_HIP_EINVAL, "k=%d outside 1..8", k);
    int rc = nmoe_check_x(ctx, x, x_dtype, ntok);
    if (rc != NMOE_HIP_OK) return rc;
    float *lg = logits != NULL ? logits : ctx->logits;
    rc = nmoe_moe_router_logits(ctx, router, x, x_dtype, ntok, lg, stream);
    if (rc != NMOE_HIP_OK) return rc;
    return nmoe_moe_topk(ctx, lg, ntok, router->num_experts, k, idx, w, NULL, stream);
}
