/*
 * shared.hip -- the shared expert of a Qwen3.6 MoE layer on gfx950.
 *
 * The reference evaluates it in two kernels:
 *   - nmoe_route_shared_q4 (metal/kernels.metal:384-514): rows 0-511 give
 *     the shared activation SiLU(gate.x) * (up.x), rows 512-767 the router
 *     logits, row 768 the shared-expert gate score;
 *   - the shared down inside nmoe_expert_down_combine_q4 (:1520-1537).
 * Here the shared expert has its own launches (two for few tokens, three on
 * the matrix cores for many); the router logits stay with the router kernels.  Weights are the model's q4 tensors as stored
 * (w = q*scale + bias, math.m:206-234), each row reduced by one wavefront.
 */
#include "nmoe_device.h"

/* Wavefront w of block b reduces row 4b + w of gate and of up (rows
 * 0..511); block 128 wavefront 0 reduces the score row.  Lane L owns the
 * words L, L+64, L+128, L+192 of a 256-word row (columns 8 word .. +7) and
 * accumulates acc + fma(q, s*x, b*x) per column, the reference's form for
 * these rows (kernels.metal:444-460, 500-508); lanes combined by the pairwise
 * tree.  The row's codes and scales stay in registers over the block's
 * tokens. */
template <typename XT>
__global__ void __launch_bounds__(256) nmoe_shared_gateup_kernel(
    const uint32_t *__restrict__ gw, const uint16_t *__restrict__ gs, const uint16_t *__restrict__ gb,
    const uint32_t *__restrict__ uw, const uint16_t *__restrict__ us, const uint16_t *__restrict__ ub,
    const uint32_t *__restrict__ sw, const uint16_t *__restrict__ ss, const uint16_t *__restrict__ sb,
    const XT *__restrict__ x, int ntok, int tok_per_block, float *__restrict__ act, float *__restrict__ graw) {
    constexpr int WPR = NMOE_HIDDEN / 8, GPR = NMOE_HIDDEN / NMOE_GROUP;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int row = 4 * blockIdx.x + wave;
    const bool score = row >= NMOE_INTER;
    if (score && row != NMOE_INTER) return;
    const uint32_t *w0 = score ? sw : gw + (size_t)row * WPR;
    const uint16_t *s0 = score ? ss : gs + (size_t)row * GPR, *b0 = score ? sb : gb + (size_t)row * GPR;
    uint32_t wa[4], wb[4];
    float sa[4], ba[4], sbv[4], bbv[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = lane + 64 * j;
        wa[j] = w0[c];
        sa[j] = nmoe_bf16f(s0[c / 8]);
        ba[j] = nmoe_bf16f(b0[c / 8]);
        if (!score) {
            wb[j] = uw[(size_t)row * WPR + c];
            sbv[j] = nmoe_bf16f(us[(size_t)row * GPR + c / 8]);
            bbv[j] = nmoe_bf16f(ub[(size_t)row * GPR + c / 8]);
        }
    }
    const int t0 = blockIdx.y * tok_per_block, t1 = min(ntok, t0 + tok_per_block);
    for (int t = t0; t < t1; t++) {
        const XT *xt = x + (size_t)t * NMOE_HIDDEN;
        float ga = 0.0f, ua = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float xv[8];
            nmoe_load_cols<XT>(xt, (lane + 64 * j) * 8, 8, xv);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                ga = nmoe_router_q4_term(ga, (wa[j] >> (4 * i)) & 0xFu, sa[j], ba[j], xv[i]);
                if (!score) ua = nmoe_router_q4_term(ua, (wb[j] >> (4 * i)) & 0xFu, sbv[j], bbv[j], xv[i]);
            }
        }
        ga = nmoe_wave_sum_tree(ga);
        if (score) {
            if (lane == 0) graw[t] = ga;
        } else {
            ua = nmoe_wave_sum_tree(ua);
            if (lane == 0) act[(size_t)t * NMOE_INTER + row] = nmoe_silu_dev(ga) * ua;
        }
    }
}

/* Wavefront w of block b reduces row 4b + w (of 2048) of the shared down
 * against act: lane L owns word L of the 64-word row (columns 8L..8L+7) and
 * accumulates fma(q, s, b) * x per column, the reference's form for this
 * matrix (kernels.metal:1533), as one fma. */
__global__ void __launch_bounds__(256) nmoe_shared_down_kernel(const uint32_t *__restrict__ dw,
                                                               const uint16_t *__restrict__ ds,
                                                               const uint16_t *__restrict__ db,
                                                               const float *__restrict__ act, int ntok,
                                                               int tok_per_block, float *__restrict__ out) {
    constexpr int WPR = NMOE_INTER / 8, GPR = NMOE_INTER / NMOE_GROUP;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int row = 4 * blockIdx.x + wave;
    const uint32_t wv = dw[(size_t)row * WPR + lane];
    const float s = nmoe_bf16f(ds[(size_t)row * GPR + lane / 8]), b = nmoe_bf16f(db[(size_t)row * GPR + lane / 8]);
    const int t0 = blockIdx.y * tok_per_block, t1 = min(ntok, t0 + tok_per_block);
    for (int t = t0; t < t1; t++) {
        float xv[8];
        nmoe_load_cols<float>(act + (size_t)t * NMOE_INTER, 8 * lane, 8, xv);
        float acc = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) acc = __builtin_fmaf(__builtin_fmaf((float)((wv >> (4 * i)) & 0xFu), s, b), xv[i], acc);
        acc = nmoe_wave_sum_tree(acc);
        if (lane == 0) out[(size_t)t * NMOE_HIDDEN + row] = acc;
    }
}

/* ------------------------------------------------ many tokens: matrix cores */

/* From NMOE_SHARED_MM_MIN tokens on, three launches:
 *
 *   prep  the codes of gate, up and down as bf16(q - 8) (exact) in matrix-core
 *         operand order, scales and biases as aligned copies, x as PL bf16
 *         planes whose sum is x exactly (one for bf16 x; three for fp32 x, 8
 *         significant bits each) in operand order, the sums of x over each
 *         64-column group as three bf16 parts, and the score row (in the
 *         per-token kernel's order, so the same bits).
 *   gate/up  act = SiLU(g) * u, stored as three bf16 planes (exact) in the
 *         down product's operand order, with the sums of 16 columns.
 *   down  shared_out.
 *
 * With c = b + 8 s, w = s (q - 8) + c and
 *     sum_k w_k x_k = sum_g s_g P_g + sum_g c_g xs_g,  P_g = sum (q_k - 8) x_k:
 * every product entering an MFMA is exact and P_g, the scaled sum and the
 * correction are fp32, as the per-token kernels' sums are (measured against
 * 64 bits: no larger an error).  The codes are centred (not 128 + q as in
 * the routed experts' GEMMs) so that nothing cancels.
 *
 * Operand order (v_mfma_f32_16x16x32_bf16): lane l holds row l % 16 and k =
 * 8 (l / 16) .. + 7 of a 32-deep slice, so a matrix is stored as [16-row
 * block][slice][lane][8] and an operand is one contiguous 1 KB load of a
 * wavefront. */

typedef __attribute__((ext_vector_type(8))) __bf16 nmoe_sh_bf16x8;
typedef __attribute__((ext_vector_type(4))) float nmoe_sh_f32x4;

#define NMOE_SH_GU_SL (NMOE_HIDDEN / 32) /* slices of a gate/up row: 64 */
#define NMOE_SH_DN_SL (NMOE_INTER / 32)  /* slices of a down row: 16 */
#define NMOE_SH_GU_G (NMOE_HIDDEN / NMOE_GROUP)
#define NMOE_SH_DN_G (NMOE_INTER / NMOE_GROUP)

/* The launches' scratch (device): nmoe_sh_layout. */
struct nmoe_sh_ws {
    uint4 *wgu;     /* [64 row blocks: gate 0..31, up 32..63][64][64] */
    uint4 *wdn;     /* [128][16][64] */
    uint16_t *sgu;  /* [1024][32] scales, then c as three bf16 parts [3][1024][32] */
    uint16_t *sdn;  /* [2048][8] scales, then [2048][8] biases */
    uint4 *xp;      /* [PL][tb][64][64] */
    uint4 *xs3;     /* [3][tb][64] */
    uint4 *ap;      /* [3][tb][16][64] */
    float *asq;     /* [tb * 16][32] sums of 16 act columns */
};

__device__ __forceinline__ nmoe_sh_f32x4 nmoe_sh_mfma(uint4 a, uint4 b, nmoe_sh_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(nmoe_sh_bf16x8, a),
                                                   __builtin_bit_cast(nmoe_sh_bf16x8, b), c, 0, 0, 0);
}

/* A 16-byte load from a buffer resource. */
__device__ __forceinline__ uint4 nmoe_sh_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, 0));
}

/* v as three bf16 whose sum is v (truncations: 8 + 8 + 8 significant bits). */
__device__ __forceinline__ void nmoe_sh_split3(float v, uint32_t p[3]) {
    const uint32_t h = __float_as_uint(v) & 0xffff0000u;
    const float r = v - __uint_as_float(h);
    const uint32_t m = __float_as_uint(r) & 0xffff0000u;
    const float l = r - __uint_as_float(m);
    p[0] = h >> 16;
    p[1] = m >> 16;
    p[2] = __float_as_uint(l) >> 16;
}

/* Blocks 0 .. NMOE_SH_WB - 1: the codes, one wavefront a (row block, 8
 * slices); the next NMOE_SH_SB: scales and biases, 8 a thread; then four
 * blocks for each 16 tokens: planes and group sums, a wavefront 4 slices;
 * then one wavefront a token: the score row.  b0: the first of them this
 * launch runs (the weights' are done once for all chunks of a call). */
#define NMOE_SH_WU ((1024 / 16) * (NMOE_SH_GU_SL / 8) + (NMOE_HIDDEN / 16) * (NMOE_SH_DN_SL / 8))
#define NMOE_SH_WB (NMOE_SH_WU / 4)
#define NMOE_SH_SB ((1024 * NMOE_SH_GU_G + 2 * NMOE_HIDDEN * NMOE_SH_DN_G) / 8 / 256)
template <typename XT>
__global__ void __launch_bounds__(256) nmoe_shared_prep_kernel(nmoe_hip_shared_expert se, nmoe_sh_ws ws, const XT *x,
                                                               int ntok, int ntb, int b0, float *graw) {
    constexpr int PL = sizeof(XT) == 2 ? 1 : 3;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, b = blockIdx.x + b0;
    if (b < NMOE_SH_WB) {
        constexpr int GUU = (1024 / 16) * (NMOE_SH_GU_SL / 8);
        const int u = 4 * b + wave;
        const bool gu = u < GUU;
        const int rb = gu ? u / (NMOE_SH_GU_SL / 8) : (u - GUU) / (NMOE_SH_DN_SL / 8);
        const int s0 = 8 * (gu ? u % (NMOE_SH_GU_SL / 8) : (u - GUU) % (NMOE_SH_DN_SL / 8));
        const int nsl = gu ? NMOE_SH_GU_SL : NMOE_SH_DN_SL;
        const int row = 16 * (gu ? rb & 31 : rb) + (lane & 15);
        const uint32_t *src = (gu ? (rb < 32 ? se.gate.w : se.up.w) : se.down.w) + (size_t)row * (4 * nsl) + (lane >> 4);
        uint4 *dst = (gu ? ws.wgu : ws.wdn) + ((size_t)rb * nsl + s0) * 64 + lane;
        uint32_t w[8];
#pragma unroll
        for (int j = 0; j < 8; j++) w[j] = src[4 * (s0 + j)];
#pragma unroll
        for (int j = 0; j < 8; j++) {
            uint32_t o[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float f0 = (float)((w[j] >> (8 * i)) & 15u) - 8.0f, f1 = (float)((w[j] >> (8 * i + 4)) & 15u) - 8.0f;
                o[i] = (__float_as_uint(f0) >> 16) | (__float_as_uint(f1) & 0xffff0000u);
            }
            dst[64 * j] = make_uint4(o[0], o[1], o[2], o[3]);
        }
        return;
    }
    if (b < NMOE_SH_WB + NMOE_SH_SB) {
        const int i = 8 * (256 * (b - NMOE_SH_WB) + (int)threadIdx.x); /* first of 8 values of one tensor */
        constexpr int GU = NMOE_INTER * NMOE_SH_GU_G, DN = NMOE_HIDDEN * NMOE_SH_DN_G;
        uint32_t v[4];
        if (i < 2 * GU) { /* gate and up: s, and c = b + 8 s in three parts */
            const nmoe_hip_qtensor &m = i < GU ? se.gate : se.up;
            uint32_t sv[8], c[8][3];
#pragma unroll
            for (int j = 0; j < 8; j++) {
                sv[j] = m.scales[i % GU + j];
                nmoe_sh_split3(__builtin_fmaf(8.0f, nmoe_bf16f(sv[j]), nmoe_bf16f(m.biases[i % GU + j])), c[j]);
            }
#pragma unroll
            for (int p = 0; p < 4; p++) {
#pragma unroll
                for (int j = 0; j < 4; j++)
                    v[j] = p == 0 ? sv[2 * j] | (sv[2 * j + 1] << 16) : c[2 * j][p - 1] | (c[2 * j + 1][p - 1] << 16);
                *(uint4 *)(ws.sgu + p * 2 * GU + i) = make_uint4(v[0], v[1], v[2], v[3]);
            }
        } else if (i < 2 * GU + 2 * DN) {
            const int q = i - 2 * GU;
            const uint16_t *src = (q < DN ? se.down.scales : se.down.biases) + q % DN;
#pragma unroll
            for (int j = 0; j < 4; j++) v[j] = (uint32_t)src[2 * j] | ((uint32_t)src[2 * j + 1] << 16);
            *(uint4 *)(ws.sdn + q) = make_uint4(v[0], v[1], v[2], v[3]);
        }
        return;
    }
    const int u = b - NMOE_SH_WB - NMOE_SH_SB;
    if (u < 4 * ntb) {
        const int tb = u >> 2, s0 = 16 * (u & 3) + 4 * wave;
        const int t = min(16 * tb + (lane & 15), ntok - 1); /* rows past the last token repeat it; never stored */
        const XT *xt = x + (size_t)t * NMOE_HIDDEN + 32 * s0 + 8 * (lane >> 4);
        uint4 *o = ws.xp + ((size_t)tb * NMOE_SH_GU_SL + s0) * 64 + lane;
        const size_t plane = (size_t)ntb * NMOE_SH_GU_SL * 64;
        float v[4][8], sum[2] = {0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < 4; j++) nmoe_load_cols<XT>(xt, 32 * j, 8, v[j]);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            uint32_t p[8][3];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                sum[j >> 1] += v[j][i];
                if (PL == 3)
                    nmoe_sh_split3(v[j][i], p[i]);
                else
                    p[i][0] = __float_as_uint(v[j][i]) >> 16;
            }
#pragma unroll
            for (int pl = 0; pl < PL; pl++)
                o[pl * plane + 64 * j] = make_uint4(p[0][pl] | (p[1][pl] << 16), p[2][pl] | (p[3][pl] << 16),
                                                    p[4][pl] | (p[5][pl] << 16), p[6][pl] | (p[7][pl] << 16));
        }
        uint32_t part[2][3];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            sum[j] += __shfl_xor(sum[j], 16);
            sum[j] += __shfl_xor(sum[j], 32);
            nmoe_sh_split3(sum[j], part[j]);
        }
        /* groups s0 / 2 and s0 / 2 + 1: one word of the operand */
        const int g = s0 >> 1;
        if (lane < 16)
#pragma unroll
            for (int i = 0; i < 3; i++)
                ((uint32_t *)(ws.xs3 + ((size_t)i * ntb + tb) * 64 + 16 * (g >> 3) + lane))[(g & 7) >> 1] =
                    part[0][i] | (part[1][i] << 16);
        return;
    }
    const int t = 4 * (u - 4 * ntb) + wave;
    if (t >= ntok) return;
    float acc = 0.0f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int c = lane + 64 * j;
        const uint32_t w = se.score.w[c];
        const float s = nmoe_bf16f(se.score.scales[c / 8]), bb = nmoe_bf16f(se.score.biases[c / 8]);
        float xv[8];
        nmoe_load_cols<XT>(x + (size_t)t * NMOE_HIDDEN, 8 * c, 8, xv);
#pragma unroll
        for (int i = 0; i < 8; i++) acc = nmoe_router_q4_term(acc, (w >> (4 * i)) & 0xFu, s, bb, xv[i]);
    }
    acc = nmoe_wave_sum_tree(acc);
    if (lane == 0) graw[t] = acc;
}

/* One product: a block owns MB 16-token blocks x 64 weight rows (gate/up: 32
 * gate rows and the up rows of the same columns); its four wavefronts take a
 * quarter of K each and add their sums in LDS, so a chain is 16 (gate/up) or
 * 4 (down) slices long and nothing is shared, or waited for, before the end.
 * Operands go straight from their operand-order copies into registers.
 * Bound: the two operands' way from the L2 (64 x 64 tiles read 16 KB of them
 * for 32 MFMAs), at 2,048 and more tokens (4,096, fp32 x: gate/up's matrix
 * cores busy 35 % of the launch, no unit 57 %); the launches and one chain's
 * latency below.  Measured (three launches, us, fp32 x / bf16 x, against the
 * per-token kernels): 64 tokens 22 / 21 from 32 / 31, 251 tokens 26 / 25 from
 * 107 / 96, 1,000 tokens 41 / 35 from 415 / 367, 4,096 tokens 121 / 94 from
 * 1,662 / 1,473. */
template <int PL, int MB, bool GU>
__global__ void __launch_bounds__(256, 2) nmoe_shared_mm_kernel(nmoe_sh_ws ws, int ntok, int ntb, int mtiles, int swz,
                                                                float *out) {
    constexpr int NSL = GU ? NMOE_SH_GU_SL : NMOE_SH_DN_SL, SL = NSL / 4;
    constexpr int G = NSL / 2;
    static_assert(SL % 4 == 0, "whole pairs of groups");
    constexpr int NT = GU ? 16 : 32; /* 64-row tiles */
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int col = lane & 15, kb = lane >> 4;
    /* swz: each die (block index mod 8) takes every eighth token tile, all
     * its row tiles in turn, so the tile's x stays in that die's L2 */
    const int bi = blockIdx.x;
    const int mt = swz ? (bi >> 3) / NT * 8 + (bi & 7) : bi / NT, n = swz ? (bi >> 3) % NT : bi % NT;
    if (mt >= mtiles) return;
    const int s0 = wave * SL; /* the wavefront's slices */
    int rb[4];
#pragma unroll
    for (int j = 0; j < 4; j++) rb[j] = GU ? (j < 2 ? 2 * n + j : 30 + 2 * n + j) : 4 * n + j;
    /* Loads through raw buffer resources: one scalar offset a tile and slice
     * on top of the lane's 16 bytes, and (as these are intrinsics) they stay
     * where the ring issues them. */
    const __amdgpu_buffer_rsrc_t ar = nmoe_buffer(GU ? ws.xp : ws.ap),
                                 br = nmoe_buffer(GU ? ws.wgu : ws.wdn);
    const uint16_t *sc = GU ? ws.sgu : ws.sdn, *bs = sc + (GU ? 1024 : NMOE_HIDDEN) * G;
    uint32_t aoff[MB][PL], boff[4]; /* bytes */
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int p = 0; p < PL; p++) aoff[m][p] = ((uint32_t)(p * ntb + min(mt * MB + m, ntb - 1)) * NSL + (uint32_t)s0) * 1024u;
#pragma unroll
    for (int j = 0; j < 4; j++) boff[j] = ((uint32_t)rb[j] * NSL + (uint32_t)s0) * 1024u;

    nmoe_sh_f32x4 acc[MB][4];
    const nmoe_sh_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[m][j] = zero;
    /* rings of DA slices of x (or act) operands and DB of weight operands: a
     * slice's registers are asked for again as soon as its products used them */
    constexpr int DA = MB == 4 ? 1 : MB == 2 && PL == 3 ? 2 : 4, DB = DA < 4 ? 2 : 4;
    uint4 a[DA][PL][MB], b[DB][4];
    auto load_a = [&](int buf, int p, int s) {
#pragma unroll
        for (int m = 0; m < MB; m++) a[buf][p][m] = nmoe_sh_load(ar, 16u * lane, aoff[m][p] + 1024u * (uint32_t)s);
    };
    auto load_b = [&](int buf, int s) {
#pragma unroll
        for (int j = 0; j < 4; j++) b[buf][j] = nmoe_sh_load(br, 16u * lane, boff[j] + 1024u * (uint32_t)s);
    };
    const __amdgpu_buffer_rsrc_t sr = nmoe_buffer(sc);
    auto load_s = [&](int j, int g) { /* the scales of groups g and g + 1 (from the wavefront's first) */
        return (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(sr, 2 * G * col, 32 * G * rb[j] + s0 + 2 * g, 0);
    };
    uint32_t sw[2][4];
#pragma unroll
    for (int j = 0; j < 4; j++) sw[0][j] = load_s(j, 0);
#pragma unroll
    for (int q = 0; q < DB; q++) load_b(q, q);
#pragma unroll
    for (int q = 0; q < DA; q++)
#pragma unroll
        for (int p = PL - 1; p >= 0; p--) load_a(q, p, q);
#pragma unroll 1
    for (int s = 0; s < SL; s += 4) { /* two groups */
        nmoe_sh_f32x4 P[MB][4];
#pragma unroll
        for (int j = 0; j < 4; j++) sw[1][j] = load_s(j, min(s / 2 + 2, SL / 2 - 2));
#pragma unroll
        for (int q = 0; q < 4; q++) {
#pragma unroll
            for (int p = PL - 1; p >= 0; p--) { /* the smallest part first */
#pragma unroll
                for (int m = 0; m < MB; m++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        P[m][j] = nmoe_sh_mfma(a[q % DA][p][m], b[q % DB][j], !(q & 1) && p == PL - 1 ? zero : P[m][j]);
                load_a(q % DA, p, min(s + q + DA, SL - 1));
            }
            load_b(q % DB, min(s + q + DB, SL - 1));
            if (q & 1)
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float sv = __uint_as_float(q == 3 ? sw[0][j] & 0xffff0000u : sw[0][j] << 16);
#pragma unroll
                    for (int m = 0; m < MB; m++)
#pragma unroll
                        for (int i = 0; i < 4; i++) acc[m][j][i] = __builtin_fmaf(sv, P[m][j][i], acc[m][j][i]);
                }
        }
#pragma unroll
        for (int j = 0; j < 4; j++) sw[0][j] = sw[1][j];
    }

    /* units (token block m, row pair q): tiles q and q + 2 */
    __shared__ nmoe_sh_f32x4 red[4 * MB * 4 * 64];
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int j = 0; j < 4; j++) red[((wave * MB + m) * 4 + j) * 64 + lane] = acc[m][j];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MB; m++)
#pragma unroll
        for (int q = 0; q < 2; q++) {
            if (((2 * m + q) & 3) != wave) continue;
            const int tb = mt * MB + m;
            if (tb >= ntb) continue;
            nmoe_sh_f32x4 v[2];
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int j = q + 2 * h;
                const int row = 16 * rb[j] + col;
                nmoe_sh_f32x4 r[4];
#pragma unroll
                for (int w = 0; w < 4; w++) r[w] = red[((w * MB + m) * 4 + j) * 64 + lane];
                v[h] = (r[0] + r[1]) + (r[2] + r[3]);
                if (GU) {
                    /* sum_g c_g xs_g on the matrix cores, both factors as
                     * three bf16 parts: the products down to 2^-24, smallest
                     * first */
                    nmoe_sh_f32x4 cc = zero;
                    uint4 xv[3], cv[3];
#pragma unroll
                    for (int p = 0; p < 3; p++) {
                        xv[p] = ws.xs3[((size_t)p * ntb + tb) * 64 + lane];
                        cv[p] = *(const uint4 *)(bs + (size_t)(1024 * p + row) * G + 8 * kb);
                    }
#pragma unroll
                    for (int o = 2; o >= 0; o--)
#pragma unroll
                        for (int p = 0; p <= o; p++) cc = nmoe_sh_mfma(xv[p], cv[o - p], cc);
                    v[h] = v[h] + cc;
                } else { /* sum_g as_g (b_g + 8 s_g): lane k of the fp32 MFMA is groups kb and 4 + kb */
                    nmoe_sh_f32x4 cc = zero;
#pragma unroll
                    for (int h4 = 0; h4 < 2; h4++) {
                        const int g = 4 * h4 + kb;
                        const float4 a4 = *(const float4 *)(ws.asq + (size_t)(16 * tb + col) * 32 + 4 * g);
                        const float cv = __builtin_fmaf(8.0f, nmoe_bf16f(sc[(size_t)row * G + g]), nmoe_bf16f(bs[(size_t)row * G + g]));
                        cc = __builtin_amdgcn_mfma_f32_16x16x4f32((a4.x + a4.y) + (a4.z + a4.w), cv, cc, 0, 0, 0);
                    }
                    v[h] = v[h] + cc;
                }
            }
            if (GU) {
                /* (the product of as[] fused into the first add of its sum would
                 * round differently in the two lanes of a pair, and a token's
                 * sums then depend on whether it sits in an even or an odd row) */
#pragma clang fp contract(off)
                /* act column 32 n + 16 q + col of tokens 4 kb .. + 3: slice n,
                 * k 16 q + col of the down product's operand */
                const int k = 16 * q + col;
                float as[4], ao[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    as[i] = nmoe_silu_dev(v[0][i]) * v[1][i];
                    ao[i] = nmoe_dpp_f<NMOE_DPP_XOR1>(as[i]); /* the neighbouring column */
                }
                /* even columns store tokens 0 and 1 of the pair, odd ones 2 and 3 */
                const bool odd = col & 1;
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const float lo = odd ? ao[2 + i] : as[i], hi = odd ? as[2 + i] : ao[i];
                    uint32_t pa[3], pb[3];
                    nmoe_sh_split3(lo, pa);
                    nmoe_sh_split3(hi, pb);
                    const int tr = 4 * kb + (odd ? 2 + i : i);
#pragma unroll
                    for (int p = 0; p < 3; p++)
                        ((uint32_t *)(ws.ap + (((size_t)p * ntb + tb) * NMOE_SH_DN_SL + n) * 64 + tr + 16 * (k >> 3)))[(k & 7) >> 1] =
                            pa[p] | (pb[p] << 16);
                }
                float sm[4];
#pragma unroll
                for (int i = 0; i < 4; i++) sm[i] = nmoe_dpp_group_sum<16>(as[i]);
                const float s01 = col & 1 ? sm[1] : sm[0], s23 = col & 1 ? sm[3] : sm[2];
                if (col < 4) ws.asq[(size_t)(16 * tb + 4 * kb + col) * 32 + 2 * n + q] = col & 2 ? s23 : s01;
            } else {
#pragma unroll
                for (int h = 0; h < 2; h++)
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const int t = 16 * tb + 4 * kb + i;
                        if (t < ntok) out[(size_t)t * NMOE_HIDDEN + 16 * rb[q + 2 * h] + col] = v[h][i];
                    }
            }
        }
}

/* Tokens from which the matrix-core launches run: their three launches take
 * 20 to 22 us up to 64 tokens, the per-token kernels 18 to 19 at 32 and 21 to
 * 22 at 37. */
#define NMOE_SHARED_MM_MIN 36

/* Tokens the three launches take at a time, which bounds their scratch (15,680
 * bytes a token and 6.6 MB of the weights' copies) at 264 MB.  Chunks of 4,096
 * would take 71 MB, but a call of 4,097 to 16,384 bf16 tokens 4 to 9 % longer
 * (8,192: 172 and 179 us; fp32 x 229 and 238, 16,384: 528 and 477). */
#define NMOE_SHARED_CHUNK 16384

/* Scratch of the matrix-core launches, every part a multiple of 1 KB. */
static size_t nmoe_sh_layout(size_t max_tokens, uint8_t *base, nmoe_sh_ws *ws) {
    const size_t tb = (max_tokens + 15) / 16;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        uint8_t *p = base + at;
        at += (bytes + 1023) / 1024 * 1024;
        return p;
    };
    ws->wgu = (uint4 *)take((size_t)64 * NMOE_SH_GU_SL * 1024);
    ws->wdn = (uint4 *)take((size_t)(NMOE_HIDDEN / 16) * NMOE_SH_DN_SL * 1024);
    ws->sgu = (uint16_t *)take((size_t)4 * 1024 * NMOE_SH_GU_G * 2);
    ws->sdn = (uint16_t *)take((size_t)2 * NMOE_HIDDEN * NMOE_SH_DN_G * 2);
    ws->xp = (uint4 *)take(3 * tb * NMOE_SH_GU_SL * 1024);
    ws->xs3 = (uint4 *)take(3 * tb * 1024);
    ws->ap = (uint4 *)take(3 * tb * NMOE_SH_DN_SL * 1024);
    ws->asq = (float *)take(tb * 16 * 32 * sizeof(float));
    return at;
}

/* The shared expert's scratch: the per-token kernels' activations, then, in
 * contexts of enough tokens, the matrix-core launches'. */
#define NMOE_SH_ACT_BYTES ((size_t)(NMOE_SHARED_MM_MIN - 1) * NMOE_INTER * sizeof(float))
static_assert(NMOE_SH_ACT_BYTES % 1024 == 0, "the parts after it stay aligned");
extern "C" size_t nmoe_shared_scratch_bytes(int max_tokens) {
    nmoe_sh_ws ws;
    if (max_tokens < NMOE_SHARED_MM_MIN) return (size_t)max_tokens * NMOE_INTER * sizeof(float);
    return NMOE_SH_ACT_BYTES + nmoe_sh_layout((size_t)min(max_tokens, NMOE_SHARED_CHUNK), NULL, &ws);
}

template <int PL, int MB, bool GU>
static void nmoe_shared_mm_launch(const nmoe_sh_ws &ws, int ntok, int ntb, float *out, hipStream_t s) {
    const int mtiles = (ntb + MB - 1) / MB, swz = mtiles >= 16;
    const int blocks = (swz ? (mtiles + 7) / 8 * 8 : mtiles) * (GU ? 16 : 32);
    hipLaunchKernelGGL((nmoe_shared_mm_kernel<PL, MB, GU>), dim3(blocks), dim3(256), 0, s, ws, ntok, ntb, mtiles, swz,
                       out);
}

template <int MB>
static void nmoe_shared_mm_pair(const nmoe_sh_ws &ws, bool bf, int ntok, int ntb, float *out, hipStream_t s) {
    if (bf)
        nmoe_shared_mm_launch<1, MB, true>(ws, ntok, ntb, out, s);
    else
        nmoe_shared_mm_launch<3, MB, true>(ws, ntok, ntb, out, s);
    nmoe_shared_mm_launch<3, MB, false>(ws, ntok, ntb, out, s);
}

static void nmoe_shared_mm(nmoe_hip_ctx *ctx, const nmoe_hip_shared_expert *se, const void *x, int x_dtype, int ntok,
                           float *shared_out, float *graw, hipStream_t s) {
    nmoe_sh_ws ws;
    (void)nmoe_sh_layout((size_t)min(ctx->max_tokens, NMOE_SHARED_CHUNK), (uint8_t *)ctx->s_act + NMOE_SH_ACT_BYTES, &ws);
    const bool bf = x_dtype == NMOE_HIP_BF16;
    for (int t0 = 0; t0 < ntok; t0 += NMOE_SHARED_CHUNK) {
        const int n = min(ntok - t0, NMOE_SHARED_CHUNK), ntb = (n + 15) / 16;
        const int b0 = t0 == 0 ? 0 : NMOE_SH_WB + NMOE_SH_SB;
        const dim3 gp(NMOE_SH_WB + NMOE_SH_SB - b0 + 4 * ntb + (n + 3) / 4);
        float *so = shared_out + (size_t)t0 * NMOE_HIDDEN;
        if (bf)
            hipLaunchKernelGGL(nmoe_shared_prep_kernel<uint16_t>, gp, dim3(256), 0, s, *se, ws,
                               (const uint16_t *)x + (size_t)t0 * NMOE_HIDDEN, n, ntb, b0, graw + t0);
        else
            hipLaunchKernelGGL(nmoe_shared_prep_kernel<float>, gp, dim3(256), 0, s, *se, ws,
                               (const float *)x + (size_t)t0 * NMOE_HIDDEN, n, ntb, b0, graw + t0);
        /* the smallest token tile whose gate/up grid (16 blocks a tile) is one
         * round of the 256 CUs, then the largest: 16 against 32 and 64 tokens a
         * tile (fp32 x, us) 26 / 30 / 35 at 251 tokens, 35 / 32 / 35 at 512, 55
         * / 44 / 41 at 1,000, 186 / 136 / 121 at 4,096 */
        if (ntb <= 16)
            nmoe_shared_mm_pair<1>(ws, bf, n, ntb, so, s);
        else if (ntb <= 32)
            nmoe_shared_mm_pair<2>(ws, bf, n, ntb, so, s);
        else
            nmoe_shared_mm_pair<4>(ws, bf, n, ntb, so, s);
    }
}

int nmoe_check_x(nmoe_hip_ctx *ctx, const void *x, int x_dtype, int ntok);

static bool nmoe_qtensor_ok(const nmoe_hip_qtensor &q) {
    return q.w != NULL && q.scales != NULL && q.biases != NULL && nmoe_aligned(q.w, 4) && nmoe_aligned(q.scales, 2) &&
           nmoe_aligned(q.biases, 2);
}

extern "C" int nmoe_moe_shared_expert(nmoe_hip_ctx *ctx, const nmoe_hip_shared_expert *se, const void *x,
                                      int x_dtype, int ntok, float *shared_out, float *shared_gate_raw,
                                      void *stream) {
    if (ctx == NULL) return NMOE_HIP_EINVAL;
    if (se == NULL || !nmoe_qtensor_ok(se->gate) || !nmoe_qtensor_ok(se->up) || !nmoe_qtensor_ok(se->down) ||
        !nmoe_qtensor_ok(se->score))
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "shared expert: NULL or misaligned tensor (w 4 B, scales/biases 2 B)");
    int rc = nmoe_check_x(ctx, x, x_dtype, ntok);
    if (rc != NMOE_HIP_OK) return rc;
    if (shared_out == NULL || shared_gate_raw == NULL || !nmoe_aligned(shared_out, 16))
        return nmoe_fail(ctx, NMOE_HIP_EINVAL, "shared_out (16-byte aligned) and shared_gate_raw are required");
    if (ntok >= NMOE_SHARED_MM_MIN) {
        nmoe_shared_mm(ctx, se, x, x_dtype, ntok, shared_out, shared_gate_raw, nmoe_stream_of(ctx, stream));
        NMOE_HIP_TRY(ctx, hipGetLastError());
        return NMOE_HIP_OK;
    }
    /* tokens a block: the fewer, the more wavefronts hide a row's loads; the
     * more, the fewer times a row is read.  1 / 2 / 4 a block (fp32 x, both
     * launches, us): 7.1 / 7.6 / 10.1 at 4 tokens, 10.0 / 9.1 / 10.6 at 8,
     * 14.8 / 12.8 / 12.7 at 16, 23.7 / 19.4 / 19.0 at 32 */
    const int tpb = ntok <= 4 ? 1 : ntok <= 12 ? 2 : 4;
    const dim3 ggu(NMOE_INTER / 4 + 1, (ntok + tpb - 1) / tpb), gdn(NMOE_HIDDEN / 4, (ntok + tpb - 1) / tpb);
    hipStream_t s = nmoe_stream_of(ctx, stream);
    if (x_dtype == NMOE_HIP_BF16)
        hipLaunchKernelGGL(nmoe_shared_gateup_kernel<uint16_t>, ggu, dim3(256), 0, s, se->gate.w, se->gate.scales,
                           se->gate.biases, se->up.w, se->up.scales, se->up.biases, se->score.w, se->score.scales,
                           se->score.biases, (const uint16_t *)x, ntok, tpb, ctx->s_act, shared_gate_raw);
    else
        hipLaunchKernelGGL(nmoe_shared_gateup_kernel<float>, ggu, dim3(256), 0, s, se->gate.w, se->gate.scales,
                           se->gate.biases, se->up.w, se->up.scales, se->up.biases, se->score.w, se->score.scales,
                           se->score.biases, (const float *)x, ntok, tpb, ctx->s_act, shared_gate_raw);
    hipLaunchKernelGGL(nmoe_shared_down_kernel, gdn, dim3(256), 0, s, se->down.w, se->down.scales, se->down.biases,
                       (const float *)ctx->s_act, ntok, tpb, shared_out);
    NMOE_HIP_TRY(ctx, hipGetLastError());
    return NMOE_HIP_OK;
}
