// attn16.h -- the batch attention of attn.h (infer.c:1017-1058) on fp16 matrix cores with
// fp32-like accuracy: k_attn_tile's work split (AQ_T tokens of one head against a chunk of
// positions, the same partial-result slots for k_attn_merge), with both products on
// v_mfma_f32_16x16x32_f16 over operands split into fp16 hi and lo (x = hi + lo to ~22 bits, as
// the expert GEMMs split their activations): a product of two split operands is hi.hi +
// hi.lo + lo.hi in fp32 (the dropped lo.lo is ~2^-22 of it).
//
// The cache entries come in the split form attn_prep_run writes once per position (dense.h: ksp
// rows scaled by 2^-e[p]). A tile is A16_P positions' rows, one contiguous run that lands in
// shared memory by DMA while the tile before it is used. A wave has 16 tokens to itself: it
// forms the transposed scores S^T = K Q^T (rows positions, columns tokens), so that a lane's
// eight scores all belong to its token and, as exponentials, are in place as the B operand of
// the transposed weighted sum O^T = V^T P^T, whose A operand is the same K rows read through the
// transposing shared-memory load. Queries (B operands) and the sum stay in registers for the
// whole chunk (272 of a wave's 512 registers, so one wave a SIMD), and a tile needs one barrier
// and no exchange between waves.
//
// What bounds it: per 32 positions a wave issues 204 MFMAs of 16 clocks (3264) and some 700 other
// instructions, 4 clocks each, of which those between the two products (the softmax) overlap
// nothing: the matrix cores are busy 35 % of the time, the waves issue 46 % of it, are ready 40 %
// and wait 14 %. 1024 tokens at
// position 3072 (20 heads): 576 us, 478 TFLOP/s of split products; with the scores and
// exponentials exchanged through shared memory, the rows' transposed copy staged beside them
// and four barriers per 16 positions it took 1030.
//
// Softmax reference: the exponentials are taken against a token's reference score m, which
// follows the running maximum only when a score passes m + A16_SLACK, so the sum is
// rescaled a few times a chunk and not once a tile. For the weighted sum they are scaled by
// 2^(A16_PUP + e[p] - eR), eR at least every e[p] of the tile, so that fp16 holds them (e^6 2^6 <
// 2^15); eR follows the tile's largest e upward at once and downward when it is more than
// A16_EDOWN above it, so that a split exponential's error stays at 2^-25 of the largest's or less.
// Downward the sum grows by as much, so a step down stops where the sum would pass 2^A16_XMAX, and
// a tile of zero entries alone, whose products are zero at any scale, moves nothing (a16_scale).
#pragma once

#include "attn.h"

#define A16_P 32                    // positions a tile: the K dimension of the weighted sum's MFMA
#define A16_BLOCK 256               // a wave per SIMD (up to 512 registers each), 16 tokens a wave
#define A16_NKS (AQ_KQ_MAX / 32)    // 32-column steps of a row
#define A16_NCB (AT_KV_MAX / 16)    // 16-column blocks of the weighted sum
#define A16_STAGE (A16_P * SPL_KROW * 2)
#define A16_SLACK 6.0f
#define A16_PUP 6
#define A16_EDOWN 6
#define A16_EMIN (-200)             // below any entry's exponent (spl_exp: -163 at least)
#define A16_XMAX 100
static_assert(AQ_T == 16 * A16_BLOCK / 64, "16 tokens a wave");
static_assert(AQ_KQ_MAX == SPL_KCOLS && AT_KV_MAX <= SPL_KCOLS, "the split rows hold the widest entry");
static_assert(A16_STAGE % 16 == 0, "16-byte DMA slots");
static_assert(16 * SPL_KROW * 2 + 2 * SPL_KCOLS + 2 * AT_KV_MAX < 65536, "one base register for a stage's reads");

// s_waitcnt immediate (gfx9 encoding) for lgkmcnt(n) alone, n <= 15
#define A16_WAIT_LGKM(n) (0xC07F | ((n) << 8))

// The scale exponent that follows eR at a tile whose largest is em (SPL_EMPTY: zero entries
// alone), with the sum's magnitudes below 2^xa (A16_ZERO: the sum is zero, and moves at no cost).
#define A16_ZERO (-1000)
__host__ __device__ constexpr int a16_scale(int eR, int em, int xa) {
    if (em == SPL_EMPTY) return eR;
    if (em >= eR || xa == A16_ZERO) return em;
    const int room = xa < A16_XMAX ? A16_XMAX - xa : 0;
    return em > eR - room ? em : eR - room;
}
constexpr bool a16_scale_bounded() {
    for (int eR = A16_EMIN; eR <= 113; eR += 7)
        for (int em = -163; em <= 113; em += 12)
            for (int xa = -126; xa <= 129; xa += 5) {
                const int e = a16_scale(eR, em, xa), x = xa + eR - e;
                if (e < em || (e < eR && x > A16_XMAX) || (e > em && e != eR && x != A16_XMAX)) return false;
                if (a16_scale(eR, SPL_EMPTY, xa) != eR || a16_scale(eR, em, A16_ZERO) != em) return false;
            }
    return true;
}
static_assert(a16_scale_bounded(), "a step down lands on the tile's exponent or on the sum's bound");

typedef _Float16 a16_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 a16_h4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) a16_h4 a16_lds_h4;

// The 16-lane group's 4 rows x 16 columns of halves, transposed: lane i of the group names
// the 8 bytes at row i / 4, columns 4 (i % 4) .. + 3, and gets column i of the four rows.
__device__ static inline a16_h4 a16_tr(const _Float16 *p) {
    typedef short s4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s4 lds_s4;
    return __builtin_bit_cast(a16_h4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4 *)p));
}

// The maximum over the four lanes l % 16 + {0, 16, 32, 48}.
__device__ static inline float a16_max4(float v) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ static inline float a16_sum4(float v) {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    u2 r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// e^x for x <= A16_SLACK in nine instructions: 2^(x log2 e), the product split into its rounded
// value and what that leaves out (log2 e to 48 bits), which joins as e^r = 1 + r (|r| < 2^-16).
// Within 1.3 ulp of e^x where that is a normal number (1.26 at worst over every float of [-104, 6]),
// 0 below (v_exp_f32 flushes) and for -inf; NaN stays NaN.
__device__ static inline float a16_exp(float x) {
    const float L = 1.44269504f, L2 = 1.92596299e-8f, LN2 = 0.693147181f;  // log2 e = L + L2
    x = x < -100.0f ? -100.0f : x;
    const float t = __fmul_rn(x, L), r = fmaf(x, L2, fmaf(x, L, -t));
    const float e = __builtin_amdgcn_exp2f(t);
    return fmaf(e, __fmul_rn(r, LN2), e);
}

__global__ __launch_bounds__(A16_BLOCK, 1) void k_attn_tile16(AttnTileArgs g) {
    __shared__ __align__(16) uint8_t stg[2][A16_STAGE];  // tiles j and j + 1
    const AttnArgs &a = g.a;
    const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lg = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    // blocks dispatched longest first, so that short ones fill the CUs at the end: chunk by
    // chunk (the earlier chunks are the full ones), and in a chunk the later token tiles
    // (which attend more of its positions) first, the heads of a tile in a row
    const int L = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z), per = gridDim.y * gridDim.z;
    const int c = L / per, t0 = AQ_T * (gridDim.y - 1 - (L % per) / gridDim.z), h = (L % per) % gridDim.z;
    const int kv = a.kv, rope = a.rope, KQ = kv + rope, H = a.H, nch = a.nblk;
    const int tl = min(g.n, t0 + AQ_T);    // the tile's tokens t0 .. tl - 1
    const int r0 = c * g.chunk;
    const int r1 = min(r0 + g.chunk, a.pos + tl);  // the chunk's positions any of them attends
    auto slot = [&](int t) { return ((size_t)t * nch + c) * H + h; };  // partial-result slot of token t
    if (r0 >= r1) {
        for (int i = tid; i < (tl - t0) * kv; i += A16_BLOCK) a.part_ctx[slot(t0 + i / kv) * kv + i % kv] = 0.0f;
        if (tid < tl - t0) {
            a.part_ml[slot(t0 + tid) * 2] = -INFINITY;
            a.part_ml[slot(t0 + tid) * 2 + 1] = 0.0f;
        }
        return;
    }
    const int ntile = (r1 - r0 + A16_P - 1) / A16_P;

    // a tile by DMA into stage st: A16_P rows, contiguous in the cache and in shared memory (each
    // wave an 18 KB run and the first wave the last KB; the DMA's offset field steps the address
    // and the destination alike, so a base serves four). Rows past r1 hold what an earlier prompt
    // left, and an exponential of 0 doesn't take an inf or NaN out of a sum: the buffer ends
    // at r1, past which its loads give zeros.
    auto issue = [&](int s0, int st) {
        constexpr int KB = A16_STAGE / 1024, PER = KB / 4;
        static_assert(KB * 1024 == A16_STAGE && KB == 4 * PER + 1 && PER % 4, "whole waves of DMA, one past four equal runs");
        const uint8_t *ks = reinterpret_cast<const uint8_t *>(a.ksp + (size_t)s0 * SPL_KROW);
        const int end = min(r1 - s0, A16_P) * SPL_KROW * 2;
        const auto *dst = (const __attribute__((address_space(3))) uint8_t *)&stg[0][0] + st * A16_STAGE;
        auto run = [&](auto N, int kb) {
            dma_buf<decltype(N)::value>(ks + 1024 * kb, end - 1024 * kb, 16 * lane, (const lds_void *)(dst + 1024 * kb));
        };
#pragma unroll
        for (int r = 0; r + 4 <= PER; r += 4) run(std::integral_constant<int, 4>{}, PER * w + r);
        run(std::integral_constant<int, PER % 4>{}, PER * w + PER / 4 * 4);
        if (w == 0) run(std::integral_constant<int, 1>{}, KB - 1);
    };
    issue(r0, 0);  // before the queries' loads: the two share a round trip

    // the lane's token and its query as B operands: step s holds columns 32 s + 8 lg .. + 7 (an
    // 8-column group lies inside one part, since kv and KQ are multiples of 16), scaled by 2^-eq
    const int tw = t0 + 16 * w, t = tw + l16;
    a16_h8 qh[A16_NKS], ql[A16_NKS];
    int eq;
    {
        const int tq = min(t, g.n - 1);  // past the batch: any token (not stored)
        const float *qa = a.q_abs + ((size_t)tq * H + h) * kv, *qp = a.q_pe + ((size_t)tq * H + h) * rope - kv;
        float4 qv[A16_NKS][2];
        float mx = 0.0f;
#pragma unroll
        for (int s = 0; s < A16_NKS; s++) {
            const int col = 32 * s + 8 * lg;
            const float *src = col < kv ? qa + col : qp + col;
            qv[s][0] = col < KQ ? *(const float4 *)src : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            qv[s][1] = col < KQ ? *(const float4 *)(src + 4) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
#pragma unroll
        for (int s = 0; s < A16_NKS; s++)
#pragma unroll
            for (int k = 0; k < 2; k++)
                mx = fmaxf(mx, fmaxf(fmaxf(fabsf(qv[s][k].x), fabsf(qv[s][k].y)), fmaxf(fabsf(qv[s][k].z), fabsf(qv[s][k].w))));
        eq = spl_exp(a16_max4(mx));
#pragma unroll
        for (int s = 0; s < A16_NKS; s++) {
            const float xs[8] = {qv[s][0].x, qv[s][0].y, qv[s][0].z, qv[s][0].w, qv[s][1].x, qv[s][1].y, qv[s][1].z, qv[s][1].w};
#pragma unroll
            for (int k = 0; k < 8; k++) {
                _Float16 hi, lo;
                spl_split(ldexpf(xs[k], -eq), hi, lo);
                qh[s][k] = hi;
                ql[s][k] = lo;
            }
            // in accumulator registers, which the matrix cores read as well: the vector registers
            // don't hold everything, and what the compiler moves out of them it copies at each use
            asm volatile("" : "+a"(ql[s]));
        }
    }

    aq_f4 acc[A16_NCB];  // O^T: column block cb, columns 16 cb + 4 lg + r of the lane's token
#pragma unroll
    for (int i = 0; i < A16_NCB; i++) acc[i] = (aq_f4){0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, l = 0.0f;  // the token's reference score; the lane's part of its sum
    int eR = A16_EMIN;              // the scale of acc: 2^(eR - A16_PUP)

    // the wave's tiles: those that any of its tokens attends (the later ones it only passes on)
    const int past = a.pos + tw + 15 - r0, nt = past < 0 ? 0 : min(ntile, past / A16_P + 1);
    int j = 0;
    // on to tile j: this wave's part of it has landed, then every wave's has and none still
    // reads tile j - 1, whose stage takes tile j + 1
    auto next = [&]() {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        block_barrier();
        if (j + 1 < ntile) issue(r0 + A16_P * (j + 1), (j + 1) & 1);
    };
    a16_h4 vb[3][2][4];  // the weighted sum's operands: see vload
    // column blocks cb and cb + 1, rows 4 lg .. + 3 and 16 + 4 lg .. + 3 of each transposed (the
    // lane names row 4 lg + l16 / 4), hi then lo
    auto vload = [&](a16_h4 (&o)[2][4], int cb) {
        const _Float16 *vr = reinterpret_cast<const _Float16 *>(stg[j & 1]) + (4 * lg + (l16 >> 2)) * SPL_KROW + 4 * (l16 & 3);
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const _Float16 *p = vr + 16 * (cb + k);
            o[k][0] = a16_tr(p);
            o[k][1] = a16_tr(p + 16 * SPL_KROW);
            o[k][2] = a16_tr(p + SPL_KCOLS);
            o[k][3] = a16_tr(p + 16 * SPL_KROW + SPL_KCOLS);
        }
    };
    float v[8];  // tile j's scores: position s0 + 16 (i / 4) + 4 lg + i % 4 of the lane's token
    int ep[8];   // and those positions' exponents
    float mx;    // the lane's largest score
    int em;      // and largest exponent of the chunk's own positions
    auto scores = [&]() {
        const int s0 = r0 + A16_P * j;
        const _Float16 *K = reinterpret_cast<const _Float16 *>(stg[j & 1]);
        // S^T: position block pb, lane holds positions s0 + 16 pb + 4 lg + r of its token
        // (the hi.hi products in three chains of steps, so that a score is rounded no more often
        // than sums of column quarters would be, and the small cross products in one)
        aq_f4 d[2][4];
#pragma unroll
        for (int pb = 0; pb < 2; pb++)
#pragma unroll
            for (int k = 0; k < 4; k++) d[pb][k] = (aq_f4){0.0f, 0.0f, 0.0f, 0.0f};
        const _Float16 *kr = K + l16 * SPL_KROW + 8 * lg;
        // operands requested two steps ahead: with a wave per SIMD nothing else hides the
        // latency of a shared-memory read, and left to itself the compiler asks for a step's
        // operands right before their products
        a16_h8 kb[3][4];  // a step's rows l16 and l16 + 16: hi, hi, lo, lo
        auto kload = [&](a16_h8 (&o)[4], int s) {
            o[0] = *(const a16_h8 *)(kr + 32 * s);
            o[1] = *(const a16_h8 *)(kr + 16 * SPL_KROW + 32 * s);
            o[2] = *(const a16_h8 *)(kr + SPL_KCOLS + 32 * s);
            o[3] = *(const a16_h8 *)(kr + 16 * SPL_KROW + SPL_KCOLS + 32 * s);
        };
        kload(kb[0], 0);
        kload(kb[1], 1);
#pragma unroll
        for (int s = 0; s < A16_NKS; s++) {
            if (s + 2 < A16_NKS) kload(kb[(s + 2) % 3], s + 2);
            __builtin_amdgcn_sched_barrier(0);
            if (s + 2 < A16_NKS) __builtin_amdgcn_s_waitcnt(A16_WAIT_LGKM(8));
            else if (s + 1 < A16_NKS) __builtin_amdgcn_s_waitcnt(A16_WAIT_LGKM(4));
            else __builtin_amdgcn_s_waitcnt(A16_WAIT_LGKM(0));
            const a16_h8 *o = kb[s % 3];
            d[0][s % 3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o[0], qh[s], d[0][s % 3], 0, 0, 0);
            d[1][s % 3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o[1], qh[s], d[1][s % 3], 0, 0, 0);
            d[0][3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o[0], ql[s], d[0][3], 0, 0, 0);
            d[1][3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o[1], ql[s], d[1][3], 0, 0, 0);
            d[0][3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o[2], qh[s], d[0][3], 0, 0, 0);
            d[1][3] = __builtin_amdgcn_mfma_f32_16x16x32_f16(o[3], qh[s], d[1][3], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; i++) ep[i] = *(const int *)(K + (16 * (i >> 2) + 4 * lg + (i & 3)) * SPL_KROW + SPL_KEXP);
        vload(vb[0], 0);  // ahead of the softmax
        vload(vb[1], 2);
        const int lim = min(r1 - 1, a.pos + t);  // the token's last position of the chunk
        mx = -INFINITY;
        em = SPL_EMPTY;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const int s = s0 + 16 * (i >> 2) + 4 * lg + (i & 3);
            const aq_f4 *dp = d[i >> 2];
            const int k = i & 3;
            const float x = (dp[0][k] + dp[1][k]) + (dp[2][k] + dp[3][k]);
            const float y = __fmul_rn(ldexpf(x, eq + ep[i]), a.kq_scale);
            v[i] = s <= lim ? y : -INFINITY;
            mx = fmaxf(mx, v[i]);
            em = max(em, s < r1 ? ep[i] : SPL_EMPTY);
        }
    };
    a16_h8 ph, pl;  // P^T: k slot i is position 16 (i / 4) + 4 lg + i % 4 of the tile
    auto exps = [&]() {
        const float mu = m == -INFINITY ? 0.0f : m;  // (no position yet: every exponential is 0)
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float e = a16_exp(__fsub_rn(v[i], mu));
            l = __fadd_rn(l, e);
            _Float16 hi, lo;
            spl_split(ldexpf(e, ep[i] - eR + A16_PUP), hi, lo);
            ph[i] = hi;
            pl[i] = lo;
        }
    };
    if (nt > 0) {
        next();
        scores();
        bool more = true;
        // The inner loop runs while the reference and eR hold; the rescale between its runs is
        // kept out of it, because a branch around it inside made the compiler move the whole sum
        // out of the accumulator registers and back in every tile (256 instructions).
        while (more) {
            {
                const float mn = fmaxf(m, a16_max4(mx));
                const int et = __builtin_amdgcn_readfirstlane((int)a16_max4((float)em));  // the same for every l16
                int xa = A16_ZERO;
                if (j > 0 && et < eR) {
                    float ax = 0.0f;
#pragma unroll
                    for (int i = 0; i < A16_NCB; i++)
#pragma unroll
                        for (int r = 0; r < 4; r++) ax = fmaxf(ax, fabsf(acc[i][r]));
                    const unsigned b = __builtin_amdgcn_readfirstlane(__float_as_uint(wave_max_f(ax)));
                    if (b) xa = (int)(b >> 23) - 126;
                }
                const int eT = a16_scale(eR, et, xa);
                float cr = mn == -INFINITY ? 1.0f : expf(__fsub_rn(m, mn));  // 0 while m is -inf
                l = __fmul_rn(l, cr);
                cr = ldexpf(cr, eR - eT);
#pragma unroll
                for (int i = 0; i < A16_NCB; i++)
#pragma unroll
                    for (int r = 0; r < 4; r++) acc[i][r] = __fmul_rn(acc[i][r], cr);
                m = mn;
                eR = eT;
            }
            exps();
            for (;;) {
                // O^T += V^T P^T
#pragma unroll
                for (int cb = 0; cb < A16_NCB; cb += 2) {
                    if (cb + 4 < A16_NCB) vload(vb[(cb / 2 + 2) % 3], cb + 4);
                    __builtin_amdgcn_sched_barrier(0);
                    if (cb + 4 < A16_NCB) __builtin_amdgcn_s_waitcnt(A16_WAIT_LGKM(15));
                    else if (cb + 2 < A16_NCB) __builtin_amdgcn_s_waitcnt(A16_WAIT_LGKM(8));
                    else __builtin_amdgcn_s_waitcnt(A16_WAIT_LGKM(0));
                    const a16_h4(*o)[4] = vb[cb / 2 % 3];
                    a16_h8 vh[2], vl[2];
#pragma unroll
                    for (int k = 0; k < 2; k++) {
                        vh[k] = __builtin_shufflevector(o[k][0], o[k][1], 0, 1, 2, 3, 4, 5, 6, 7);
                        vl[k] = __builtin_shufflevector(o[k][2], o[k][3], 0, 1, 2, 3, 4, 5, 6, 7);
                    }
#pragma unroll
                    for (int k = 0; k < 2; k++) acc[cb + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[k], ph, acc[cb + k], 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 2; k++) acc[cb + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[k], pl, acc[cb + k], 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 2; k++) acc[cb + k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl[k], ph, acc[cb + k], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
                j++;
                more = j < nt;
                if (!more) break;
                next();
                scores();
                // a score past the reference's slack, or an exponent outside eR's range
                if (__any(mx > m + A16_SLACK || em > eR) || (!__any(em >= eR - A16_EDOWN) && __any(em > SPL_EMPTY))) break;
                exps();
            }
        }
    }
    for (; j < ntile; j++) next();  // (its part of the other waves' tiles)
    l = a16_sum4(l);
    if (t < tl) {
        float *out = a.part_ctx + slot(t) * kv;
#pragma unroll
        for (int cb = 0; cb < A16_NCB; cb++)
            if (16 * cb < kv)
                *(float4 *)(out + 16 * cb + 4 * lg) = make_float4(ldexpf(acc[cb][0], eR - A16_PUP), ldexpf(acc[cb][1], eR - A16_PUP),
                                                                  ldexpf(acc[cb][2], eR - A16_PUP), ldexpf(acc[cb][3], eR - A16_PUP));
        if (lg == 0) {
            a.part_ml[slot(t) * 2] = m;
            a.part_ml[slot(t) * 2 + 1] = l;
        }
    }
}
