// gemm.h -- the dense Q8_0 products of a prefill batch (matvec_q80_rows, infer.c:765-786,
// for every token of the batch) as MFMA GEMMs: each weight panel is read once per tile of
// up to QG_TT_MAX tokens instead of once per token.
//
//   k_norm_split  each token's input row, normalised as glm.c normalises it when the
//                 product takes rmsnorm(x) * w (infer.c:746-752), in the split form of the
//                 grouped expert GEMMs (grouped.h): fp16 hi and lo with one exponent per row;
//   k_gemm_q8     y[t][r] = sum_g s[r][g] * (q[r][g] . x_t[g]) for a tile of 64 rows of the
//                 matrix (four waves of 16) and up to QG_TT_MAX tokens, with epilogues for glm.c's
//                 SwiGLU pair (infer.c:1078-1080) and residual add (infer.c:1061, 1083).
//
// Weights stay in glm.c's row-major Q8_0 form with fp32 scales, which the decode products
// (dense.h) read too. Per 32-column block (v_mfma_f32_16x16x32_f16, group size 32) or
// 16-column group (v_mfma_f32_16x16x16_f16, group size 16): the block's int8 weights converted to fp16 exactly, two MFMAs (hi, then lo of the inputs)
// into one fp32 accumulator, and one fma applying the group's fp32 scale into the running
// fp32 sum; 2^e at the end. The inputs carry 22 significant bits, so each product is
// within ~2^-21 of fp32's.
//
// Per-head products (k_b and v_b, whose row groups of x_rows rows read their own slice of
// the input, x_stride apart) run as groups: a block's rows lie inside one group.
//
// Block order is XCD-aware: the blocks of one 64-row panel (its token tiles) run on one XCD,
// so the panel is fetched from HBM once and then read from that XCD's L2 (k_gemm_q8).
#pragma once

#include <type_traits>

#include "common.h"

#define QG_BLOCK 256
#define QG_TT_MAX 64            // tokens per tile: 32 or 64 (qg_tokens)
#define QG_KC 64                // columns per staged chunk
#define QG_RB (QG_KC * 2)       // bytes of one staged row (one plane of one token)
#define QG_RG (QG_RB / 16)      // 16-byte groups per staged row
#define QG_XCD 8                // XCDs the dispatcher deals blocks over, round robin
#define QG_GEMM_MIN_TOKENS 8    // smaller batches take the per-token products (dense.h)

enum { QG_PLAIN = 0, QG_RESID = 1, QG_PAIR = 2 };

struct QgArgs {
    const int8_t *q, *q2;      // [rows][cols] int8 (q2: up, for QG_PAIR)
    const float *s, *s2;       // [rows][cols / gs] fp32 scales
    const __half *xs;          // split inputs [n][2][xcols]: hi, lo
    const int *xe;             // [n] their exponents
    const __half *zeros;       // 16 bytes of zeros (staged past the last column)
    float *y;                  // y[t * ldy + r]
    const float *resid;        // QG_RESID: y = resid[t * ldr + r] + dot
    int rows, cols, gs, n, xcols, ldy, ldr;
    int x_rows, x_stride;      // row group g (x_rows rows) reads split columns g * x_stride ..
    int bpg, groups, tiles;    // 64-row blocks per group, groups, token tiles
    float *y_b;                // QG_PLAIN with rows_b > 0: also y_b[t * rows_b + r] = q2 (scales s2) . v,
    int rows_b;                // rows_b rows of the same columns
};

typedef _Float16 qg_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 qg_h4 __attribute__((ext_vector_type(4)));
typedef float qg_f4 __attribute__((ext_vector_type(4)));
typedef float qg_f2 __attribute__((ext_vector_type(2)));
typedef unsigned qg_u2 __attribute__((ext_vector_type(2)));

// ---- the inputs' split form ---------------------------------------------------------

// One block per token row t of x (row t at x + t * ldx, n columns, n a multiple of 8):
// v = rmsnorm(x) * norm when norm is given (glm.c's operations: fp64 sum of squares, fp32
// mean, 1 / sqrtf of mean + 1e-5, then (x * inv) * w), else v = x; then
// sp[t][0][:] = fp16(v 2^-e), sp[t][1][:] = fp16(v 2^-e - hi), ex[t] = e, with e from
// max |v| so that the row's largest value sits near 2^14.
#define QG_SPLIT_MAX 40  // row values a thread holds: rows of up to 40 x QG_BLOCK = 10240 columns
// NK: the values a thread holds (n <= NK x QG_BLOCK; the launch takes the fewest of 2, 8,
// 20, 40 that hold the row, so a 2048-column row issues 8 loads a thread, not 40; the
// values past n add nothing, so every NK gives the same bits)
template <int NK>
__global__ __launch_bounds__(QG_BLOCK) void k_norm_split(const float *__restrict__ x, int ldx, int n,
                                                         const float *__restrict__ norm, __half *__restrict__ sp,
                                                         int *__restrict__ ex) {
    __shared__ double red_d[QG_BLOCK / 64];
    __shared__ float red_f[QG_BLOCK / 64];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const float *src = x + (size_t)t * ldx;
    // the row read once: thread tid holds columns tid + QG_BLOCK k
    float v[NK], nw[NK];
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int i = tid + QG_BLOCK * k;
        v[k] = i < n ? src[i] : 0.0f;
        nw[k] = norm && i < n ? norm[i] : 0.0f;
    }
    float inv = 1.0f;
    if (norm) {
        double ss = 0.0;
#pragma unroll
        for (int k = 0; k < NK; k++)
            if (tid + QG_BLOCK * k < n) ss += (double)v[k] * (double)v[k];
        ss = wave_sum_dpp(ss);
        if (lane == 0) red_d[w] = ss;
        __syncthreads();
        ss = (red_d[0] + red_d[1]) + (red_d[2] + red_d[3]);
        const float mean = (float)(ss / (double)n);
        inv = __fdiv_rn(1.0f, sqrt_rn_f32(__fadd_rn(mean, 1e-5f)));
#pragma unroll
        for (int k = 0; k < NK; k++) v[k] = __fmul_rn(__fmul_rn(v[k], inv), nw[k]);
    }
    float mx = 0.0f;
#pragma unroll
    for (int k = 0; k < NK; k++)
        if (tid + QG_BLOCK * k < n) mx = fmaxf(mx, fabsf(v[k]));
    mx = wave_max_f(mx);
    if (lane == 0) red_f[w] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red_f[0], red_f[1]), fmaxf(red_f[2], red_f[3]));
    int e = 0;
    if (mx > 0.0f && isfinite(mx)) {
        int k;
        (void)frexpf(mx, &k);
        e = k - 14;
    }
    if (tid == 0) ex[t] = e;
    __half *hi = sp + (size_t)t * 2 * n, *lo = hi + n;
#pragma unroll
    for (int k = 0; k < NK; k++) {
        const int i = tid + QG_BLOCK * k;
        if (i < n) {
            const float xs = ldexpf(v[k], -e);
            const __half h = __float2half_rn(xs);
            hi[i] = h;
            lo[i] = __float2half_rn(xs - __half2float(h));
        }
    }
}

// ---- the GEMM -----------------------------------------------------------------------

// Eight (or four) int8 weights as fp16, exactly: byte b becomes the fp16 with bits
// 0x64 (b ^ 0x80) = 1152 + q, and one packed subtract removes the 1152.
__device__ static inline unsigned qg_pair(unsigned u, unsigned sel) {
    return __builtin_amdgcn_perm(0x64646464u, u ^ 0x80808080u, sel);
}
__device__ static inline qg_h8 qg_i8_to_h8(unsigned lo, unsigned hi) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const unsigned w[4] = {qg_pair(lo, 0x07010700u), qg_pair(lo, 0x07030702u), qg_pair(hi, 0x07010700u),
                           qg_pair(hi, 0x07030702u)};
    qg_h8 r;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        const h2 v = __builtin_bit_cast(h2, w[k]) - off;
        r[2 * k] = v[0];
        r[2 * k + 1] = v[1];
    }
    return r;
}
__device__ static inline qg_h4 qg_i8_to_h4(unsigned u) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    const h2 off = {(_Float16)1152.0f, (_Float16)1152.0f};
    const h2 a = __builtin_bit_cast(h2, qg_pair(u, 0x07010700u)) - off;
    const h2 b = __builtin_bit_cast(h2, qg_pair(u, 0x07030702u)) - off;
    qg_h4 r = {a[0], a[1], b[0], b[1]};
    return r;
}

// One stage of the chunk pipeline in shared memory: every operand of a chunk of QG_KC
// columns arrives by DMA that the compiler does not track, so its only waits are the
// pipeline's exact vmcnt counts. (Weights loaded into registers instead make the compiler
// wait, at the pipeline loop's join, for every outstanding load, the next chunk's
// included.)
//   act  [TT tokens][2 planes][QG_KC] fp16, row r = 2 token + plane, its 16-byte groups
//        XOR-swizzled by token % 8 so that an A-operand read (16 tokens) spreads over the banks;
//   w    [NM matrices][64 rows][QG_KC] int8, row r's 16-byte groups swizzled by (r / 4) % 4;
//   s    [NM][256] fp32: row r's scales of the chunk's NB blocks at r NB + b.
template <int NM, int TT>
struct QgStageBuf {
    uint8_t act[TT * 2 * QG_RB];
    uint8_t w[NM][64 * QG_KC];
    float s[NM][QG_BLOCK];
};

// Per-thread sources of a tile's DMA: NA activation slots (16 bytes), and for each matrix
// one weight slot (16 bytes of row t / 4 of the panel) and one scale slot (4 bytes), as
// offsets of chunk 0 from the tile's first token's split row, the panel's first weight and its
// first scale; chunk kc's lie QG_KC columns (halves, weights) and QG_KC / KB scales times kc on.
template <int NA>
struct QgSrc {
    const __half *act0;             // the tile's first token, at the group's first column
    const int8_t *w0;               // first weight of the panel's first row (of the first matrix)
    const float *s0;                // first scale of the panel's first row
    ptrdiff_t dw, ds;               // the second matrix's distance
    unsigned act[NA], wo, so;       // the slots' byte offsets
    unsigned short col[NA];         // the activation slots' first columns within a chunk
    unsigned short w_col, s_blk;    // the weight slot's first column and the scale slot's group
};

template <int NA, int KB, int NM>
__device__ static inline QgSrc<NA> qg_src_init(const QgArgs &a, int t0, int c_off, int row0, int nrows) {
    const int tid = threadIdx.x & (QG_BLOCK - 1);
    const int ng = a.cols / KB;
    QgSrc<NA> g;
    g.act0 = a.xs + (size_t)t0 * 2 * a.xcols + c_off;
    g.w0 = a.q + (size_t)row0 * a.cols;
    g.s0 = a.s + (size_t)row0 * ng;
    g.dw = NM == 2 ? a.q2 - a.q : 0;
    g.ds = NM == 2 ? a.s2 - a.s : 0;
#pragma unroll
    for (int it = 0; it < NA; it++) {
        const int s = QG_BLOCK * it + tid, r = s / QG_RG, p = s % QG_RG, tok = r >> 1;
        const int j = p ^ (tok & 7);  // the slot holds logical group j of its row
        const int t = t0 + tok < a.n ? tok : a.n - 1 - t0;
        g.col[it] = 8 * j;
        g.act[it] = 2u * ((2u * t + (r & 1)) * a.xcols + 8 * j);
    }
    const int wr = tid >> 2, wg = (tid & 3) ^ ((wr >> 2) & 3);  // slot tid holds group wg of row wr
    g.w_col = 16 * wg;
    g.wo = (unsigned)(wr < nrows ? wr : 0) * a.cols + 16 * wg;
    constexpr int NB = QG_KC / KB;
    const int sr = tid / NB;  // slots past the panel's 64 rows (NB = 2) load row 0
    g.s_blk = tid % NB;
    g.so = 4u * ((unsigned)(sr < nrows ? sr : 0) * ng + tid % NB);
    return g;
}

template <int NA, int KB, int NM, int TT>
__device__ static inline void qg_issue(const QgArgs &a, const QgSrc<NA> &g, QgStageBuf<NM, TT> &sb, int c0) {
    const int w = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    const __half *act = g.act0 + c0;
    const int8_t *wq = g.w0 + c0;
    const float *ws = g.s0 + c0 / KB;
    if (c0 + QG_KC <= a.cols) {
#pragma unroll
        for (int it = 0; it < NA; it++) dma_s<16>(act, g.act[it], (const lds_void *)(sb.act + 16 * (64 * w + QG_BLOCK * it)));
#pragma unroll
        for (int m = 0; m < NM; m++) {
            dma_s<16>(wq + (m ? g.dw : 0), g.wo, (const lds_void *)(sb.w[m] + 1024 * w));
            dma_s<4>(ws + (m ? g.ds : 0), g.so, (const lds_void *)(sb.s[m] + 64 * w));
        }
        return;
    }
    // the last chunk's part past the last column: zeros for the inputs, any weights and scales
#pragma unroll
    for (int it = 0; it < NA; it++) {
        const __half *src = c0 + g.col[it] < a.cols ? (const __half *)((const char *)act + g.act[it]) : a.zeros;
        dma16_untracked(gbl((const void *)src), (lds_void *)(sb.act + 16 * (64 * w + QG_BLOCK * it)));
    }
    const unsigned wo = c0 + g.w_col < a.cols ? g.wo : g.wo - g.w_col;
    const unsigned so = c0 + KB * g.s_blk < a.cols ? g.so : g.so - 4 * g.s_blk;
#pragma unroll
    for (int m = 0; m < NM; m++) {
        dma_s<16>(wq + (m ? g.dw : 0), wo, (const lds_void *)(sb.w[m] + 1024 * w));
        dma_s<4>(ws + (m ? g.ds : 0), so, (const lds_void *)(sb.s[m] + 64 * w));
    }
}

// KB = 32: A operand of A tile i, plane pl, block b of the chunk: lane l holds token
// 16 i + l % 16, columns 32 b + 8 (l / 16) .. +8.
__device__ static inline qg_h8 qg_a8(const uint8_t *act, int i, int pl, int b) {
    const int lane = threadIdx.x & 63, tok = 16 * i + (lane & 15), r = 2 * tok + pl;
    const int j = 4 * b + (lane >> 4), p = j ^ (tok & 7);
    return *(const qg_h8 *)(act + r * QG_RB + 16 * p);
}
// KB = 16: columns 16 b + 4 (l / 16) .. +4.
__device__ static inline qg_h4 qg_a4(const uint8_t *act, int i, int pl, int b) {
    const int lane = threadIdx.x & 63, tok = 16 * i + (lane & 15), r = 2 * tok + pl;
    const int col = 16 * b + 4 * (lane >> 4), j = col >> 3, p = j ^ (tok & 7);
    return *(const qg_h4 *)(act + r * QG_RB + 16 * p + 2 * (col & 7));
}
// The lane's weight bytes of panel row r, columns c .. c + n (n = 8 or 4, inside a group).
__device__ static inline const uint8_t *qg_w(const uint8_t *w, int r, int c) {
    const int g = (c >> 4) ^ ((r >> 2) & 3);
    return w + r * QG_KC + 16 * g + (c & 15);
}

// The chunk's products: every operand is read from shared memory before the first is used (a
// read's latency is paid once a chunk, not once a block), and the MFMAs of different blocks
// and A tiles, which do not depend on each other, lie between a hi product and its lo.
template <int NA, int KB>
__device__ static inline void qg_mma(const uint8_t *act, const uint8_t *wm, const float *sm, int left, int r, float (*acc)[4]) {
    const qg_f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const int lane = threadIdx.x & 63;
    constexpr int NB = QG_KC / KB;
    typedef typename std::conditional<KB == 32, qg_h8, qg_h4>::type frag;
    typedef typename std::conditional<KB == 32, qg_u2, unsigned>::type raw;
    raw q[NB];
    float sc[NB];
    frag A[2][NB][NA];
#pragma unroll
    for (int b = 0; b < NB; b++) q[b] = *(const raw *)qg_w(wm, r, KB * b + KB / 4 * (lane >> 4));
#pragma unroll
    for (int b = 0; b < NB; b++) sc[b] = sm[r * NB + b];
#pragma unroll
    for (int pl = 0; pl < 2; pl++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int i = 0; i < NA; i++) {
                if constexpr (KB == 32) A[pl][b][i] = qg_a8(act, i, pl, b);
                else A[pl][b][i] = qg_a4(act, i, pl, b);
            }
    frag B[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        if constexpr (KB == 32) B[b] = qg_i8_to_h8(q[b].x, q[b].y);
        else B[b] = qg_i8_to_h4(q[b]);
        if (KB * b >= left) sc[b] = 0.0f;  // past the last column
    }
    qg_f4 d[NB][NA];
#pragma unroll
    for (int pl = 0; pl < 2; pl++)
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int i = 0; i < NA; i++) {
                if constexpr (KB == 32) d[b][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A[pl][b][i], B[b], pl ? d[b][i] : zero, 0, 0, 0);
                else d[b][i] = __builtin_amdgcn_mfma_f32_16x16x16f16(A[pl][b][i], B[b], pl ? d[b][i] : zero, 0, 0, 0);
            }
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) acc[i][k] = fmaf(d[b][i][k], sc[b], acc[i][k]);
}

// The tile of block (panel, token tile): wave w takes rows 16 w .. +16 of the panel. The
// chunks run double-buffered with one barrier each: a step waits for its own chunk's loads
// and for the wave's shared-memory reads of the chunk before, then on the block, after which
// that chunk's stage takes the next chunk while this one is multiplied. (Three, four and six
// stages measured no faster at 201 and 1024 tokens: what a chunk cost was its instructions.)
template <int NA, int KB, int MODE, int NM, int TT, int NH>
__device__ __attribute__((always_inline)) static void qg_tile(const QgArgs &a, int panel, int tt,
                                                             QgStageBuf<NM, TT> (&bufs)[NH][2]) {
    const int tid = threadIdx.x, lane = tid & 63;
    const int half = NH == 1 ? 0 : __builtin_amdgcn_readfirstlane(tid / QG_BLOCK), w = (tid >> 6) & 3;
    QgStageBuf<NM, TT>(&buf)[2] = bufs[half];
    const int g = panel / a.bpg, rb = panel % a.bpg;
    const int row0 = g * a.x_rows + 64 * rb;                         // the panel's first row
    const int left = min(a.x_rows - 64 * rb, a.rows - row0);
    const int nrows = left < 64 ? left : 64;                         // its rows (of 64)
    const int pr = 16 * w + (lane & 15);                             // the lane's panel row
    const bool row_on = pr < nrows;
    const int t0 = TT * tt;
    const QgSrc<NA> src = qg_src_init<NA, KB, NM>(a, t0, g * a.x_stride, row0, nrows);
    float acc[NA][4], acc2[NA][4];
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) acc[i][k] = acc2[i][k] = 0.0f;
    const int nkc = (a.cols + QG_KC - 1) / QG_KC;
    auto compute = [&](const QgStageBuf<NM, TT> &sb, int kc) {
        qg_mma<NA, KB>(sb.act, sb.w[0], sb.s[0], a.cols - kc * QG_KC, pr, acc);
        if (NM == 2) qg_mma<NA, KB>(sb.act, sb.w[NM - 1], sb.s[NM - 1], a.cols - kc * QG_KC, pr, acc2);
    };
    // half h's chunks are h, h + NH, ...
    if (half < nkc) qg_issue<NA, KB, NM, TT>(a, src, buf[0], half * QG_KC);
    for (int j = 0; j * NH < nkc; j++) {
        const int kc = j * NH + half;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        block_barrier();  // chunk kc has landed, and chunk kc - NH is done with
        if (kc + NH < nkc) qg_issue<NA, KB, NM, TT>(a, src, buf[(j + 1) & 1], (kc + NH) * QG_KC);
        if (kc < nkc) compute(buf[j & 1], kc);
    }
    if (NH == 2) {
        // the odd chunks' sums through shared memory (the stages, once every wave is done with them)
        float *x = reinterpret_cast<float *>(&bufs[0][0]) + (tid & (QG_BLOCK - 1));
        static_assert(NH == 1 || sizeof(bufs) >= sizeof(float) * 8 * NA * QG_BLOCK, "the sums fit the stages");
        __syncthreads();
        if (half == 1) {
#pragma unroll
            for (int i = 0; i < NA; i++)
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    x[QG_BLOCK * (4 * i + k)] = acc[i][k];
                    if (NM == 2) x[QG_BLOCK * (4 * (NA + i) + k)] = acc2[i][k];
                }
        }
        __syncthreads();
        if (half == 1) return;
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                acc[i][k] = __fadd_rn(acc[i][k], x[QG_BLOCK * (4 * i + k)]);
                if (NM == 2) acc2[i][k] = __fadd_rn(acc2[i][k], x[QG_BLOCK * (4 * (NA + i) + k)]);
            }
    }
    // lane l holds tokens 16 i + 4 (l / 16) + k of panel row pr
    const int r = row0 + pr;
#pragma unroll
    for (int i = 0; i < NA; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const int t = t0 + 16 * i + 4 * (lane >> 4) + k;
            if (row_on && t < a.n) {
                const int e = a.xe[t];
                const float v = ldexpf(acc[i][k], e);
                float out;
                if (MODE == QG_PAIR) {
                    const float u = ldexpf(acc2[i][k], e);
                    out = v / (1.0f + expf(-v)) * u;  // infer.c:1078-1080
                } else if (MODE == QG_RESID) {
                    out = a.resid[(size_t)t * a.ldr + r] + v;  // infer.c:1061, 1083
                } else {
                    out = v;
                }
                a.y[(size_t)t * a.ldy + r] = out;
            }
        }
}

// f(NA) with NA the tile's A-tile count (1..4, block-uniform) as a compile-time constant.
template <int N, typename Body>
__device__ __attribute__((always_inline)) static inline void qg_with_na(int na, Body &&f) {
    if constexpr (N > 1) {
        if (na < N) {
            qg_with_na<N - 1>(na, f);
            return;
        }
    }
    f(std::integral_constant<int, N>{});
}

// Grid: one block per (64-row panel, token tile), in XCD-aware order: linear block id b
// runs on XCD b % 8, which takes panels xcd, xcd + 8, ... (its weights stay in its L2); its
// blocks take token tile 0 for each of those panels, then tile 1, ..., so that the blocks
// resident together share their tokens' inputs in L2 (walking one panel's tiles before the
// next streamed the whole input once per panel: 603 MB fetched per attn_out call of a
// 1024-token batch, for 31.5 MB of weights and inputs).
// What bounds the large products is instruction issue: a chunk's eight or sixteen MFMAs take 128 or
// 256 clocks of a wave, and everything else in it has to stay near that. Counters, shares of the
// waves' cycles: gate/up of 1024 tokens at group size 32 (the matrix cores busy 33 % of the
// time, 5.4 vector instructions an MFMA) 43 % issuing, 32 % ready and not issued, 25 % waiting for
// data or a barrier; attn_out there (29 %, 5.0) 43, 28 and 29 %; gate/up of 201 tokens at group size 16
// (35 %, 4.7) 44, 30 and 26 %. The small products wait as much as they issue, too few waves being
// there: attn_out of 201 tokens (18 %, 5.8) 36, 23 and 40 %, k_b and v_b 18 to 37, 19 to 36 and 44 to
// 55 %. Hence scalar base addresses stepped
// along the rows (no vector instruction a DMA, no division by the group size), operands read
// together, the accumulators in vector registers (launch bounds that leave the matrix cores no
// use for their own, whose every read is an instruction). Before and after, us, with the rules
// below: group size 16, 201 tokens: attn_out 74 -> 41, layer 0's gate/up 137 -> 84, q_a and kv_a
// 30 + 30 -> 18; group size 32, 1024 tokens: attn_out 107 -> 79, gate/up 318 -> 240.
template <int KB, int MODE, int TT, int NH>
__global__ __launch_bounds__(QG_BLOCK *NH, NH == 2 ? 2 : TT > 32 ? (MODE == QG_PAIR || KB == 16 ? 2 : 3) : MODE == QG_PAIR ? 3 : 4)
void k_gemm_q8(QgArgs a) {
    constexpr int NM = MODE == QG_PAIR ? 2 : 1;
    __shared__ __align__(16) QgStageBuf<NM, TT> buf[NH][2];
    const int b = blockIdx.x, xcd = b % QG_XCD, k = b / QG_XCD;
    const int na_ = a.bpg * a.groups, nb_ = a.rows_b ? (a.rows_b + 63) / 64 : 0;  // panels of the matrix, of the second
    const int ppx = (na_ + nb_ + QG_XCD - 1) / QG_XCD;  // panels per XCD
    int panel = (k % ppx) * QG_XCD + xcd;
    const int tt = k / ppx;
    if (panel >= na_ + nb_) return;
    if (MODE == QG_PLAIN && panel >= na_) {  // the second product of the same inputs
        panel -= na_;
        a.q = a.q2;
        a.s = a.s2;
        a.y = a.y_b;
        a.rows = a.x_rows = a.rows_b;
        a.bpg = nb_;
        a.ldy = a.rows_b;
    }
    const int left = a.n - TT * tt;
    const int na = __builtin_amdgcn_readfirstlane(left >= TT ? TT / 16 : (left + 15) >> 4);
    qg_with_na<TT / 16>(na, [&](auto NA) { qg_tile<decltype(NA)::value, KB, MODE, NM, TT, NH>(a, panel, tt, buf); });
}

// Tokens per tile for n tokens and `panels` 64-row panels on n_cu compute units: 64 where that
// leaves every CU two blocks (a chunk's weights are converted once for twice the tokens) and the
// rows are long enough for it to tell, else 32, which is twice the blocks. Both sides round the
// lines, us, 32 and 64 tokens a tile (GLM-4.7-Flash's products):
//   blocks, gate/up (160 panels, 2048 columns; the line at 193 tokens): group size 16, 128 tokens 52.9
//     and 61.4, 201: 77.0 and 76.4, 256: 88.1 and 96.3 (640 blocks, 512 at once), 384: 135 and
//     122, 1024: 332 and 294; group size 32, 128 tokens 45.0 and 45.1, 201: 69.2 and 60.1, 1024: 277 and 228;
//   blocks, attn_out (32 panels, 5120 columns; at 961): group size 16, 896 tokens 103 and 107, 1024:
//     108 and 108; group size 32, 768 tokens 66.2 and 66.3, 896: 84.0 and 68.1, 1024: 89.2 and 73.5;
//   columns, 1024 tokens: k_b (192 columns) 29.8 and 38.9 at group size 16, 29.8 and 33.2 at 32; v_b
//     (512) 33.4 and 38.8, 31.8 and 32.2; q_b (768) 41.7 and 46.9, 33.8 and 30.8.
static inline int qg_tokens(int n, int panels, int cols, int n_cu) {
    return cols >= 1024 && (size_t)panels * ((n + 63) / 64) >= 2 * (size_t)n_cu ? 64 : 32;
}
// Whether the 32-token tiles' blocks run two halves of four waves, each every other chunk: where
// there are too few blocks to give each SIMD two waves of them, which hide each other's waits. Us
// with one and two halves: attn_out at group size 16, 16 tokens 37.8 and 27.3, 256: 48.6 and 37.9,
// 448 (448 blocks) 56.6 and 57.9, 512 (512 blocks, the line) 59.4 and 60.2; at group size 32, 256
// tokens 44.1 and 38.5, 448: 51.2 and 44.6, 512: 53.2 and 46.6; q_a and kv_a in one launch, 201 tokens 21.2
// and 17.4 (19.4 and 15.4 at group size 32), 768 (504 blocks) 33.2 and 37.4. Short rows cross earlier:
// v_b (512 columns), 96 tokens (240 blocks) 8.6 and 7.8, 160 (400) 10.1 and 11.2.
static inline bool qg_halves(int n, int panels, int n_cu) { return (size_t)panels * ((n + 31) / 32) < 2 * (size_t)n_cu; }
