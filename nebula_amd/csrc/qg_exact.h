// Products in the reference's fixed summation order on the fp32 matrix cores:
// out[t][r] = sum_k W[r][k] x[t][k] where chain j (0..31) adds k = j, j + 32,
// ... in ascending k with one fused multiply-add each, then the tree
// 16/8/4/2/1 joins the 32 chains (cpu.c:122-139, gpu.cu:154-180).  Each of an
// output's chains is a sequence of rank-1 updates over one k per step, and
// v_mfma_f32_16x16x1_4b_f32 is one such step for four chains of a 16 x 16
// output tile: with K = 1 every output element is a single fused
// multiply-add, rounded once, so the results equal the scalar chains bit for
// bit (subnormals, signed zeros and infinities included).
//
// Used by qg_matmul (qg_ops.hip) and by the prefill router (qg_prefill.hip).
#pragma once
#include "qg_frag.h"

typedef float qg_f16v __attribute__((ext_vector_type(16)));

// A tile is TOK = 16 N16 + 4 N4 tokens x 16 RR weight rows; K streams in
// stages of CH chunks of 128 columns (4 steps of every chain).  The
// workgroup's 8 waves split the chains: wave w owns chains 2w, 2w + 1, 2w +
// 16, 2w + 17 (the four blocks of its MFMAs) for the whole tile, so every
// weight is decoded by exactly one lane, straight into its operand register,
// the tree's first level (stride 16) joins a wave's own accumulators and its
// last (stride 1) a lane's pair.
//
// Shared memory: token rows (and F32 weight rows) as fp32 in column order, row
// r's 16-byte unit m (of 8 per step) at position m ^ (r & 7) of its step, so
// the rows of an operand read hit different banks; they arrive by 16-byte
// direct copies, XR stages in a ring.  The quantised rows stay raw bytes (RB
// per 256 columns, a multiple of 16), RS superblocks in a ring; each wave
// copies 2 RR rows and forms their scales (Q4_K: d*s and -(dmin*m) per group;
// IQ4_NL, Q8_0: d per block) in fp32 one superblock ahead.
// RB: row bytes per 256 columns; TF: floats per row of a superblock's scales,
// padded so that the rows of a read start in distinct banks.
template <int TYPE> struct XmRaw;
template <> struct XmRaw<QT_F32> { static constexpr int RB = 0, TF = 0; };
template <> struct XmRaw<QT_Q4_K> { static constexpr int RB = 144, TF = 20; };
template <> struct XmRaw<QT_IQ4_NL> { static constexpr int RB = 144, TF = 12; };
template <> struct XmRaw<QT_Q8_0> { static constexpr int RB = 272, TF = 12; };

template <int TYPE, int N16, int N4, int RR, int CH, int XR, int RS>
struct XmShape {
    static constexpr int TOK = 16 * N16 + 4 * N4, ROWS = 16 * RR, RB = XmRaw<TYPE>::RB, TF = XmRaw<TYPE>::TF;
    static constexpr int WROWS = 2 * RR;                                       // weight rows copied by one wave
    static constexpr int XB = CH * TOK * 512, WB = RB ? 0 : CH * ROWS * 512;   // bytes of one stage's tokens / F32 weights
    static constexpr int RAW = ROWS * RB, TAB = ROWS * TF * 4;                 // bytes of one superblock's raw rows / scales
    static constexpr int RED = 8 * TOK * ROWS * 8;                             // partial sums of the epilogue
    static constexpr int BUF = XR * (XB + WB) + RS * RAW + 2 * TAB;
    static constexpr int LDS = BUF > RED ? BUF : RED;
};

struct XmArgs {
    float *out; int ldo;                  // out[t * ldo + r]
    const uint8_t *w; size_t stride;      // weight rows
    int rows, cols;                       // cols a multiple of 128 CH (F32) or 256
    const float *x; int nt;
    const float *bias;                    // added to the finished sums, or null
    int ntt, nrt;                         // token tiles, row tiles
};

// Workgroup -> tile: each XCD (workgroup b runs on XCD b % 8) takes one run
// of the tiles, ordered in groups of up to 8 token tiles x every row tile, so
// the tiles that run together on an XCD share its L2's copy of their rows.
QG_DEV void xm_tile(int b, int ntt, int nrt, int &tt, int &rt) {
    const int n = ntt * nrt, q = n / 8, rem = n % 8, xcd = b % 8;
    const int i = xcd * q + min(xcd, rem) + b / 8;
    const int g = i / (8 * nrt), gw = min(8, ntt - 8 * g), k = i - g * 8 * nrt;
    tt = 8 * g + k % gw;
    rt = k / gw;
}

template <int TYPE, int N16, int N4, int RR, int CH, int XR, int RS, int OCC>
__global__ __launch_bounds__(512, OCC) void xm_kernel(XmArgs A) {
    using S = XmShape<TYPE, N16, N4, RR, CH, XR, RS>;
    constexpr int TOK = S::TOK, ROWS = S::ROWS, RB = S::RB, TF = S::TF;
    constexpr int NX = (TOK + 15) / 16, NW = RB ? 0 : RR;   // 16-byte copies per wave and chunk
    extern __shared__ uint4 s_dyn[];
    constexpr bool LUT = TYPE == QT_IQ4_NL && N16 >= 2;
    __shared__ float s_lut[LUT ? 16 : 1];
    if (LUT && threadIdx.x < 16) s_lut[threadIdx.x] = (float)qg_iq4nl_lut[threadIdx.x];
    uint8_t *lds = (uint8_t *)s_dyn;
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // two wide workgroups share a CU and would run their operand reads and
    // their products in step; a standing difference in priority lets one's
    // products run under the other's reads (z 6144 x 2560, 2048 tokens: 731 ->
    // 720 us)
    if (N16 >= 2 && ((blockIdx.x >> 8) & 1)) __builtin_amdgcn_s_setprio(1);
    int tt, rt;
    xm_tile(blockIdx.x, A.ntt, A.nrt, tt, rt);
    const int t0 = tt * TOK, r0 = rt * ROWS, n = min(TOK, A.nt - t0), nr = min(ROWS, A.rows - r0);
    const int nst = A.cols / (128 * CH), nsb = A.cols / 256;
    float *xs = (float *)lds, *ws = (float *)(lds + XR * S::XB);
    uint8_t *raw = lds + XR * (S::XB + S::WB);
    float *tab = (float *)(raw + RS * S::RAW);

    // A chunk of R rows is 32 R units, 4 R of them per wave: copy i fills
    // units 4 R wave + 64 i + lane; unit position u of a row holds step u / 8,
    // unit (u % 8) ^ (row & 7).  Rows past the tile's end repeat its last one.
    auto src_off = [&](int first, int last) {
        const int U = first + lane, row = U >> 5, u = U & 31, m = (u & 7) ^ (row & 7);
        return (uint32_t)min(row, last) * (uint32_t)A.cols * 4u + (uint32_t)((u >> 3) * 128 + m * 16);
    };
    uint32_t xo[NX], wo[NW ? NW : 1];
#pragma unroll
    for (int i = 0; i < NX; i++) xo[i] = src_off(4 * TOK * wave + 64 * i, n - 1);
#pragma unroll
    for (int i = 0; i < NW; i++) wo[i] = src_off(4 * ROWS * wave + 64 * i, nr - 1);
    const uint8_t *xb = (const uint8_t *)(A.x + (size_t)t0 * A.cols), *wb = A.w + (size_t)r0 * A.stride;
    // stage c (past the last: the last again, into a slot that nobody reads)
    auto copy_stage = [&](int c) {
        const int slot = c % XR, cc = min(c, nst - 1);
#pragma unroll
        for (int q = 0; q < CH; q++) {
#pragma unroll
            for (int i = 0; i < NX; i++)
                if (64 * (i + 1) <= 4 * TOK || lane < 4 * TOK - 64 * i)
                    dma16_scalar(xo[i], xb + (size_t)(cc * CH + q) * 512, xs + (slot * CH + q) * (TOK * 128) + 4 * (4 * TOK * wave + 64 * i));
#pragma unroll
            for (int i = 0; i < NW; i++)
                dma16_scalar(wo[i], wb + (size_t)(cc * CH + q) * 512, ws + (slot * CH + q) * (ROWS * 128) + 4 * (4 * ROWS * wave + 64 * i));
        }
    };
    // raw superblock s: the wave's rows v (row 16 (v / 2) + 2 wave + v % 2)
    constexpr int PC = RB ? RB / 16 : 1;
    uint32_t ro = 0;
    if constexpr (RB != 0) {
        const int v = min(lane / PC, S::WROWS - 1), r = 16 * (v >> 1) + 2 * wave + (v & 1);
        ro = (uint32_t)min(r, nr - 1) * (uint32_t)A.stride + (uint32_t)(lane % PC) * 16u;
    }
    auto copy_raw = [&](int s) {
        if constexpr (RB != 0) {
            if (lane < S::WROWS * PC) dma16_scalar(ro, wb + (size_t)min(s, nsb - 1) * RB, raw + (s % RS) * S::RAW + wave * (S::WROWS * RB));
        }
    };
    // the scales of the wave's rows in superblock s
    auto scales = [&](int s) {
        if constexpr (RB != 0) {
            if (lane < S::WROWS * 8) {
                const int v = lane >> 3, g = lane & 7, r = 16 * (v >> 1) + 2 * wave + (v & 1);
                const uint8_t *p = raw + (s % RS) * S::RAW + (wave * S::WROWS + v) * RB;
                float *d = tab + (s & 1) * (ROWS * TF) + r * TF;
                if constexpr (TYPE == QT_Q4_K) {
                    const uint8_t *sc = p + 4;
                    const int b0 = sc[g], b4 = sc[4 + g], bm = sc[g & 3], b1 = sc[4 + (g & 3)];
                    const float ds = qg_half_u16(*(const uint16_t *)p), dmin = qg_half_u16(*(const uint16_t *)(p + 2));
                    const int sv = g < 4 ? (b0 & 63) : ((b4 & 15) | ((bm >> 6) << 4));
                    const int mv = g < 4 ? (b4 & 63) : ((b4 >> 4) | ((b1 >> 6) << 4));
                    *(float2 *)(d + 2 * g) = make_float2(ds * (float)sv, -(dmin * (float)mv));
                } else {
                    d[g] = qg_half_u16(*(const uint16_t *)(p + RB / 8 * g));
                }
            }
        }
    };

    // operands: row l % 16 of a 16-row tile, chain 2 wave + blk % 2 + 16 (blk
    // / 2) with blk = l / 16; a 4-token tile's lanes take token l % 4.  fo:
    // step 0 of the row's fp32 values (step i is 32 floats on)
    const int cu = (wave >> 1) + 4 * (lane >> 5), cd = 2 * (wave & 1) + ((lane >> 4) & 1), chain = 4 * cu + cd;
    const int fo = (lane & 15) * 128 + 4 * (cu ^ (lane & 7)) + cd;
    const int fo4[2] = {(lane & 3) * 128 + 4 * (cu ^ (lane & 3)) + cd, (lane & 3) * 128 + 4 * (cu ^ (4 + (lane & 3))) + cd};
    const int rawo = ((lane & 15) >> 1) * (S::WROWS * RB) + (lane & 1) * RB;  // the lane's row in a raw superblock (+ 2 rr RB)
    // the lane's weights of chunk c (128 columns): 4 steps of its chain per row tile
    auto weights = [&](int c, float (&b)[4][RR]) {
        if constexpr (RB != 0) {
            const int s = c >> 1, h = c & 1;
            const uint8_t *rs = raw + (s % RS) * S::RAW + rawo;
            const float *tb = tab + (s & 1) * (ROWS * TF) + (lane & 15) * TF;
#pragma unroll
            for (int r = 0; r < RR; r++) {
                const uint8_t *p = rs + 2 * r * RB;
                if constexpr (TYPE == QT_Q4_K) {
                    const uint32_t q0 = p[16 + 64 * h + chain], q1 = p[48 + 64 * h + chain];
                    const float4 s01 = *(const float4 *)(tb + r * (16 * TF) + 8 * h), s23 = *(const float4 *)(tb + r * (16 * TF) + 8 * h + 4);
                    b[0][r] = __builtin_fmaf(s01.x, (float)(q0 & 15u), s01.y);
                    b[1][r] = __builtin_fmaf(s01.z, (float)(q0 >> 4), s01.w);
                    b[2][r] = __builtin_fmaf(s23.x, (float)(q1 & 15u), s23.y);
                    b[3][r] = __builtin_fmaf(s23.z, (float)(q1 >> 4), s23.w);
                } else if constexpr (TYPE == QT_Q8_0) {
                    const int8_t *k = (const int8_t *)(p + 136 * h + 2 + chain);
                    const float4 d = *(const float4 *)(tb + r * (16 * TF) + 4 * h);
                    b[0][r] = d.x * (float)k[0];
                    b[1][r] = d.y * (float)k[34];
                    b[2][r] = d.z * (float)k[68];
                    b[3][r] = d.w * (float)k[102];
                } else {
                    // chains below 16 are the low nibbles of a block's bytes
                    const uint8_t *k = p + 72 * h + 2 + (chain & 15);
                    const uint32_t sh = 4 * (lane >> 5);
                    const float4 d = *(const float4 *)(tb + r * (16 * TF) + 4 * h);
                    if constexpr (N16 >= 2) {  // fewer vector instructions (6144 x 2560, 2048 tokens: 832 -> 799 us)
                        b[0][r] = d.x * s_lut[(k[0] >> sh) & 15];
                        b[1][r] = d.y * s_lut[(k[18] >> sh) & 15];
                        b[2][r] = d.z * s_lut[(k[36] >> sh) & 15];
                        b[3][r] = d.w * s_lut[(k[54] >> sh) & 15];
                    } else {                   // no second trip to shared memory
                        uint32_t q = k[0] | ((uint32_t)k[18] << 8) | ((uint32_t)k[36] << 16) | ((uint32_t)k[54] << 24);
                        q = iq4_lookup((q >> sh) & 0x0F0F0F0Fu);  // table value + 128 per byte
                        b[0][r] = d.x * ((float)(q & 0xffu) - 128.0f);
                        b[1][r] = d.y * ((float)((q >> 8) & 0xffu) - 128.0f);
                        b[2][r] = d.z * ((float)((q >> 16) & 0xffu) - 128.0f);
                        b[3][r] = d.w * ((float)(q >> 24) - 128.0f);
                    }
                }
            }
        }
    };
    qg_f16v acc[N16 ? N16 : 1][RR];
    qg_f4 acc4[N4 ? N4 : 1][RR];
#pragma unroll
    for (int t = 0; t < N16; t++)
#pragma unroll
        for (int r = 0; r < RR; r++)
#pragma unroll
            for (int i = 0; i < 16; i++) acc[t][r][i] = 0.0f;
#pragma unroll
    for (int t = 0; t < N4; t++)
#pragma unroll
        for (int r = 0; r < RR; r++) acc4[t][r] = qg_f4{0.0f, 0.0f, 0.0f, 0.0f};

    // Raw superblocks are copied RD ahead, stages XR - 1 ahead, the stage
    // first.  Copies complete in issue order: the wait that ends iteration c
    // leaves the copies issued after stage c + 1's.  Superblock s is used from
    // iteration 2 s (CH 1) or s (CH 2) on and its scales are formed in the
    // iteration before, which RD and the waits allow for.
    constexpr int RD = RS - 1;
    static_assert(!RB || (CH == 2 ? RD >= XR + 1 : RD >= 2), "raw ring depth");
    static_assert(XR == 2 || XR == 3, "stage ring depth");
    static_assert(S::WROWS * PC <= 64, "a wave copies its raw rows with one instruction");
    constexpr int ST = CH * (NX + NW);   // copies per wave and stage
    if constexpr (RB != 0) {
#pragma unroll
        for (int s = 0; s < RD; s++) copy_raw(s);
    }
#pragma unroll
    for (int c = 0; c < XR - 1; c++) copy_stage(c);
    wait_vmem_but<(XR - 2) * ST>();
    scales(0);
    __syncthreads();
    for (int c = 0; c < nst; c++) {
        copy_stage(c + XR - 1);
        if constexpr (RB != 0) {
            if (CH == 2) copy_raw(c + RD);
            else if ((c & 1) == 0) copy_raw((c >> 1) + RD);
        }
#pragma unroll
        for (int q = 0; q < CH; q++) {
            const float *X = xs + ((c % XR) * CH + q) * (TOK * 128), *W = ws + ((c % XR) * CH + q) * (ROWS * 128);
            float b[4][RR], a[4][N16 ? N16 : 1], a4[4][N4 ? N4 : 1];
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int t = 0; t < N16; t++) a[i][t] = X[t * 2048 + fo + 32 * i];
#pragma unroll
                for (int t = 0; t < N4; t++) a4[i][t] = X[N16 * 2048 + t * 512 + fo4[t & 1] + 32 * i];
                if constexpr (RB == 0) {
#pragma unroll
                    for (int r = 0; r < RR; r++) b[i][r] = W[r * 2048 + fo + 32 * i];
                }
            }
            weights(c * CH + q, b);
            // a small IQ4_NL tile's operands are ready before the first product
            // (17 tokens, 2560 x 6144: 27.2 -> 25.3 us; Q4_K, Q8_0 and the wide
            // tiles lose by it)
            if (TYPE == QT_IQ4_NL && N16 < 2) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int t = 0; t < N16; t++)
#pragma unroll
                    for (int r = 0; r < RR; r++) acc[t][r] = __builtin_amdgcn_mfma_f32_16x16x1f32(a[i][t], b[i][r], acc[t][r], 0, 0, 0);
#pragma unroll
                for (int t = 0; t < N4; t++)
#pragma unroll
                    for (int r = 0; r < RR; r++) acc4[t][r] = __builtin_amdgcn_mfma_f32_4x4x1f32(a4[i][t], b[i][r], acc4[t][r], 0, 0, 0);
            }
        }
        if constexpr (RB != 0) {  // past the last superblock: its copy again, never read
            if (CH == 2) scales(c + 1);
            else if (c & 1) scales((c >> 1) + 1);
        }
        constexpr int LEFT = (XR - 2) * ST;
        if constexpr (RB == 0) {
            wait_vmem_but<LEFT>();
        } else if constexpr (CH == 2) {
            wait_vmem_but<LEFT + XR - 1>();
        } else if constexpr (XR == 3) {
            wait_vmem_but<LEFT + 1>();
        } else {
            if ((c & 1) == 0) wait_vmem_but<1>();
            else wait_vmem_but<0>();
        }
        __syncthreads();
    }
    wait_vmem();
    __syncthreads();
    // the tree: stride 16 within the wave, 8, 4 and 2 across the waves, 1 last
    float2 *red = (float2 *)lds;
#pragma unroll
    for (int t = 0; t < N16; t++)
#pragma unroll
        for (int r = 0; r < RR; r++)
#pragma unroll
            for (int q = 0; q < 4; q++)
                red[(wave * TOK + 16 * t + 4 * (lane >> 4) + q) * ROWS + 16 * r + (lane & 15)] =
                    make_float2(acc[t][r][q] + acc[t][r][8 + q], acc[t][r][4 + q] + acc[t][r][12 + q]);
#pragma unroll
    for (int t = 0; t < N4; t++)
#pragma unroll
        for (int r = 0; r < RR; r++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float v = acc4[t][r][i] + __shfl_xor(acc4[t][r][i], 32);  // blocks 0 + 2, 1 + 3
                const float o = __shfl_xor(v, 16);
                if (lane < 16) red[(wave * TOK + 16 * N16 + 4 * t + i) * ROWS + 16 * r + lane] = make_float2(v, o);
            }
    __syncthreads();
    for (int o = tid; o < TOK * ROWS; o += 512) {
        float2 v[8];
#pragma unroll
        for (int k = 0; k < 8; k++) v[k] = red[k * (TOK * ROWS) + o];
        const int t = o / ROWS, r = o % ROWS;
        const float e = ((v[0].x + v[4].x) + (v[2].x + v[6].x)) + ((v[1].x + v[5].x) + (v[3].x + v[7].x));
        float sum = e + (((v[0].y + v[4].y) + (v[2].y + v[6].y)) + ((v[1].y + v[5].y) + (v[3].y + v[7].y)));
        if (t < n && r < nr) {
            if (A.bias) sum += A.bias[r0 + r];
            A.out[(size_t)(t0 + t) * A.ldo + r0 + r] = sum;
        }
    }
}

// Estimated cost of a launch of tiles of `tr` rows x `tt` tokens, in tenths of
// one full round of the small tile (16 x 16, 3 workgroups per CU), fitted to
// 2560-column timings: the small tile in rounds of 768 workgroups; the wide
// ones (32 x 32, 16 x 64; 2 per CU, half the operand reads and decoding per product)
// in rounds of 512 that take twice as long (31 against 16 us), 1.4 times while
// every CU has one (22 us).
static inline long xm_cost(int rows, int nt, int tr, int tt) {
    const long b = (long)((rows + tr - 1) / tr) * ((nt + tt - 1) / tt);
    if (tr * tt == 256) return 10 * ((b + 767) / 768);
    return b <= 256 ? 14 : 20 * ((b + 511) / 512);
}
// Whether 32 x 32 tiles are faster than 16 x 16: where they save rounds (Q4_K
// 6144 x 2560, 300 tokens: 126 against 163 us), and not where they leave CUs idle
// (IQ4_NL 2560 x 6144, 33 tokens: 34 against 55 us).
static inline bool xm_wide(int rows, int nt) { return xm_cost(rows, nt, 32, 32) <= xm_cost(rows, nt, 16, 16); }

// Token tiles per launch (at least 1) of a matrix with nrt row tiles.
static inline int xm_slice(int nrt) {
    constexpr int TILES = (1 << 23) - 1;
    const int n = TILES / nrt;
    return n < 1 ? 1 : n > QG_MAX_TOKENS ? QG_MAX_TOKENS : n;
}
// A launch holds fewer than 2^32 threads, 2^23 tiles: more (Q8_0 outputs of 2^31 and
// more elements) go out in slices of whole token tiles.  Rows alone stay below
// that (a matrix of 2^27 rows is past what the vector chains' launch takes, too).
template <int TYPE, int N16, int N4, int RR, int CH, int XR, int RS, int OCC>
void xm_run(XmArgs A, hipStream_t s) {
    using S = XmShape<TYPE, N16, N4, RR, CH, XR, RS>;
    A.nrt = (A.rows + S::ROWS - 1) / S::ROWS;
    const int nt = A.nt, most = xm_slice(A.nrt) * S::TOK;
    for (int t = 0; t < nt; t += most) {
        A.nt = nt - t < most ? nt - t : most;
        A.ntt = (A.nt + S::TOK - 1) / S::TOK;
        xm_kernel<TYPE, N16, N4, RR, CH, XR, RS, OCC><<<A.ntt * A.nrt, 512, S::LDS, s>>>(A);
        A.out += (size_t)most * A.ldo;
        A.x += (size_t)most * A.cols;
    }
}
