// Grouped products of short row lists: the prefill's gate/up and down for
// batches whose experts have few rows each, where an item's time is that of
// streaming and converting its weights.
//
// pf_gateup_kernel / pf_down_iq_kernel stage 64-row tiles and spend about 300
// instructions of every wave per 32 weight rows x 128 K columns whatever the
// tile's rows.  Here a tile is 8 rows, whose hi and lo planes are the 16 rows
// of one MFMA, and up to TM tiles keep their activation fragments in registers
// for a whole run of weight blocks, so a block costs its conversion (once) and
// one MFMA per 32 columns and tile, with no activation traffic and no K steps.
//
// Work is dealt as equal shares of one sequence: groups in expert order (the
// empty ones left out, the shared expert last), a group's rows cut into runs
// of up to 8 TM rows, a run's weight rows into units; a unit of a run with T
// tiles is priced SP_C0 + T.  Neighbouring shares go to one XCD, so the runs
// of one expert share its L2.
#pragma once
#include "qg_frag.h"
#include <type_traits>

constexpr int SP_C0 = 2;            // price of a unit's copies and conversion, in tiles' products
constexpr int SP_NG = QG_EXPERTS + 1;

// The list of groups, built by every workgroup from the CSR offsets (512
// counts: cheaper than another launch), and this workgroup's share: positions
// (group x of the list, its run, unit, unit number in the sequence) of its
// first unit and of the next share's.  The prefix sums of price and runs that
// find the share are scratch of the build.
struct SpList { uint16_t xe[SP_NG + 1]; int nx, pos[2][4], wave[3][16]; };
constexpr int SP_SCRATCH = 2 * (SP_NG + 1) * 4;   // bytes of the build's prefix sums

// rows of group e: first CSR row (shared expert: first token) and count
QG_DEV int2 sp_rows(const int *s_off, int e, int nt) {
    return e == QG_EXPERTS ? make_int2(0, nt) : make_int2(s_off[e], s_off[e + 1] - s_off[e]);
}

// Fills the list (all NT threads of the block; s_off filled and visible;
// scratch: SP_SCRATCH bytes, free again on return) and finds part `part` of
// `parts` of the sequence.
template <int NT, int TM>
QG_DEV void sp_build(SpList &S, void *scratch, const int *s_off, int nt, bool shared, int units, int part, int parts) {
    constexpr int PER = (QG_EXPERTS + NT - 1) / NT, NWV = NT / 64;
    int *s_cost = (int *)scratch, *s_runs = s_cost + SP_NG + 1;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int v[3] = {0, 0, 0}, n_[PER];  // non-empty groups, cost, runs of the thread's experts
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int e = tid * PER + i, n = e < QG_EXPERTS ? s_off[e + 1] - s_off[e] : 0;
        n_[i] = n;
        const int runs = (n + 8 * TM - 1) / (8 * TM);
        v[0] += n > 0;
        v[1] += SP_C0 * runs + (n + 7) / 8;
        v[2] += runs;
    }
    int in[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        in[c] = v[c];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(in[c], d);
            if (lane >= d) in[c] += o;
        }
        if (lane == 63) S.wave[c][wv] = in[c];
    }
    __syncthreads();
    int ex[3], tot[3];
#pragma unroll
    for (int c = 0; c < 3; c++) {
        int b = 0, t = 0;
#pragma unroll
        for (int w = 0; w < NWV; w++) {
            const int k = S.wave[c][w];
            if (w < wv) b += k;
            t += k;
        }
        ex[c] = b + in[c] - v[c];
        tot[c] = t;
    }
#pragma unroll
    for (int i = 0; i < PER; i++) {
        const int n = n_[i];
        if (n > 0) {
            S.xe[ex[0]] = (uint16_t)(tid * PER + i);
            s_cost[ex[0]] = ex[1];
            s_runs[ex[0]] = ex[2];
            const int runs = (n + 8 * TM - 1) / (8 * TM);
            ex[0]++;
            ex[1] += SP_C0 * runs + (n + 7) / 8;
            ex[2] += runs;
        }
    }
    if (tid == 0) {
        int nx = tot[0], c = tot[1], r = tot[2];
        if (shared) {
            S.xe[nx] = QG_EXPERTS;
            s_cost[nx] = c;
            s_runs[nx] = r;
            const int runs = (nt + 8 * TM - 1) / (8 * TM);
            nx++;
            c += SP_C0 * runs + (nt + 7) / 8;
            r += runs;
        }
        s_cost[nx] = c;
        s_runs[nx] = r;
        S.nx = nx;
    }
    __syncthreads();
    const int nx = S.nx;
    const long long total = (long long)s_cost[nx] * units;
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const long long q = total * (part + k) / parts;
        if (q >= total) {
            if (tid == 0) { S.pos[k][0] = nx; S.pos[k][1] = S.pos[k][2] = 0; S.pos[k][3] = s_runs[nx] * units; }
            continue;
        }
        for (int x = tid; x < nx; x += NT) {
            const long long c0 = (long long)s_cost[x] * units, c1 = (long long)s_cost[x + 1] * units;
            if (q < c0 || q >= c1) continue;
            int rem = (int)(q - c0);
            const int n = sp_rows(s_off, S.xe[x], nt).y, runs = s_runs[x + 1] - s_runs[x];
            const int full = units * (SP_C0 + TM);
            int tau = min(rem / full, runs - 1);
            rem -= tau * full;
            const int T = tau < runs - 1 ? TM : (n + 7) / 8 - TM * (runs - 1);
            int u = (rem + SP_C0 + T - 1) / (SP_C0 + T), xx = x;
            if (u >= units) {
                u = 0;
                if (++tau == runs) { tau = 0; xx++; }
            }
            S.pos[k][0] = xx;
            S.pos[k][1] = tau;
            S.pos[k][2] = u;
            S.pos[k][3] = (s_runs[x] + (xx == x ? tau : runs)) * units + u;
        }
    }
    __syncthreads();
}

// The run at (x, tau): its group, first row (CSR position; shared expert:
// token), rows (1 .. 8 TM), tiles, and the runs of its group.
struct SpItem { int e, base, n, T, runs; };
template <int TM>
QG_DEV SpItem sp_item(const SpList &S, const int *s_off, int nt, int x, int tau) {
    SpItem it;
    it.e = __builtin_amdgcn_readfirstlane(S.xe[x]);
    const int2 r = sp_rows(s_off, it.e, nt);
    const int all = __builtin_amdgcn_readfirstlane(r.y);
    it.base = __builtin_amdgcn_readfirstlane(r.x) + 8 * TM * tau;
    it.n = min(8 * TM, all - 8 * TM * tau);
    it.T = (it.n + 7) >> 3;
    it.runs = (all + 8 * TM - 1) / (8 * TM);
    return it;
}

// The workgroup's part: neighbouring parts on one XCD (workgroup b runs on
// XCD b % 8).
QG_DEV int sp_part() {
    const int b = blockIdx.x, G = gridDim.x;
    return G % 8 ? b : (b % 8) * (G / 8) + b / 8;
}

// A fragment that the compiler must hold from here on (it waits for the load
// here, not behind copies that it does not count).
QG_DEV void sp_pin(qg_half8 &f) {
    qg_i4 v = __builtin_bit_cast(qg_i4, f);
    asm volatile("" : "+v"(v));
    f = __builtin_bit_cast(qg_half8, v);
}
QG_DEV void sp_pin(float2 &f) { asm volatile("" : "+v"(f.x), "+v"(f.y)); }

// FULL (decode batches, which take the place of the generic kernels and keep
// their arithmetic): the group sums of x and of mid in fp32 and SwiGLU with
// qg_expf and a division, where prefill has two fp16 values and the hardware's
// exponential and reciprocal.  The sums of 32 values of one sign then reach
// past 65504, as the values' own planes do.
template <bool FULL> using SpMin = std::conditional_t<FULL, MinF32, MinPlanes>;

// ---- gate/up: K split over the waves ----
// Wave w (of W = D / 256) multiplies superblock w of a sub-unit's 16 gate and 16
// up rows (144 bytes each, copied two sub-units ahead into the wave's ring of
// three slots, row r's 9 pieces rotated by r / 8 for the banks).  The partial
// sums of up to NB sub-units meet in shared memory before a barrier, after
// which 2 T waves per sub-unit apply SwiGLU, so that with one tile the products
// of four sub-units run without a barrier and every wave has a share of their
// epilogue.  A unit is 32 F rows (two sub-units), the group of a Q4_K down's
// min term.
constexpr int SP_SLOT = 32 * 9;     // 16-byte pieces of a sub-unit's rows per wave
constexpr int SP_CPB = 6;           // copies per sub-unit and wave
template <int W, int TM> struct SpGu {
    // tile slots of the partial sums: what 160 KB leave beside the rings
    static constexpr int TS = W == 8 ? 6 : 2;
    static constexpr int RING = W * 3 * SP_SLOT * 16, RED = W * 2 * TS * 64 * 8, LDS = RING + RED;
    static_assert(W >= 2 * TM && TS >= TM, "a wave per tile and token of a lane pair");
    // sub-units per barrier with M tiles
    static constexpr int batch(int M) { return min_(min_(4, TS) / M, W / (2 * M)) > 0 ? min_(min_(4, TS) / M, W / (2 * M)) : 1; }
    static constexpr int min_(int a, int b) { return a < b ? a : b; }
};

struct SpGuArgs {
    int nt, D, F;
    const int *offsets, *row_token;
    const uint8_t *gate, *up, *sh_gate, *sh_up; size_t rb;   // Q4_K rows of D
    const _Float16 *xp, *xsp;
    _Float16 *midp, *msp;            // [rows][2][F] (down format order), [rows][2][F/32] (FULL: fp32 [rows][F/32], as xsp)
    int down_fmt, sh_down_fmt;
    const int *tiles;                // if not null, *tiles: the 64-row tiles have the batch
};

// Returns false, with nothing done, where the 64-row tiles have the batch.
template <int W, int TM, bool FULL>
QG_DEV bool gateup_sp(const SpGuArgs &A) {
    extern __shared__ uint4 s_dyn[];
    __shared__ SpList S;
    __shared__ int s_off[QG_EXPERTS + 1];
    __shared__ float s_gs[W][4];   // 16-row sums of the jobs' tile rows (Q4_K down format)
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, kq = lane >> 4;
    const int tiles = A.tiles ? *A.tiles : 0;   // arrives with the offsets
    for (int i = tid; i <= QG_EXPERTS; i += 64 * W) s_off[i] = A.offsets[i];
    __syncthreads();
    if (tiles) return false;
    using MIN = SpMin<FULL>;
    const int D = A.D, F = A.F, nsr = F / 16;   // sub-units per run
    const int fmts = A.down_fmt | A.sh_down_fmt << 8;   // (chosen between by address, they keep A in scratch)
    sp_build<64 * W, TM>(S, s_dyn, s_off, A.nt, A.sh_gate != nullptr, F / 32, sp_part(), gridDim.x);
    const int nsub = 2 * __builtin_amdgcn_readfirstlane(S.pos[1][3] - S.pos[0][3]);
    if (nsub <= 0) return true;  // block-uniform
    uint4 *ring = s_dyn + (size_t)wave * 3 * SP_SLOT;
    float2 *red = (float2 *)(s_dyn + SpGu<W, TM>::RING / 16);

    // copies: piece 64 i + lane of a slot, at c_off[i] from its matrix's first
    // row of the sub-unit; pieces 0..143 are gate rows, the others up rows, so
    // piece run 2 goes out as two copies of 16 and 48 lanes
    uint32_t c_off[5];
#pragma unroll
    for (int i = 0; i < 5; i++) {
        const int sl = min(i * 64 + lane, SP_SLOT - 1), row = sl / 9, pc = sl - 9 * row, rot = row >> 3;
        c_off[i] = (uint32_t)((row & 15) * A.rb) + (uint32_t)(wave * 144 + 16 * (pc - rot + (pc < rot ? 9 : 0)));
    }
    int cx = __builtin_amdgcn_readfirstlane(S.pos[0][0]), ctau = __builtin_amdgcn_readfirstlane(S.pos[0][1]);
    int csub = 2 * __builtin_amdgcn_readfirstlane(S.pos[0][2]), cruns = 0;
    int x = cx, tau = ctau, sub = csub;
    const uint8_t *bg = nullptr, *bu = nullptr;   // gate and up rows of the sub-unit to copy next
    auto set_copy = [&]() {
        const SpItem it = sp_item<TM>(S, s_off, A.nt, cx, ctau);
        cruns = it.runs;
        const bool sh = it.e == QG_EXPERTS;
        const size_t at = (size_t)csub * 16 * A.rb;
        bg = (sh ? A.sh_gate : A.gate + (size_t)it.e * F * A.rb) + at;
        bu = (sh ? A.sh_up : A.up + (size_t)it.e * F * A.rb) + at;
    };
    auto copy_next = [&](int slot) {
        uint4 *dst = ring + slot * SP_SLOT;
        dma16_scalar(c_off[0], bg, dst);
        dma16_scalar(c_off[1], bg, dst + 64);
        if (lane < 16) dma16_scalar(c_off[2], bg, dst + 128);
        else dma16_scalar(c_off[2], bu, dst + 128);
        dma16_scalar(c_off[3], bu, dst + 192);
        if (lane < SP_SLOT - 256) dma16_scalar(c_off[4], bu, dst + 256);
        if (++csub == nsr) {
            csub = 0;
            if (++ctau == cruns) { ctau = 0; cx++; }
            if (cx < __builtin_amdgcn_readfirstlane(S.nx)) set_copy();
        } else {
            bg += 16 * A.rb;
            bu += 16 * A.rb;
        }
    };
    set_copy();
    copy_next(0);
    copy_next(1);   // a unit has two sub-units
    int it = 0, qc = 0;
    auto run = [&](const SpItem &R, int cnt, auto MC) {
        constexpr int M = decltype(MC)::value;
        const bool sh = R.e == QG_EXPERTS;
        // activation fragments of this wave's superblock: plane row r = (row
        // r / 2 of the tile, plane r % 2); rows past the tile's repeat its
        // last (their products are never kept)
        qg_half8 af[M][8];
        typename MIN::Sums sf[M];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int n = min(8, R.n - 8 * m), k = R.base + 8 * m + min(j >> 1, n - 1);
            const int tok = sh ? k : A.row_token[k];
            const _Float16 *xr = A.xp + ((size_t)tok * 2 + (j & 1)) * D + (size_t)wave * 256 + kq * 8;
#pragma unroll
            for (int f = 0; f < 8; f++) af[m][f] = ld_frag(xr + f * 32);
            sf[m] = MIN::load(A.xsp, (size_t)tok, W, wave, j, kq);
        }
#pragma unroll
        for (int m = 0; m < M; m++) {
#pragma unroll
            for (int f = 0; f < 8; f++) sp_pin(af[m][f]);
            sp_pin(sf[m]);
        }
        const int fmt = (fmts >> (sh ? 8 : 0)) & 0xff;
        constexpr int NB = SpGu<W, TM>::batch(M);
        constexpr bool TWO = NB == 1 && SpGu<W, TM>::TS >= 2 * M;   // sub-units alternate between two sum buffers
        float half = 0.0f;   // NB == 1: the first 16 rows' sum of the unit's 32-row group
        __syncthreads();     // the previous run's sums have been read
        for (int c = 0; c < cnt; c += NB) {
            const int nb = min(NB, cnt - c);
            float2 *rd = red + (TWO ? (c & 1) * (W * 2 * M * 64) : 0);
            for (int b = 0; b < nb; b++, it++) {
                if (it + 2 < nsub) copy_next(qc == 0 ? 2 : qc - 1);
                if (it + 2 < nsub) wait_vmem_but<2 * SP_CPB>();
                else if (it + 1 < nsub) wait_vmem_but<SP_CPB>();
                else wait_vmem();
                float2 y[2][M];
                ksplit_products<M, MIN>(ring + qc * SP_SLOT, af, sf, j, kq, y);
                qc = qc == 2 ? 0 : qc + 1;
#pragma unroll
                for (int cb = 0; cb < 2; cb++)
#pragma unroll
                    for (int m = 0; m < M; m++) rd[(((b * M + m) * 2 + cb) * W + wave) * 64 + lane] = y[cb][m];
            }
            __syncthreads();
            // jobs: sub-unit b, tile m, row 2 kq + t2 of it; F row j
            const int b = wave / (2 * M), m = (wave % (2 * M)) >> 1, t2 = wave & 1, idx = 8 * m + 2 * kq + t2;
            const int row = (sh ? A.nt * QG_TOP : 0) + R.base + idx;
            float s16 = 0.0f;
            if (b < nb) {
                float g = 0.0f, u = 0.0f;
#pragma unroll
                for (int w = 0; w < W; w++) {
                    const float2 ga = rd[(((b * M + m) * 2 + 0) * W + w) * 64 + lane], ua = rd[(((b * M + m) * 2 + 1) * W + w) * 64 + lane];
                    g += t2 ? ga.y : ga.x;
                    u += t2 ? ua.y : ua.x;
                }
                const int pos = plane_pos(fmt, (sub + c + b) * 16 + j);
                const float mv = FULL ? qg_swiglu(g, u) : qg_swiglu_fast(g, u);
                if (idx < R.n) {
                    _Float16 *mp = A.midp + (size_t)row * 2 * F;
                    const _Float16 hv = (_Float16)mv;
                    mp[pos] = hv;
                    mp[F + pos] = (_Float16)(mv - (float)hv);
                }
                if (fmt == QT_Q4_K) {
                    s16 = mv;
                    s16 += __shfl_xor(s16, 1);
                    s16 += __shfl_xor(s16, 2);
                    s16 += __shfl_xor(s16, 4);
                    s16 += __shfl_xor(s16, 8);
                    if (NB > 1 && j == 0) s_gs[wave][kq] = s16;
                }
            }
            if (!TWO) __syncthreads();  // the sums have been read
            if (fmt == QT_Q4_K && b < nb) {
                // the odd sub-unit's job writes its group's sum (a batch
                // starts and ends on even sub-units when NB > 1)
                const int sb = sub + c + b;
                if (sb & 1) {
                    const float sum = s16 + (NB > 1 ? s_gs[wave >= 2 * M ? wave - 2 * M : 0][kq] : half);
                    if (FULL && j == 0 && idx < R.n) {
                        ((float *)A.msp)[(size_t)row * (F / 32) + (sb >> 1)] = sum;
                    } else if (j == 0 && idx < R.n) {
                        _Float16 *gp = A.msp + (size_t)row * 2 * (F / 32) + (sb >> 1);
                        const _Float16 hs = (_Float16)sum;
                        gp[0] = hs;
                        gp[F / 32] = (_Float16)(sum - (float)hs);
                    }
                }
                half = s16;
            }
        }
    };
    while (it < nsub) {
        const SpItem R = sp_item<TM>(S, s_off, A.nt, x, tau);
        const int cnt = min(nsr - sub, nsub - it);
        if (R.T == 1) run(R, cnt, std::integral_constant<int, 1>{});
        else if (TM < 3 || R.T == 2) run(R, cnt, std::integral_constant<int, 2>{});
        else run(R, cnt, std::integral_constant<int, TM>{});
        sub = 0;
        if (++tau == R.runs) { tau = 0; x++; }
    }
    return true;
}

template <int W, int TM, bool FULL>
__global__ __launch_bounds__(64 * W, 1) void pf_gateup_sp_kernel(SpGuArgs A) {
    gateup_sp<W, TM, FULL>(A);
}

// ---- down: a wave per 16 output rows ----
// Unit = 16 D rows of a run, over the whole K = F = 32 NB columns.  A run's mid
// rows are in registers (fragments of both planes); the workgroup's 8 waves
// take its units in turn, each copying a unit's slab (16 rows, contiguous) into
// a ring of its own, so no wave waits for another.  Rows of 288 bytes are laid
// out with 16 bytes of gap after every 4, which spreads the 16 rows of a read
// over the banks.  y rows go to the selections' slots.
template <int FMT, int NB> struct SpDn {
    static constexpr int RB = FMT == QT_Q4_K ? NB / 8 * 144 : NB * 18;   // row bytes
    static constexpr int GAP = RB == 288 ? 16 : 0;
    static constexpr int GP = RB / 4 + GAP / 16;                        // pieces per 4 rows
    static constexpr int PCS = 4 * GP, CP = (PCS + 63) / 64;           // pieces and copies per unit
    static constexpr int SLOT = PCS * 16, LDS = 8 * 3 * SLOT;
    static_assert(RB % 4 == 0 && 4 * RB % 16 == 0, "four rows are whole pieces");
};

struct SpDnArgs {
    int nt, D;
    const int *offsets, *row_slot;
    const uint8_t *down, *sh_down;   // rows of FMT, the shared expert's too
    const _Float16 *midp, *msp;
    float *slots;                    // [rows][D]: slot t*10+k, shared rows at nt*10+t
    const int *tiles;                // as SpGuArgs
};

// Returns false, with nothing done, where the 64-row tiles have the batch.
template <int FMT, int NB, int TM, bool FULL>
QG_DEV bool down_sp(const SpDnArgs &A) {
    using C = SpDn<FMT, NB>;
    constexpr int F = 32 * NB, RB = C::RB, CP = C::CP;
    extern __shared__ uint4 s_dyn[];
    __shared__ SpList S;
    __shared__ int s_off[QG_EXPERTS + 1];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, j = lane & 15, kq = lane >> 4;
    const int tiles = A.tiles ? *A.tiles : 0;   // arrives with the offsets
    for (int i = tid; i <= QG_EXPERTS; i += 512) s_off[i] = A.offsets[i];
    __syncthreads();
    if (tiles) return false;
    const int D = A.D, units = D / 16;
    static_assert(C::LDS >= SP_SCRATCH, "the build's scratch fits the rings");
    sp_build<512, TM>(S, s_dyn, s_off, A.nt, A.sh_down != nullptr, units, sp_part(), gridDim.x);
    const int mine = __builtin_amdgcn_readfirstlane(S.pos[1][3] - S.pos[0][3]) - wave;   // this wave: units wave, wave + 8, ...
    if (mine <= 0) return true;  // no block barrier from here on
    const int nu = (mine + 7) / 8;
    uint8_t *ring = (uint8_t *)s_dyn + (size_t)wave * 3 * C::SLOT;
    uint32_t c_off[CP];
#pragma unroll
    for (int i = 0; i < CP; i++) {
        const int p = min(i * 64 + lane, C::PCS - 1), g = p / C::GP, w = min(p - g * C::GP, RB / 4 - 1);
        c_off[i] = (uint32_t)(g * 4 * RB + 16 * w);
    }
    int x = __builtin_amdgcn_readfirstlane(S.pos[0][0]), tau = __builtin_amdgcn_readfirstlane(S.pos[0][1]);
    int u = __builtin_amdgcn_readfirstlane(S.pos[0][2]) + wave;
    const int nx = __builtin_amdgcn_readfirstlane(S.nx);
    SpItem R = sp_item<TM>(S, s_off, A.nt, x, tau);
    // unit u past the run's end: into the next run
    auto settle = [&](int &sx, int &st, int &su, SpItem &it) {
        bool moved = false;
        while (su >= units) {
            su -= units;
            if (++st == it.runs) { st = 0; sx++; }
            if (sx >= nx) return moved;
            it = sp_item<TM>(S, s_off, A.nt, sx, st);
            moved = true;
        }
        return moved;
    };
    settle(x, tau, u, R);
    int cx = x, ctau = tau, cu = u;
    SpItem CR = R;
    auto copy_next = [&](int slot) {
        const uint8_t *b = (CR.e == QG_EXPERTS ? A.sh_down : A.down + (size_t)CR.e * D * RB) + (size_t)cu * 16 * RB;
#pragma unroll
        for (int i = 0; i < CP; i++)
            if (64 * (i + 1) <= C::PCS || lane < C::PCS - 64 * i) dma16_scalar(c_off[i], b, ring + slot * C::SLOT + 1024 * i);
        cu += 8;
        settle(cx, ctau, cu, CR);
    };
    copy_next(0);
    if (nu > 1) copy_next(1);
    int k = 0, qc = 0;
    const int ro = j * RB + (j >> 2) * C::GAP;   // the lane's row in a slot
    auto run = [&](int cnt, auto MC) {
        constexpr int M = decltype(MC)::value;
        const bool sh = R.e == QG_EXPERTS;
        using MIN = SpMin<FULL>;
        constexpr int NSB = FMT == QT_Q4_K ? NB / 8 : 1;
        qg_half8 af[M][NB];
        typename MIN::Sums sf[M][NSB];
        int sl[M][2];
#pragma unroll
        for (int m = 0; m < M; m++) {
            const int n = min(8, R.n - 8 * m), idx = R.base + 8 * m;
            const size_t row = (size_t)((sh ? A.nt * QG_TOP : 0) + idx + min(j >> 1, n - 1));
            const _Float16 *mr = A.midp + (row * 2 + (j & 1)) * F + kq * 8;
#pragma unroll
            for (int b = 0; b < NB; b++) af[m][b] = ld_frag(mr + b * 32);
            if constexpr (FMT == QT_Q4_K) {
#pragma unroll
                for (int s = 0; s < NSB; s++) sf[m][s] = MIN::load(A.msp, row, NSB, s, j, kq);
            }
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const int i = min(2 * kq + h, n - 1);
                sl[m][h] = sh ? A.nt * QG_TOP + idx + i : A.row_slot[idx + i];
            }
        }
#pragma unroll
        for (int m = 0; m < M; m++) {
#pragma unroll
            for (int b = 0; b < NB; b++) sp_pin(af[m][b]);
            if constexpr (FMT == QT_Q4_K)
#pragma unroll
                for (int s = 0; s < NSB; s++) sp_pin(sf[m][s]);
            asm volatile("" : "+v"(sl[m][0]), "+v"(sl[m][1]));
        }
        for (int c = 0; c < cnt; c++, k++) {
            if (k + 2 < nu) copy_next(qc == 0 ? 2 : qc - 1);
            // only the next two units' copies may be outstanding (the stores
            // between them make this stricter, never looser)
            if (k + 2 < nu) wait_vmem_but<2 * CP>();
            else if (k + 1 < nu) wait_vmem_but<CP>();
            else wait_vmem();
            const uint8_t *row = ring + qc * C::SLOT + ro;
            qc = qc == 2 ? 0 : qc + 1;
            qg_f4 y[M];
#pragma unroll
            for (int m = 0; m < M; m++) y[m] = qg_f4{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (FMT == QT_IQ4_NL) {
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const uint16_t *p16 = (const uint16_t *)(row + 18 * b);
                    const float d = qg_half_u16(p16[0]);
                    const qg_half8 bf = iq4_frag4((uint32_t)p16[1 + 2 * kq] | ((uint32_t)p16[2 + 2 * kq] << 16));
#pragma unroll
                    for (int m = 0; m < M; m++) {
                        const qg_f4 acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[m][b], bf, qg_f4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; i++) y[m][i] = __builtin_fmaf(d, acc[i], y[m][i]);
                    }
                    if ((b & 7) == 7) __builtin_amdgcn_sched_barrier(0);  // eight blocks' operands live at a time
                }
            } else {
#pragma unroll
                for (int s = 0; s < NSB; s++) {
                    const uint8_t *p = row + 144 * s;
                    const Q4kHeader h = q4k_header(*(const uint4 *)p);
                    const uint4 ch0 = *(const uint4 *)(p + 16 + 16 * kq), ch1 = *(const uint4 *)(p + 80 + 16 * kq);
                    qg_half2 scA, ofA, scB, ofB;
                    gq_scales(h.S[0], kq, scA, ofA);
                    gq_scales(h.S[1], kq, scB, ofB);
                    qg_f4 p0[M], p1[M];
#pragma unroll
                    for (int m = 0; m < M; m++) p0[m] = p1[m] = qg_f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int f = 0; f < 4; f++) {
                        const qg_half8 b0 = gq_frag(ch0, f, scA[f >> 1], ofA[f >> 1]), b1 = gq_frag(ch1, f, scB[f >> 1], ofB[f >> 1]);
#pragma unroll
                        for (int m = 0; m < M; m++) {
                            p0[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[m][8 * s + f], b0, p0[m], 0, 0, 0);
                            p1[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[m][8 * s + 4 + f], b1, p1[m], 0, 0, 0);
                        }
                    }
                    const MIN mins(h, kq);
#pragma unroll
                    for (int m = 0; m < M; m++) {
                        const qg_f4 mm = mins.term(sf[m][s]);
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            y[m][i] = __builtin_fmaf(h.d, p0[m][i] + p1[m][i], __builtin_fmaf(-h.dmin, mm[i], y[m][i]));
                    }
                }
            }
            // rows 4 kq .. 4 kq + 3: tile rows 2 kq and 2 kq + 1, hi and lo plane
#pragma unroll
            for (int m = 0; m < M; m++) {
                const int n = R.n - 8 * m;
                float *o = A.slots + u * 16 + j;
                if (2 * kq < n) o[(size_t)sl[m][0] * D] = y[m][0] + y[m][1];
                if (2 * kq + 1 < n) o[(size_t)sl[m][1] * D] = y[m][2] + y[m][3];
            }
            u += 8;
        }
    };
    while (k < nu) {
        const int cnt = min((units - u + 7) / 8, nu - k);   // this wave's units of the run
        if (TM == 1 || R.T == 1) run(cnt, std::integral_constant<int, 1>{});
        else run(cnt, std::integral_constant<int, TM>{});
        settle(x, tau, u, R);
    }
    wait_vmem();  // no copy may land in shared memory after the workgroup ends
    return true;
}

template <int FMT, int NB, int TM, bool FULL>
__global__ __launch_bounds__(512, 1) void pf_down_sp_kernel(SpDnArgs A) { down_sp<FMT, NB, TM, FULL>(A); }
