// The dense layer of gemm.hip on smaller output tiles, for the sizes between decoding and full scoring batches: at 65 - 2,000 rows 256 x 256 tiles are
// 16 - 190 workgroups on 256 CUs (a 4,096-column layer of 161 rows at K = 11,008: 16 workgroups, 187 us where the 90 MB of weights take 15 us).
//
// What bounds it: the rate at which a CU takes operands in.  Without products or LDS reads the k-loop runs no faster: 58 - 72 GB/s a CU, whatever the
// tile and however deep the ring (loads that all hit the L2 reach 105 - 130), because every stage waits for the L2 miss of its newest weight lines
// and a CU holds about 64 KB in flight.  Hence large tiles (bytes per product fall with the tile's sides), parts of K where large tiles are too few
// for the chip, and weight lines shared by neighbours on one XCD.  The MFMA order over k is the persistent kernel's, so an unsplit product is bit
// for bit the same on every tile; parts of K are fp32 sums added in order by a second launch.
// Below 256 rows and above 2,048 k the tiles of neighbouring weight rows start one k-step apart (`turn`) and go round: rows lie a power of two apart, so tiles that walk k in step
// meet in the same L2 channels.  us at 65 / 161 rows, K = 4,096: 22,016 gated columns 47.1 / 56.8 -> 39.3 / 51.5, 12,288 columns 31.6 / 35.8 -> 26.7 / 33.3;
// K = 11,008, 4,096 columns 30.8 / 34.6 -> 27.4 / 32.9.  (From 256 rows on, where it gives 3 to 6 %, the gated, the ungated and the blocked forms of a layer agree bit
// for bit, whichever tiles they take.)
// Inner loop (another where X and W come in phases): a ring of NS stages of 64 k, LDS-DMA pieces spread between the products of the first half step (a burst blocks the wave on the
// vector-memory queue), the next half's fragments requested under the products of the current one, one barrier per stage.
#include <math.h>
#include <type_traits>
#include "gemm_kernel.h"
#include "../../include/evo_mi355x.h"

#define T_ROW 128                            // bytes per LDS row: one k-step of 64 bf16
typedef uint32_t t_u32x4 __attribute__((ext_vector_type(4)));

#define T_DSR(DST, ADDR, OFF) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(DST) : "v"(ADDR), "n"(OFF))

// wait until at most N of this wave's LDS reads are out, tied to the fragments that the wait is for
template <int N, int C>
__device__ __forceinline__ void t_lgkm(t_u32x4 (&f)[C]) {
    static_assert(C >= 1 && C <= 8, "fragments of one half step");
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
#pragma unroll
    for (int i = 0; i < C; ++i) asm volatile("" : "+v"(f[i]));
}

// SiLU (1), tanh-form GELU (2), square of relu (3): the arithmetic of gemm.hip's epilogue
__device__ __forceinline__ void t_act(float (&v)[8], int act) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        if (act == 3) { const float t = fmaxf(v[e], 0.f); v[e] = t * t; }
        else v[e] *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(act == 2 ? v[e] * fmaf(v[e] * v[e], -0.1029432395800235f, -2.3022081981443250f)
                                                                                   : v[e] * -1.4426950408889634f));
    }
}

// row factor and bias of eight columns n .. n + 7: one fused step where there are both, as the persistent kernel's epilogue compiles to (the same bits).
// Mode 3: `rs` the factors of the eight tokens, `rb` the row's bias; else `f` the row's factor.
template <int MODE>
__device__ __forceinline__ void t_scale_bias(float (&v)[8], const GemmArgs& a, float f, float rb, const float* rs, int n) {
    float b[8];
    if (MODE == 3) {
#pragma unroll
        for (int e = 0; e < 8; ++e) b[e] = rb;
    } else if (a.bias) {
        const uint4 q = *(const uint4*)(a.bias + n);
        b[0] = bf_lo(q.x); b[1] = bf_hi(q.x); b[2] = bf_lo(q.y); b[3] = bf_hi(q.y);
        b[4] = bf_lo(q.z); b[5] = bf_hi(q.z); b[6] = bf_lo(q.w); b[7] = bf_hi(q.w);
    }
    if (a.rs) {
        float s[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) s[e] = MODE == 3 ? rs[e] : f;
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = a.bias ? fmaf(v[e], s[e], b[e]) : v[e] * s[e];
    } else if (a.bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += b[e];
    }
}

// Rows of the statistic that a launch stores: its own.  (ss_ld is the pitch of a strip, counted from the first row of the layer: a tail that starts at row m0
// and stored up to there would reach the next strip's first rows.)
__host__ __device__ __forceinline__ int64_t t_stat_rows(const GemmArgs& a) { return a.M; }

template <int BM, int BN, int WGM, int WGN, int NS, int PER_CU, int MODE, bool XB, bool SPLIT>
__global__ __launch_bounds__(64 * WGM * WGN, PER_CU * WGM * WGN / 4) void gemm_tile_kernel(GemmArgs a, int act, float* parts, int splits) {
    constexpr int NW = WGM * WGN, WM = BM / WGM, WN = BN / WGN, MT = WM / 16, NT = WN / 16;
    constexpr int PX = BM / 8 / NW, PW = BN / 8 / NW, P = PX + PW;      // DMA pieces (8 rows, 1 KiB) of a stage per wave
    constexpr int SLAB_X = BM * T_ROW, STAGE = (BM + BN) * T_ROW;
    constexpr bool ODD = BN % 64 != 0;                           // 96 or 48 columns: column tiles as they are, the last tile of a launch may be ragged
    static_assert(PX >= 1 && PW >= 1 && NS >= 2 && PX * NW * 8 == BM && PW * NW * 8 == BN, "whole pieces per wave");
    static_assert(ODD || NT % 2 == 0, "column pairs");
    static_assert(MODE != 1 || SPLIT || WN % 64 == 0 || (ODD && WN % 32 == 0), "a wave holds both halves of its gated columns");
    static_assert(!ODD || (MODE <= 1 && !SPLIT && !XB), "the launches that take such tiles");
    constexpr bool STATS = MODE == 0 && !SPLIT && BN == 128;     // (a strip of the statistic is 128 columns)
    // PHASES (NS = 10 + n): rings of their own for X (four slots) and W (n), two stages of X fetched at even k-steps and two of W at odd ones
    constexpr bool PHASES = NS > 10;
    constexpr int NX = 4, NWS = NS - 10, SLAB_W = BN * T_ROW, W_AT = PHASES ? NX * SLAB_X : SLAB_X;      // (first of the W slots)
    static_assert(!PHASES || NWS >= 5, "W is three stages ahead");
    __shared__ __attribute__((aligned(16))) unsigned char smem[PHASES ? NX * SLAB_X + NWS * SLAB_W : NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    const int l15 = lane & 15, lq = lane >> 4;
    const int64_t kb = (int64_t)a.K * 2;
    const int nk_all = a.K / 64;

    // block b runs on XCD b % 8: every XCD gets a contiguous run of tiles, group_m row tiles next to each other before the next column tile
    int tile;
    {
        const int bid = blockIdx.x, q = a.n_tiles >> 3, r = a.n_tiles & 7, xcd = bid & 7, slot = bid >> 3;
        tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
    }
    int k0 = 0, nk = nk_all, sp = 0;
    if constexpr (SPLIT) {                                       // the parts of a tile's sum are neighbours: they read the same rows, one behind the other
        sp = tile % splits;
        tile /= splits;
        k0 = (int)((int64_t)nk_all * sp / splits);
        nk = (int)((int64_t)nk_all * (sp + 1) / splits) - k0;
    }
    int tm, tn;
    {
        const int across = MODE == 3 ? a.tiles_m : a.tiles_n, along = MODE == 3 ? a.tiles_n : a.tiles_m;   // (mode 3: the tokens are the columns)
        const int per_group = a.group_m * across;
        const int grp = tile / per_group, in_grp = tile - grp * per_group, first = grp * a.group_m;
        const int gsz = along - first < a.group_m ? along - first : a.group_m;
        const int u = in_grp / gsz, v = first + in_grp - u * gsz;
        tm = MODE == 3 ? u : v;
        tn = MODE == 3 ? v : u;
    }
    const int64_t m0 = (int64_t)tm * BM;
    const int n0 = tn * BN;

    // ---- operands: LDS row r of a slab = 128 bytes of row r of the tile, granule g of 16 bytes at slot g ^ (r & 7) (a fragment read, 16 rows x 4
    //      granules, meets no bank twice); the DMA's LDS side is lane-linear, so the lane that fills a slot fetches the granule that belongs there.
    //      W rows: LDS row 32 b + 16 t + 4 q + r holds W row 32 b + 8 q + 4 t + r, so that a lane's accumulators of a pair of column tiles are
    //      eight consecutive columns.  Rows behind the matrix read as zero (bounded descriptors).
    //      ODD: LDS row 16 t + c holds column c of column tile t; gated, tiles 2 p and 2 p + 1 are the two halves of the gated columns 16 p .. 16 p + 15.
    uint32_t xoff[PX], woff[PW];
    const int swz = ((lane & 7) ^ (lane >> 3)) & 7;
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        const int r = 8 * (wave + NW * i) + (lane >> 3);
        if constexpr (XB) {                                      // [row block of 128][K / 16][128][16]
            const int rb = (int)(m0 & 127) + r;
            xoff[i] = (uint32_t)(rb >> 7) * (uint32_t)(128 * kb) + (rb & 127) * 32u + (swz >> 1) * 4096u + (swz & 1) * 16u;
        } else xoff[i] = (uint32_t)(r * kb) + swz * 16u;
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int r = 8 * (wave + NW * i) + (lane >> 3);
        int wr = (r & ~31) + 8 * ((r >> 2) & 3) + 4 * ((r >> 4) & 1) + (r & 3);
        if constexpr (ODD) {
            wr = r;
            if (MODE == 1) {
                const int c = (r >> 5) * 16 + (r & 15), half = (r >> 4) & 1, g = ((n0 >> 1) & 31) + c;
                wr = a.w_rows ? half * (a.N >> 1) + c : (g >> 5) * 64 + half * 32 + (g & 31);
            }
        } else if (MODE == 1 && a.w_rows) wr = (wr >> 6) * 32 + (wr & 31) + ((wr >> 5) & 1) * (a.N >> 1);     // [W1; W2] as it is: 32 rows of each in turn
        woff[i] = (uint32_t)wr * (uint32_t)kb + swz * 16u;
    }
    int64_t src = n0, w_rows = a.N;                              // first row of the "W" operand and how many there are
    if (MODE == 3 && a.rs) {
        src += (int64_t)((n0 >> 8) / a.tm_tiles) * a.row_skip;
        w_rows = a.w_rows;
    }
    const bool plain_gate = MODE == 1 && a.w_rows;
    if (plain_gate) src = n0 >> 1;
    else if (ODD && MODE == 1) src = n0 >> 6 << 6;               // (whole groups of 32 rows of each half)
    const uint64_t xa = (uint64_t)a.x + (XB ? (m0 & ~(int64_t)127) : m0) * kb, wa = (uint64_t)a.w + src * kb;
    const int64_t x_left = a.M - (XB ? (m0 & ~(int64_t)127) : m0), x_most = XB ? 256 : BM, x_ok = x_left < x_most ? x_left : x_most;    // (blocked X: whole blocks, M % 128 == 0)
    // (ODD, gated: 48 columns from the first or the middle one of a group of 32 on lie in two groups; [W1; W2] as it is: both halves, below 4 GiB)
    const int64_t w_left = w_rows - src, w_most = ODD && MODE == 1 ? 128 : BN, w_ok = plain_gate || w_left < w_most ? w_left : w_most;
    const t_u32x4 rx = {(uint32_t)xa, (uint32_t)(xa >> 32) & 0xffffu, (uint32_t)(x_ok * kb), 0x00020000u};
    const t_u32x4 rw = {(uint32_t)wa, (uint32_t)(wa >> 32) & 0xffffu, (uint32_t)(w_ok * kb), 0x00020000u};
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;

    // piece `i` (of P) of k-step `s` -> ring slot at byte `slot`; past the last stage the last one again, into a slot nobody reads (constant counts)
    int at = k0, past = 1;                                       // k-step of the next stage to fetch, stages fetched after it
    if (a.turn) at += (MODE == 3 ? tm : tn) % nk;
    auto next = [&] {
        if (past < nk) at = at + 1 == k0 + nk ? k0 : at + 1;
        ++past;
    };
    auto fetch1 = [&](int s, uint32_t slot, int i) {
        const uint32_t dst = lds0 + slot + wave * 1024;
        if (i < PX)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         ::"s"(dst + i * NW * 1024), "v"(xoff[i < PX ? i : 0]), "s"(rx), "s"((uint32_t)s * (XB ? 16384u : 128u)) : "memory", "m0");
        else
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                         ::"s"(dst + W_AT + (i - PX) * NW * 1024), "v"(woff[i < PX ? 0 : i - PX]), "s"(rw), "s"((uint32_t)s * 128u) : "memory", "m0");
    };

    uint32_t x_rd[2], w_rd[2];
#pragma unroll
    for (int kh = 0; kh < 2; ++kh) {
        const int xr = wm * WM + l15, wr = wn * WN + l15;
        x_rd[kh] = lds0 + (uint32_t)(xr * T_ROW + (((4 * kh + lq) ^ xr) & 7) * 16);
        w_rd[kh] = lds0 + (uint32_t)(W_AT + wr * T_ROW + (((4 * kh + lq) ^ wr) & 7) * 16);
    }
    f32x4_t acc[NT][MT];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    t_u32x4 wf[2][NT], xf[2][MT];
    auto read = [&](uint32_t slot, int kh) {
        const uint32_t wa_ = slot + w_rd[kh], xa_ = slot + x_rd[kh];
#pragma unroll
        for (int i = 0; i < NT; ++i) T_DSR(wf[kh][i], wa_, i * 16 * T_ROW);
#pragma unroll
        for (int j = 0; j < MT; ++j) T_DSR(xf[kh][j], xa_, j * 16 * T_ROW);
    };
    if constexpr (PHASES) {
        // A CU has at most 512 lines under way and they come back in order: 57 GB/s while any of them comes from HBM (1.1 us), 129 where all hit the L2, and x behind w waits
        // with it.  Phases of the one and of the other, a barrier between them, took a probe of that intake (w : x 1 : 2) from 65 to 84 GB/s.  Even step k: X of stages
        // k + 2 and k + 3; odd step: W of stages k + n - 2 and k + n - 1 (the slots were read before the last barrier).  At the middle of a step what may still be out is all of
        // the last two phases (even), all but the first stage of the X phase (odd): the next stage's slabs are then here.
        int xk = at, wk = at, xl = nk - 1, wl = nk - 1;          // k-step of the next stage to fetch, stages left behind it
        auto on = [&](int& kk, int& left) { if (left > 0) { --left; kk = kk + 1 == k0 + nk ? k0 : kk + 1; } };        // (past the last: the same again, into a slot nobody reads)
        uint32_t xf_slot = 0, wf_slot = 0;                       // slot of the next stage to fetch
        auto one_x = [&](int i) { fetch1(xk, xf_slot, i); };
        auto one_w = [&](int i) { fetch1(wk, wf_slot, PX + i); };
        auto end_x = [&] { on(xk, xl); xf_slot = xf_slot + SLAB_X == NX * SLAB_X ? 0 : xf_slot + SLAB_X; };
        auto end_w = [&] { on(wk, wl); wf_slot = wf_slot + SLAB_W == NWS * SLAB_W ? 0 : wf_slot + SLAB_W; };
        auto some_x = [&] {
#pragma unroll
            for (int i = 0; i < PX; ++i) one_x(i);
            end_x();
        };
        auto some_w = [&] {
#pragma unroll
            for (int i = 0; i < PW; ++i) one_w(i);
            end_w();
        };
        auto read2 = [&](uint32_t xs, uint32_t ws_, int kh) {
#pragma unroll
            for (int i = 0; i < NT; ++i) T_DSR(wf[kh][i], ws_ + w_rd[kh], i * 16 * T_ROW);
#pragma unroll
            for (int j = 0; j < MT; ++j) T_DSR(xf[kh][j], xs + x_rd[kh], j * 16 * T_ROW);
        };
        auto mma2 = [&](int kh, auto phase) {                    // phase: pieces between the products, 2 stages of them (0: none, 1: X, 2: W)
            constexpr int PH_ = decltype(phase)::value, TOTAL = NT * MT, EACH = PH_ == 1 ? PX : PW, D = PH_ ? 2 * EACH : 0;
#pragma unroll
            for (int u = 0; u < TOTAL; ++u) {
                const int i = u / MT, j = u % MT;
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[kh][i]), __builtin_bit_cast(bf16x8_t, xf[kh][j]), acc[i][j], 0, 0, 0);
#pragma unroll
                for (int d = u * D / TOTAL; d < (u + 1) * D / TOTAL; ++d) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (PH_ == 1) { one_x(d % EACH); if (d % EACH == EACH - 1) end_x(); }
                    else { one_w(d % EACH); if (d % EACH == EACH - 1) end_w(); }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        };
        uint32_t xs = 0, ws_ = 0;
        auto step = [&](auto phase) {
            constexpr int PH_ = decltype(phase)::value;
            read2(xs, ws_, 1);
            t_lgkm<NT + MT>(wf[0]);
            t_lgkm<NT + MT>(xf[0]);
            __builtin_amdgcn_sched_barrier(0);
            mma2(0, phase);
            __builtin_amdgcn_sched_barrier(0);
            t_lgkm<0>(wf[1]);
            t_lgkm<0>(xf[1]);
            asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PH_ == 1 ? 2 * PW + 2 * PX : PX + 2 * PW) : "memory");
            asm volatile("s_barrier" ::: "memory");
            xs = xs + SLAB_X == NX * SLAB_X ? 0 : xs + SLAB_X;
            ws_ = ws_ + SLAB_W == NWS * SLAB_W ? 0 : ws_ + SLAB_W;
            read2(xs, ws_, 0);                                   // (behind the last stage: slots that are not used any more)
            __builtin_amdgcn_sched_barrier(0);
            mma2(1, std::integral_constant<int, 0>{});
            __builtin_amdgcn_sched_barrier(0);
        };
        some_w(); some_w(); some_x(); some_x();
#pragma unroll
        for (int i = 2; i < NWS - 1; ++i) some_w();
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PX + (NWS - 3) * PW) : "memory");       // (W 0, W 1, X 0)
        asm volatile("s_barrier" ::: "memory");
        read2(0, 0, 0);
        for (int k = 0; k < nk; k += 2) {
            step(std::integral_constant<int, 1>{});
            if (k + 1 < nk) step(std::integral_constant<int, 2>{});
        }
    } else {
    // the products of one half of a k-step; `dma`: with the P pieces of k-step `s` between them
    auto mma = [&](int kh, bool dma, int s, uint32_t fslot) {
        constexpr int TOTAL = NT * MT;
#pragma unroll
        for (int u = 0; u < TOTAL; ++u) {
            const int i = u / MT, j = u % MT;
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[kh][i]), __builtin_bit_cast(bf16x8_t, xf[kh][j]), acc[i][j], 0, 0, 0);
            if (dma) {
#pragma unroll
                for (int d = u * P / TOTAL; d < (u + 1) * P / TOTAL; ++d) {
                    __builtin_amdgcn_sched_barrier(0);
                    fetch1(s, fslot, d);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };

    // ---- the pipeline over k-steps; stage k lives in slot k % NS.  Step k:
    //        half 0   the second half's fragments are requested; products of the first, the DMA of stage k + NS - 1 spread between them (its slot held
    //                 stage k - 1, which everyone had read before the last barrier)
    //        wait     own pieces of stage k + 1 have landed, own reads of stage k are done; barrier: everyone's
    //        half 1   the first fragments of stage k + 1 are requested; products of the second half
    uint32_t slot = 0, nslot = STAGE, fslot = (NS - 1) * STAGE;
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) {
#pragma unroll
        for (int i = 0; i < P; ++i) fetch1(at, s * STAGE, i);
        next();
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * P) : "memory");
    asm volatile("s_barrier" ::: "memory");
    read(0, 0);
    for (int k = 0; k < nk; ++k) {
        read(slot, 1);
        t_lgkm<NT + MT>(wf[0]);
        t_lgkm<NT + MT>(xf[0]);
        __builtin_amdgcn_sched_barrier(0);
        mma(0, true, at, fslot);
        __builtin_amdgcn_sched_barrier(0);
        next();
        t_lgkm<0>(wf[1]);
        t_lgkm<0>(xf[1]);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * P) : "memory");
        asm volatile("s_barrier" ::: "memory");
        read(nslot, 0);                                          // (behind the last stage: a slot that is not used any more)
        __builtin_amdgcn_sched_barrier(0);
        mma(1, false, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fslot = slot;
        slot = nslot;
        nslot = nslot + STAGE == NS * STAGE ? 0 : nslot + STAGE;
    }
    }
    t_lgkm<0>(wf[0]);
    t_lgkm<0>(xf[0]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // (the tail's re-fetches land before the LDS is read again or given back)

    if constexpr (SPLIT) {                                       // this part's sums, as they are: [part][row][column]
        float* out = parts + ((int64_t)sp * a.M) * a.N;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int64_t m = m0 + wm * WM + 16 * j + l15;
            if (m < a.M) {
#pragma unroll
                for (int b = 0; b < NT / 2; ++b) {
                    float* o = out + m * a.N + n0 + wn * WN + 32 * b + 8 * lq;
                    *(f32x4_t*)o = acc[2 * b][j];
                    *(f32x4_t*)(o + 4) = acc[2 * b + 1][j];
                }
            }
        }
        return;
    }

    if constexpr (ODD) {                                         // a lane's 4 values of a column tile t are its columns 4 lq .. + 3
        const int gn = a.N >> 1;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int64_t m = m0 + wm * WM + 16 * j + l15;
            const bool ok = m < a.M;
            const float f = a.rs && ok ? a.rs[m] : 1.f;
            if constexpr (MODE == 1) {
#pragma unroll
                for (int p = 0; p < NT / 2; ++p) {
                    const int c = (n0 + wn * WN) / 2 + 16 * p + 4 * lq;
                    uint32_t o[2];
#pragma unroll
                    for (int e = 0; e < 4; e += 2) {
                        float z1[2] = {acc[2 * p][j][e], acc[2 * p][j][e + 1]}, z2[2] = {acc[2 * p + 1][j][e], acc[2 * p + 1][j][e + 1]};
                        if (a.rs) { z1[0] *= f; z1[1] *= f; z2[0] *= f; z2[1] *= f; }
                        const uint32_t u1 = pack_bf2(z1[0], z1[1]), u2 = pack_bf2(z2[0], z2[1]);                // the dense layers' bf16 outputs
                        const f32x2_t oo = act_gate2(f32x2_t{bf_lo(u1), bf_hi(u1)}, f32x2_t{bf_lo(u2), bf_hi(u2)}, act);
                        o[e >> 1] = pack_bf2(oo[0], oo[1]);
                    }
                    if (ok && c < gn) *(uint2*)(a.y + m * gn + c) = make_uint2(o[0], o[1]);
                }
            } else {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int n = n0 + wn * WN + 16 * t + 4 * lq;
                    if (!ok || n >= a.N) continue;
                    float v[8] = {acc[t][j][0], acc[t][j][1], acc[t][j][2], acc[t][j][3], 0.f, 0.f, 0.f, 0.f};
                    float b[4] = {0.f, 0.f, 0.f, 0.f};
                    if (a.bias) {
                        const uint2 q = *(const uint2*)(a.bias + n);
                        b[0] = bf_lo(q.x); b[1] = bf_hi(q.x); b[2] = bf_lo(q.y); b[3] = bf_hi(q.y);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = a.rs ? fmaf(v[e], f, b[e]) : v[e] + b[e];
                    if (a.res) {
                        const uint2 q = *(const uint2*)(a.res + m * a.N + n);
                        v[0] += bf_lo(q.x); v[1] += bf_hi(q.x); v[2] += bf_lo(q.y); v[3] += bf_hi(q.y);
                    }
                    if (act && n < a.act_cols) t_act(v, act);
                    *(uint2*)(a.y + m * a.N + n) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));      // the one rounding
                }
            }
        }
        return;
    }
    // ---- epilogue, straight from registers: a lane's 8 values of (row tile j, column pair b) are columns 32 b + 8 lq .. + 7 of row 16 j + l15
    if constexpr (MODE == 1) {
        const int gn = a.N >> 1;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int64_t m = m0 + wm * WM + 16 * j + l15;
            const float f = a.rs && m < a.M ? a.rs[m] : 1.f;
#pragma unroll
            for (int p = 0; p < WN / 64; ++p) {
                float z1[8], z2[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    z1[e] = acc[4 * p + (e >> 2)][j][e & 3];
                    z2[e] = acc[4 * p + 2 + (e >> 2)][j][e & 3];
                    if (a.rs) { z1[e] *= f; z2[e] *= f; }
                }
                uint32_t o[4];
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const uint32_t u1 = pack_bf2(z1[e], z1[e + 1]), u2 = pack_bf2(z2[e], z2[e + 1]);       // the dense layers' bf16 outputs
                    const f32x2_t oo = act_gate2(f32x2_t{bf_lo(u1), bf_hi(u1)}, f32x2_t{bf_lo(u2), bf_hi(u2)}, act);
                    o[e >> 1] = pack_bf2(oo[0], oo[1]);
                }
                if (m < a.M) *(uint4*)(a.y + m * gn + (n0 + wn * WN) / 2 + 32 * p + 8 * lq) = make_uint4(o[0], o[1], o[2], o[3]);
            }
        }
        return;
    }
    const bool on = n0 < a.act_cols, stats = STATS && a.ss;
    uint4 kept[STATS ? MT : 1][STATS ? NT / 2 : 1];              // the stored values, for the statistic
#pragma unroll
    for (int j = 0; j < MT; ++j) {
        const int64_t m = m0 + wm * WM + 16 * j + l15;
        const bool ok = m < a.M;
        const float f = MODE == 0 && a.rs && ok ? a.rs[m] : 1.f;
        const float rb = MODE == 3 && a.bias && ok ? bf_to_f(a.bias[m]) : 0.f;
#pragma unroll
        for (int b = 0; b < NT / 2; ++b) {
            const int n = n0 + wn * WN + 32 * b + 8 * lq;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] = acc[2 * b + (e >> 2)][j][e & 3];
            }
            t_scale_bias<MODE>(v, a, f, rb, MODE == 3 && a.rs ? a.rs + src + (n - n0) : nullptr, n);
            if (MODE == 0 && a.res && ok) {
                const uint4 q = *(const uint4*)(a.res + m * a.N + n);
                v[0] += bf_lo(q.x); v[1] += bf_hi(q.x); v[2] += bf_lo(q.y); v[3] += bf_hi(q.y);
                v[4] += bf_lo(q.z); v[5] += bf_hi(q.z); v[6] += bf_lo(q.w); v[7] += bf_hi(q.w);
            }
            if (MODE == 0 && act && on) t_act(v, act);
            const uint4 o = make_uint4(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7]));    // the one rounding
            if (ok) {
                if constexpr (MODE == 3) *(uint4*)(a.y + (((int64_t)(n >> 8) * a.M + m) << 8) + (n & 255)) = o;
                else *(uint4*)(a.y + m * a.N + n) = o;
            }
            if constexpr (STATS) kept[j][b] = o;
        }
    }
    if (stats) {
        // a row's 128 columns in the order of gemm.hip's epilogue (the same bits): a lane's values of strip after strip, the waves beside each other one
        // behind the other, then the four lane groups
        float* part = (float*)smem;                              // [MT rows of tiles][64 lanes] per wave row
        asm volatile("s_barrier" ::: "memory");                  // (every wave is done with the operands)
        for (int turn = 0; turn < WGN; ++turn) {
            if (wn == turn) {
#pragma unroll
                for (int j = 0; j < MT; ++j) {
                    float t = turn ? part[(wm * MT + j) * 64 + lane] : 0.f;
#pragma unroll
                    for (int b = 0; b < NT / 2; ++b) {
                        const uint32_t d[4] = {kept[STATS ? j : 0][STATS ? b : 0].x, kept[STATS ? j : 0][STATS ? b : 0].y, kept[STATS ? j : 0][STATS ? b : 0].z,
                                               kept[STATS ? j : 0][STATS ? b : 0].w};
#pragma unroll
                        for (int e = 0; e < 4; ++e) { const float lo = bf_lo(d[e]), hi = bf_hi(d[e]); t = fmaf(lo, lo, t); t = fmaf(hi, hi, t); }
                    }
                    if (turn < WGN - 1) part[(wm * MT + j) * 64 + lane] = t;
                    else {
                        t += __shfl_xor(t, 16);
                        t += __shfl_xor(t, 32);
                        const int64_t m = m0 + wm * WM + 16 * j + l15;
                        if (lq == 0 && m < t_stat_rows(a)) a.ss[(int64_t)(n0 >> 7) * a.ss_ld + m] = t;
                    }
                }
            }
            __syncthreads();
        }
    }
}

// The parts of every sum, added in the order of k, and what the product does behind it.  A thread takes eight columns of a row (mode 1: the eight
// gated columns of two strips of 32).
template <int MODE>
__global__ __launch_bounds__(256) void gemm_parts_kernel(GemmArgs a, int act, const float* __restrict__ part, int splits) {
    const int n8 = (MODE == 1 ? a.N >> 1 : a.N) >> 3;
    const int64_t id = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t m = id / n8;
    const int c8 = (int)(id - m * n8) * 8;
    const bool ok = m < a.M;                                     // (N % 128 == 0: the 16 threads of a strip are all in or all out)
    if (!ok) return;
    const int64_t plane = a.M * a.N;
    auto sum = [&](int n, float (&v)[8]) {
        const float* p = part + m * a.N + n;
        f32x4_t lo = *(const f32x4_t*)p, hi = *(const f32x4_t*)(p + 4);
        for (int s = 1; s < splits; ++s) {
            p += plane;
            lo += *(const f32x4_t*)p;
            hi += *(const f32x4_t*)(p + 4);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] = lo[e]; v[4 + e] = hi[e]; }
    };
    const float f = a.rs && MODE != 3 ? a.rs[m] : 1.f;
    if constexpr (MODE == 1) {
        const int n = (c8 >> 5) * 64 + (c8 & 31);
        float z1[8], z2[8];
        sum(n, z1);
        sum(n + 32, z2);
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            if (a.rs) { z1[e] *= f; z1[e + 1] *= f; z2[e] *= f; z2[e + 1] *= f; }
            const uint32_t u1 = pack_bf2(z1[e], z1[e + 1]), u2 = pack_bf2(z2[e], z2[e + 1]);
            const f32x2_t oo = act_gate2(f32x2_t{bf_lo(u1), bf_hi(u1)}, f32x2_t{bf_lo(u2), bf_hi(u2)}, act);
            o[e >> 1] = pack_bf2(oo[0], oo[1]);
        }
        *(uint4*)(a.y + m * (a.N >> 1) + c8) = make_uint4(o[0], o[1], o[2], o[3]);
        return;
    }
    float v[8];
    sum(c8, v);
    t_scale_bias<MODE>(v, a, f, MODE == 3 && a.bias ? bf_to_f(a.bias[m]) : 0.f,
                       MODE == 3 && a.rs ? a.rs + c8 + (int64_t)((c8 >> 8) / a.tm_tiles) * a.row_skip : nullptr, c8);
    if (MODE == 0 && a.res) {
        const uint4 q = *(const uint4*)(a.res + m * a.N + c8);
        v[0] += bf_lo(q.x); v[1] += bf_hi(q.x); v[2] += bf_lo(q.y); v[3] += bf_hi(q.y);
        v[4] += bf_lo(q.z); v[5] += bf_hi(q.z); v[6] += bf_lo(q.w); v[7] += bf_hi(q.w);
    }
    if (MODE == 0 && act && c8 < a.act_cols) t_act(v, act);
    const uint4 o = make_uint4(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7]));
    if constexpr (MODE == 3) *(uint4*)(a.y + (((int64_t)(c8 >> 8) * a.M + m) << 8) + (c8 & 255)) = o;
    else *(uint4*)(a.y + m * a.N + c8) = o;
    if (MODE == 0 && a.ss) {
        const uint32_t d[4] = {o.x, o.y, o.z, o.w};
        float t = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) { const float lo = bf_lo(d[e]), hi = bf_hi(d[e]); t = fmaf(lo, lo, t); t = fmaf(hi, hi, t); }
        t += __shfl_xor(t, 1, 16);
        t += __shfl_xor(t, 2, 16);
        t += __shfl_xor(t, 4, 16);
        t += __shfl_xor(t, 8, 16);
        if ((threadIdx.x & 15) == 0) a.ss[(int64_t)(c8 >> 7) * a.ss_ld + m] = t;
    }
}

// ---------------------------------------------------------------------------------------------------------------- which tile
// Measured times of one k-step (64 deep) of one tile on one CU, in us: 64 x 64 0.255, 128 x 64 0.435, 128 x 128 0.515, 192 x 128 0.70, 256 x 128 0.84,
// 256 x 256 (the persistent kernel) 1.12 -- all of them the pace at which a CU takes operands in (58 GB/s: 64 KB in flight, about 1 us behind the
// L2 miss that one of the CUs sharing a row pays), so a product's time is its operand rows per CU, and a larger tile moves fewer.  A launch takes the
// tile and the number of parts of K whose sum of rounds, partial sums and memory traffic is least.  At K = 4,096 / 11,008 (MI355X, us, persistent
// kernel -> this choice): 4,096 columns 68 -> 16 / 187 -> 34 at 161 rows, 72 -> 28 / 188 -> 58 at 512, 74 -> 36 / 187 -> 95 at 1,024, 75 -> 57 / 193 ->
// 147 at 2,048; 12,288 columns 76 -> 34 at 161 rows, 78 -> 58 at 512; 22,016 gated columns 82 -> 53 at 161.
struct TileKind { int bm, bn; double step_us; };
static const TileKind kinds[] = {{64, 64, 0.255}, {128, 64, 0.435}, {128, 128, 0.515}, {192, 128, 0.70}, {256, 128, 0.84}, {128, 256, 0.86},
                                 {96, 96, 0.50}, {192, 96, 0.667}, {96, 48, 0.35}, {64, 96, 0.40}, {128, 96, 0.55}};
// The next three, below 256 rows and without parts, statistics or a transposed result: narrow enough that a layer of 12,288 to 24,576 columns is one round of
// nearly all CUs.  us, before -> with them: 22,016 gated columns, K = 4,096 (172 tiles of 128 -> 230 of 96) 39.6 -> 37.7 at 65 rows, 42.2 -> 40.8 at 96, 48.0 -> 44.8
// at 129, 51.7 -> 48.7 at 161, 53.6 -> 51.4 at 192; 12,288 columns (192 tiles of 64 -> 256 of 48) 27.2 -> 24.4 at 65, 29.8 -> 27.8 at 96; 11,264 columns 30.5 -> 23.5 and 33.1 -> 26.7.  Twelve waves for
// 192 x 96 (six 49.8, four 56.7: a wave alone on its SIMD waits for its own fragments).  Not taken: 128 x 96 in step (43.4 - 45.1 at 97 - 128 rows, 42.4 - 46.6 with 128 x 128),
// 256 x 96 (66.5 against 56.5 at 193) and 192 x 48 (35.7 against 34.2).  The last two: tile_one_round, tile_one_round_gated.
#define T_ODD 6                              // first of them
// The persistent kernel on tiles of 160, 192 and 224 rows (and 256 columns): a step of 64 k takes nearly as little as its operands do, where 256 rows are a round that
// leaves a third of the chip idle or a tile that is half padding.  us, the plan without them -> with (rows of the tile): K = 4,096, 22,016 gated columns 89 -> 66 at 300 rows
// (160), 159 -> 124 at 770 (160), 163 -> 147 at 1,025 (224), 247 -> 221 at 1,600 (224), 502 -> 469 at 3,600 (224); 12,288 columns 82 -> 69 at 930 (192), 136 -> 115 at 1,300 (160);
// K = 11,008, 4,096 columns 193 -> 145 at 2,100 (160), 402 -> 353 at 6,000 (192).
static const int short_rows[] = {160, 192, 224};
// A step of 64 k of those tiles, and of 256 rows beside them: `us`, and `more` for each unit of the chip's rounds beyond `from` that is rows of the result (power).  Measured, us
// at under half, three quarters and all of a round: 160 rows 0.80, 0.90, 0.99; 192 0.86, 1.02, 1.11; 224 0.93, 1.16, 1.27; 256 1.19, 1.25, 1.43, in one round as in nine and at
// K = 2,048 to 22,528 (3,587 layers of 256 to 10,000 rows, 3 to 6 % about these; 256 rows are taken at 2 % less, which the plans of before had).  `end`: a round's first
// operands and results.
struct StepUs { int rows; double us, from, more, end; };
static const StepUs short_steps[] = {{160, 0.895, 0.76, 0.45, 2.43}, {192, 1.022, 0.76, 0.47, 2.43}, {224, 1.107, 0.66, 0.62, 2.43}};
static const StepUs whole_steps = {256, 1.16, 0.68, 0.85, 4.5};
#define T_SHORT 96                           // first of them
#define T_PERSISTENT 99

struct TilePlan { int kind; int splits; double us; int64_t rows; };      // rows: how many of M it takes

static int tile_cus() {
    static const int n = [] {
        int dev = 0, c = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
        return c < 8 ? 8 : c & ~7;
    }();
    return n;
}

// `M` tokens, `N` columns of the weight; mode 3 has them the other way round in the launch
static TilePlan tile_best(int64_t M, int64_t N, int64_t K, int mode, bool stats, bool splits_ok, bool persistent_ok) {
    const double cus = tile_cus(), nk = (double)(K / 64), flops = 2.0 * M * N * K;
    const double memory = (2.0 * (M * K + N * K) + 2.0 * M * N) / 4.9e6, power = flops / 1.56e9;
    TilePlan best = {-1, 1, 1e30, M};
    if (persistent_ok) {
        const double rounds = ceil((double)((M + 255) / 256) * (double)(N / 256) / cus);
        const double us = rounds * (nk * 1.12 + 6.0);
        best = {T_PERSISTENT, 1, us > power ? us : power, M};
        if (memory > best.us) best.us = memory;
    }
    for (int c = 0; c < T_ODD + 3; ++c) {
        const int bm = mode == 3 ? kinds[c].bn : kinds[c].bm, bn = mode == 3 ? kinds[c].bm : kinds[c].bn;      // along the tokens, along the weight
        if ((mode == 1 && c == 0) || (mode != 3 && c == 5)) continue;
        if (c >= T_ODD && (M >= 256 || mode == 3 || stats || (mode == 1) != (c < T_ODD + 2))) continue;
        if (c == T_ODD + 2 && N / 48 < 0.9 * cus) continue;      // (10,240 columns, 214 tiles: 26.3 us at 96 rows, 25.9 without)
        const double tiles = (double)((M + bm - 1) / bm) * (double)((N + bn - 1) / bn);
        for (int s = 1; s <= (splits_ok && c < T_ODD ? 8 : 1); ++s) {
            if (s == 1 && stats && bn != 128) continue;
            if (s > 1 && (tiles * s > 2 * cus || nk / s < 8 || (double)s * M * N * 4 > 256e6)) break;
            double us = ceil(tiles * s / cus) * (ceil(nk / s) * kinds[c].step_us + (mode == 1 && s == 1 ? 6.0 : 3.0));
            if (us < power * 1.05) us = power * 1.05;
            if (us < memory) us = memory;
            if (s > 1) us += 5.6 + (double)s * M * N * 8 / 4.9e6;
            if (us < best.us) best = {c, s, us, M};
        }
    }
    return best;
}

// One or two launches: whole rounds of the persistent kernel in front where the last round would leave most of the chip idle.
static int tile_plan_square(int64_t M, int64_t N, int64_t K, int mode, bool stats, bool splits_ok, bool persistent_ok, TilePlan (&out)[2]) {
    out[0] = tile_best(M, N, K, mode, stats, splits_ok, persistent_ok);
    if (!persistent_ok || mode == 3 || out[0].kind != T_PERSISTENT) return 1;
    const int64_t tn = N / 256, cus = tile_cus();
    for (int64_t rounds = (((M + 255) / 256) * tn) / cus; rounds >= 1 && rounds <= 16; --rounds) {
        const int64_t rows = rounds * cus / tn * 256;            // (as many row tiles as fit the rounds)
        if (rows < 256 || rows >= M) continue;
        TilePlan head = tile_best(rows, N, K, mode, stats, false, true), tail = tile_best(M - rows, N, K, mode, stats, splits_ok, true);
        if (head.kind == T_PERSISTENT && tail.kind != T_PERSISTENT && head.us + tail.us + 4.0 < 0.97 * out[0].us) {
            out[0] = head;                                       // (`rows` of each are set by tile_best)
            out[1] = tail;
            return 2;
        }
        break;
    }
    return 1;
}

// Ungated layers of 65 to 255 rows on tiles whose row tiles and column tiles together are nearly one round of the CUs (nine tenths and more), where the tiles above leave a quarter of the
// chip idle, and in place of 128 x 64 in one round two parts of 128 x 128: half the operand rows a CU takes in, and what a round of 128 x 64 waits for is beyond its cost rule (weights
// that come from memory; sums included).  us, before -> these, at 112 / 129 / 161 / 192 rows: 96 x 96, 12,288 columns of K = 2,048 21.5 / 20.3 / 20.8 / 22.0 -> 18.5 / 18.9 /
// 20.6 / 21.2, 4,096 37.9 / 34.4 / 35.7 / 37.8 -> 31.1 / 31.7 / 35.0 / 36.0 (phases from 161 rows on), 8,192 54.9 / 57.7 / 63.4 / 65.9 -> 52.1 / 54.1 / 60.5 / 65.5, 11,264 of 4,096 31.9 / 34.0 /
// 35.0 / 37.2 -> 31.4 / 31.0 / 34.2 / 34.6; 96 x 48, 6,144 of 4,096 22.4 / 24.5 / 26.4 / 27.9 -> 20.9 / 21.4 / 23.3 / 26.1 (of 6,144 from 145 rows on 2 to 11 % behind: parts of K); 64 x 96 at
// 193 / 224 / 255 rows there 27.2 / 29.0 / 30.8 -> 23.8 / 26.3 / 28.7; two parts at 65 / 96 / 128 rows, 16,384 of 4,096 41.0 / 39.0 / 40.7 -> 34.9 / 36.1 / 38.7, 13,824 of 5,120 47.9 / 46.6 /
// 50.1 -> 39.3 / 40.9 / 43.9, 8,192 of 4,096 at 240 36.9 -> 32.5 (of 2,048 behind: 16,384 24.0 : 26.5).  96 x 48 of short K not where its second row
// tile is nearly empty (the time before over this, 5,632 to 6,144 columns, weights cold: of 2,048 0.91 at 97 rows, 0.92 to 0.96 at 104, 1.0 at 112, 1.02 to 1.04 to 128, 1.21 to 1.45 beyond; of 2,304
// 0.93, 0.95, 1.04, 1.09; of 2,560 to 4,608 0.96 to 1.03 at 97 and 104), beyond K = 4,608 to 144 (of 5,120: 136 0.98 to 1.02, 145 0.94 to 0.97, 161 and more 0.90 to 0.96).
// 0.9: the mean of 96 x 48's and 64 x 96's times above over those before, for parts_plan's comparison (the others are wider than what comes in parts).
static void tile_one_round(int64_t M, int64_t N, int64_t K, bool splits_ok, TilePlan& plan) {
    const int64_t cus = tile_cus();
    auto round = [&](int kind) {
        const int64_t tiles = ((M + kinds[kind].bm - 1) / kinds[kind].bm) * ((N + kinds[kind].bn - 1) / kinds[kind].bn);
        return tiles <= cus && 10 * tiles >= 9 * cus;
    };
    const bool narrow = M >= (K < 2560 ? 112 : 97) && (K <= 4608 || M <= 144);
    const int kind = M <= 96 || K < 2048 ? -1 : M <= 192 && round(T_ODD) ? T_ODD : K > 5120 ? -1 : M <= 192 ? (narrow && round(T_ODD + 2) ? T_ODD + 2 : -1) : round(T_ODD + 3) ? T_ODD + 3 : -1;
    if (kind >= 0) plan = {kind, 1, 0.9 * plan.us, M};
    else if (plan.kind == 1 && plan.splits == 1 && splits_ok && K >= 4096 && 2 * ((M + 127) / 128) * (N / 128) <= cus) plan = {2, 2, plan.us, M};
}

// Gated layers of 97 to 128 rows: 128 x 96 in phases where column tiles are nearly a round, 96 x 96 where two row tiles of them are.  us at 97 / 112 / 128 rows, before -> these: 22,016 columns of
// K = 4,096 43.5 / 43.7 / 44.9 -> 41.8 / 41.8 / 42.7 (128 x 128 in phases before: 172 workgroups; 16,384 columns, 171, 40.8 : 41.5; of 2,048 0.95 to 1.0, of 2,560 to 6,144 0.97 to 1.17), 11,264 of 2,048 20.5 / 20.5 / 20.9 -> 17.0 / 17.9 / 18.4.
static void tile_one_round_gated(int64_t M, int64_t N, int64_t K, TilePlan& plan) {
    const int64_t cus = tile_cus(), across = (N + 95) / 96;
    if (M <= 96 || M > 128 || K < 2048) return;
    if (across <= cus && 8 * across >= 7 * cus) plan = {T_ODD + 4, 1, plan.us, M};
    else if (2 * across <= cus && 20 * across >= 9 * cus) plan = {T_ODD, 1, plan.us, M};
}

static double steps_us(const StepUs& s, double rows, double cols, double nk) {
    const double cus = tile_cus(), rounds = ceil(ceil(rows / s.rows) * cols / cus), full = rows / s.rows * cols / (rounds * cus);
    return rounds * (nk * (s.us + s.more * fmax(0.0, full - s.from)) + s.end);
}

// ... or one launch of the persistent kernel on 160, 192 or 224 rows.  Over 3,587 layers and sizes (K = 2,048 to 22,528, 256 to 10,000 rows) the choice is 0.4 % off the fastest of
// all plans on average (4.8 % without them), and more than 3 % behind the plan without them at seven (at most 9 %: 224 rows in a full round at K = 16,384).  Where many rounds run at
// the power limit, 256 rows are ahead (32,768 rows, 22,016 gated columns: 4.01 ms, 4.31 on 224, 4.34 on 192, 4.48 on 160).  Two launches take 3 to 9 % more than their sum, a tail
// that finds its weights in the caches nine tenths of its time.  Below 2,048 k the plans are as they were (4,096 columns at K = 1,024 could
// still go from 41 to 37 us at 4,700 rows: layers that small are launches more than work).  Below 256 rows neighbouring tiles start one k-step apart, which these do not; and
// their padding is most of a tile.
static int tile_plan(int64_t M, int64_t N, int64_t K, int mode, bool stats, bool splits_ok, bool persistent_ok, bool short_ok, TilePlan (&out)[2]) {
    const int n = tile_plan_square(M, N, K, mode, stats, splits_ok, persistent_ok, out);
    if (mode == 0 && M < 256 && !stats) tile_one_round(M, N, K, splits_ok, out[0]);
    if (mode == 1 && M < 256) tile_one_round_gated(M, N, K, out[0]);
    if (!persistent_ok || !short_ok || M < 256 || K < 2048) return n;
    const double memory = (2.0 * (M * K + N * K) + 2.0 * M * N) / 4.9e6, nk = (double)(K / 64);
    const double rows = (double)(mode == 3 ? N : M), cols = (double)((mode == 3 ? M : N) / 256);       // (mode 3: the tokens are the columns of the launch)
    double us = out[0].us;
    if (n == 2) us = 1.03 * (us + 0.9 * out[1].us + 4.0);
    else if (out[0].kind == T_PERSISTENT) us = fmax(steps_us(whole_steps, rows, cols, nk), memory);
    else if (mode == 1 && out[0].splits == 1) us -= 3.0;         // (one tile's closing with the gate: 11,008 gated columns at 390 rows 51.9 on 256 x 128, 58.8 on 160)
    int kind = -1;
    for (int i = 0; i < 3; ++i) {
        const double t = fmax(steps_us(short_steps[i], rows, cols, nk), memory);
        if (t < us) { us = t; kind = T_SHORT + i; }
    }
    if (kind < 0) return n;
    out[0] = {kind, 1, us, M};
    return 1;
}

// X and W in phases (gemm_tile_kernel) where the last row tile has 96 of its 128 rows (120 of more than four tiles), and at 150 to 192 rows on 192, 80 to 96 on 96: rows that are not there cost no intake,
// a tile without them runs ahead of those that share its weights (4,096 columns, K = 11,008: 102.6 -> 91.7 at 896 rows, 81.1 -> 92.4 at 912), and W is further
// ahead without.  us, in turn -> in phases: 12,288 columns, K = 4,096, 43.6 -> 37.9 at 256 rows, 41.6 -> 37.2 at 128, 38.6 -> 36.9 at 104, 33.0 -> 35.9 at 161; 4,096 columns,
// K = 11,008, 104 -> 93 at 1,024; 22,016 gated columns 48.0 -> 44.9 at 161, 52.5 -> 46.6 at 192, 47.9 -> 50.5 at 129 (192 rows), 39.3 -> 38.0 at 90 (96).  Parts of K: 0.94 to 1.03.
// Not where x is what comes from HBM (512 columns at 8,190 rows 34.2 -> 37.5): from four columns a row on; nor below 1,024 k (4,096 columns at 757 rows, K = 512 7.4 -> 7.9).
// -> W slots of the loop in phases, 0: the other loop.
static int tile_phases(int kind, int mode, bool xblk, int splits, int64_t M, int64_t N, int64_t K) {
    if (splits != 1 || xblk || mode > 2) return 0;
    if (kind == 2) return K >= 1024 && 4 * M <= N && (M - 1) % 128 >= (M > 512 ? 119 : 95) ? 6 : 0;
    if (kind == T_ODD) return mode == 0 ? (M > 160 ? 8 : 0) : M >= 80 && M <= 96 && K >= 4096 ? 8 : 0;
    if (kind == T_ODD + 1) return M >= 150 && M <= 192 && K >= 1024 ? 5 : 0;
    if (kind == T_ODD + 4) return 7;
    return 0;
}

// `add`: the launch that adds the parts too
template <int BM, int BN, int WGM, int WGN, int NS, int PER_CU, bool GATE>
static int tile_launch(GemmArgs a, int mode, int act, bool xblk, int splits, float* ws, hipStream_t st, bool add = true) {
    a.tiles_m = (int)((a.M + BM - 1) / BM);
    a.tiles_n = (a.N + BN - 1) / BN;
    a.group_m = 8;
    a.n_tiles = a.tiles_m * a.tiles_n * splits;
    const dim3 grid((unsigned)a.n_tiles), block(64 * WGM * WGN);
    if constexpr (BM == 128 && BN == 128) {
        if (tile_phases(2, mode, xblk, splits, a.M, a.N, a.K)) {
            if (mode == 1) hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WGM, WGN, 16, PER_CU, 1, false, false>), grid, block, 0, st, a, act, ws, splits);
            else hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WGM, WGN, 16, PER_CU, 0, false, false>), grid, block, 0, st, a, act, ws, splits);
            return evo_launch_status();
        }
    }
#define T_GO(MODE, XB, SPLIT) hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WGM, WGN, NS, PER_CU, MODE, XB, SPLIT>), grid, block, 0, st, a, act, ws, splits)
    if (splits == 1) {
        if (mode == 3) T_GO(3, false, false);
        else if (mode == 1) { if constexpr (GATE) T_GO(1, false, false); else return -1; }
        else if (xblk) T_GO(0, true, false);
        else T_GO(0, false, false);
        return evo_launch_status();
    }
    if (mode == 3) T_GO(3, false, true);
    else if (mode == 1) T_GO(1, false, true);
    else if (xblk) T_GO(0, true, true);
    else T_GO(0, false, true);
#undef T_GO
    if (!add) return evo_launch_status();
    const int64_t threads = a.M * ((mode == 1 ? a.N / 2 : a.N) / 8);
    const dim3 rgrid((unsigned)((threads + 255) / 256)), rblock(256);
    if (mode == 3) hipLaunchKernelGGL(gemm_parts_kernel<3>, rgrid, rblock, 0, st, a, act, ws, splits);
    else if (mode == 1) hipLaunchKernelGGL(gemm_parts_kernel<1>, rgrid, rblock, 0, st, a, act, ws, splits);
    else hipLaunchKernelGGL(gemm_parts_kernel<0>, rgrid, rblock, 0, st, a, act, ws, splits);
    return evo_launch_status();
}

template <int BM, int BN, int WGM, int WGN, int NS, int MODE>
static int tile_launch_odd(GemmArgs a, int act, hipStream_t st) {
    a.tiles_m = (int)((a.M + BM - 1) / BM);
    a.tiles_n = (a.N + BN - 1) / BN;
    a.group_m = 8;
    a.n_tiles = a.tiles_m * a.tiles_n;
    hipLaunchKernelGGL((gemm_tile_kernel<BM, BN, WGM, WGN, NS, 1, MODE, false, false>), dim3((unsigned)a.n_tiles), dim3(64 * WGM * WGN), 0, st, a, act, nullptr, 1);
    return evo_launch_status();
}

static bool dense_shape(int64_t mode, int64_t M, int64_t N, int64_t K) {
    return mode >= 0 && mode <= 3 && M > 0 && N > 0 && K > 0 && N % 256 == 0 && K % 64 == 0 && N < (1 << 30) && K < (1 << 22) && M < (1ll << 31) - 256
           && (mode != 3 || M % 256 == 0) && (mode != 2 || N * K * 2 < 0xffffffffll);
}

// `square`: without tiles of 160 to 224 rows
static int dense_plan(int64_t mode, bool stats, int64_t M, int64_t N, int64_t K, bool splits_ok, bool square, TilePlan (&plan)[2]) {
    splits_ok = splits_ok && M < 1024;                           // (from 1,024 rows on a row's result is the same bits in every batch: passes may be run in row groups)
    const bool persistent_ok = mode != 2 && K >= 128 && M * K * 2 < 0xffffffffll && N * K * 2 < 0xffffffffll;
    return tile_plan(M, N, K, mode == 2 ? 1 : (int)mode, stats, splits_ok, persistent_ok, !square, plan);
}

extern "C" int evo_dense_ws(int64_t mode, int64_t stats, int64_t M, int64_t N, int64_t K) {
    if (!dense_shape(mode, M, N, K)) return -1;
    int64_t most = 0;
    for (const bool square : {false, true}) {                    // (whichever form the call has)
        TilePlan plan[2];
        const int n = dense_plan(mode, stats != 0, M, N, K, true, square, plan);
        for (int i = 0; i < n; ++i)
            if (plan[i].splits > 1 && plan[i].splits * plan[i].rows * N * 4 > most) most = plan[i].splits * plan[i].rows * N * 4;
    }
    return (int)most;
}

extern "C" int evo_dense_launches(int64_t mode, int64_t stats, int64_t xblk, int64_t M, int64_t N, int64_t K, int64_t* out) {
    if (!dense_shape(mode, M, N, K) || !out || (xblk && (mode != 0 || M % 256 != 0))) return -1;
    TilePlan plan[2];
    const int n = dense_plan(mode, stats != 0, M, N, K, true, xblk != 0, plan);
    int64_t m0 = 0;
    for (int i = 0; i < n; ++i) {
        const TilePlan& t = plan[i];
        const TileKind tile = t.kind == T_PERSISTENT ? TileKind{256, 256, 0} : t.kind >= T_SHORT ? TileKind{short_rows[t.kind - T_SHORT], 256, 0} : kinds[t.kind];
        const int bm = mode == 3 ? tile.bn : tile.bm, bn = mode == 3 ? tile.bm : tile.bn;
        GemmArgs a;
        a.M = t.rows;
        a.ss_ld = (M + 255) / 256 * 256;
        const int64_t tiles_end = (t.rows + bm - 1) / bm * bm;   // (the persistent kernel stores the statistic of whole tiles)
        const int64_t stored = !stats ? 0 : t.kind != T_PERSISTENT && t_stat_rows(a) < tiles_end ? t_stat_rows(a) : tiles_end;
        const int64_t row[8] = {m0, t.rows, bm, bn, t.splits, t.kind >= T_SHORT, m0 + stored, tile_phases(t.kind, (int)mode, xblk != 0, t.splits, t.rows, N, K)};
        for (int k = 0; k < 8; ++k) out[8 * i + k] = row[k];
        m0 += t.rows;
    }
    return n;
}

extern "C" int evo_dense_plan(int64_t mode, int64_t stats, int64_t M, int64_t N, int64_t K, int64_t* out) {
    int64_t row[16];
    const int n = out ? evo_dense_launches(mode, stats, 0, M, N, K, row) : -1;
    for (int i = 0; i < n; ++i)
        for (int k = 0; k < 7; ++k) out[7 * i + k] = row[8 * i + k];
    return n;
}

// Parts of K that the norm behind a layer adds (rmsnorm_parts_kernel, closing_parts_kernel), 65 to 1,023 rows and up to 8,192 columns: without a launch of their own (5.5 us at 161 rows)
// parts pay in more layers and in larger numbers.  us, layer and norm in their own launches -> parts and norm, K = 4,096, 11,008 and 16,384 of 4,096 columns: 65 rows 20.5 -> 17.0,
// 33.9 -> 28.6, 39.3 -> 35.0; 161 rows 23.2 -> 22.3, 38.6 -> 36.3, 46.8 -> 44.2; 512 rows 39.1 -> 33.8, 64.3 -> 63, 81.5 -> 78.5; 8,192 x 8,192 56.4 -> 45.8 at 161 rows, 84 -> 81 at 512; over 842
// layers and sizes of 1,024 to 8,192 columns 1.17 x with rmsnorm_parts_kernel, over 601 1.12 x with closing_parts_kernel, weights cold, three and six of them 2 to 5 % behind.
// `parts_us`, fitted to 2,100 launches (5 % off them): the k-steps of a part, the parts' bytes, written and read, and the weights'; two, four and eight parts start a power of two
// apart and meet in the L2's channels.  One round of the chip; parts of 64 x 64 tiles as far as they have a CU each, eight of 192 rows on never (7 : 8 at K = 16,384 44 : 50).
// 128 x 128 in one sum and in step beyond 512 rows takes by its last row tile what its own cost rule does not know: 0.89 to 1.03 of that with 4 to 32 rows there, 1.07 to 1.17 with 100 and
// more, not 1.1 (4,096 columns of 5,632 at 900 rows 51.4 in one sum, 57.7 in two parts; 780 49.0 : 54.4; of 4,096 at 660 37.5 : 39.0, 600 41.2 : 38.2; at 540 it is taken still, 36.1 : 37.3).  And no parts of fewer than 13
// k-steps on 192 rows and more of up to 4,096 columns that 64 x 64 takes in one round: 3,072 columns of 3,072 at 151 rows 18.3 : 20.3, 4,096 of 4,096 at 138 20.7 : 21.5 (on 128 x 128, 16
// k-steps, they are ahead there: 145 rows 21.2 -> 19.6, 161 22.2 -> 20.2, all with the fp32 stream's norm).
struct PartsUs { int kind; double us, base; };
static const PartsUs parts_us[] = {{0, 0.21, 6.0}, {2, 0.43, 6.6}, {3, 0.55, 5.5}, {4, 0.665, 4.4}};
static TilePlan parts_plan(int64_t M, int64_t N, int64_t K) {
    TilePlan best = {-1, 0, 1e30, M}, own[2];
    // (narrow rows leave the norm's threads idle: 512 x 1,024 8.8 -> 10.4 at 540 rows, 1,024 x 4,096 18.8 -> 21.8 at 870)
    if (M < 65 || M >= 1024 || N > 8192 || (N < 2048 && 2 * M > N) || !dense_shape(0, M, N, K)) return best;
    const double cus = tile_cus(), nk = (double)(K / 64), power = 2.2e-9 * (double)M * N * K / 1.56;
    for (const PartsUs& p : parts_us) {
        const double tiles = (double)((M + kinds[p.kind].bm - 1) / kinds[p.kind].bm) * (double)((N + kinds[p.kind].bn - 1) / kinds[p.kind].bn);
        for (int s = 2; s <= 8 && tiles * s <= cus && nk / s >= 8 && (s < 8 || p.kind < 3); ++s) {
            const double us = ceil(nk / s) * p.us + p.base + 0.58e-6 * (double)(s * M * N * 4) + ((s & (s - 1)) == 0 ? 0.081e-6 : 0.066e-6) * (double)(N * K * 2);
            if (us < best.us) best = {p.kind, s, us, M};
        }
    }
    const int n = dense_plan(0, false, M, N, K, true, false, own);
    const bool tiles128 = n == 1 && own[0].kind == 2 && own[0].splits == 1 && M > 512 && !tile_phases(2, 0, false, 1, M, N, K);
    const double beyond = tiles128 ? 0.93 + 0.27 * (double)((M - 1) % 128 + 1) / 128 : 1.1;
    const double apart = beyond * (n == 2 ? own[0].us + own[1].us + 4.0 : own[0].us) + 1.3 + 0.47e-6 * (double)(M * N * 2);
    const bool few_steps = N <= 4096 && best.kind >= 3 && own[0].kind == 0 && own[0].splits == 1 && nk / best.splits < 13;
    if (few_steps || fmax(best.us, power) > 0.97 * apart) best.splits = 0;
    return best;
}

extern "C" int evo_dense_parts(int64_t M, int64_t N, int64_t K) { return parts_plan(M, N, K).splits; }

extern "C" int evo_dense_parts_bf16(const void* x, const void* w, float* ws, int64_t M, int64_t N, int64_t K, int64_t parts, void* stream) {
    const TilePlan t = parts_plan(M, N, K);
    if (!x || !w || !ws || parts < 2 || parts != t.splits || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)ws) & 15)) return -1;
    GemmArgs a;
    a.x = (const unsigned char*)x; a.w = (const unsigned char*)w; a.bias = nullptr; a.res = nullptr; a.y = nullptr;
    a.M = M; a.N = (int)N; a.K = (int)K;
    a.turn = M < 256 && K > 2048 ? 1 : 0;
    hipStream_t st = (hipStream_t)stream;
    if (t.kind == 0) return tile_launch<64, 64, 2, 2, 5, 2, false>(a, 0, 0, false, t.splits, ws, st, false);
    if (t.kind == 2) return tile_launch<128, 128, 4, 2, 5, 1, true>(a, 0, 0, false, t.splits, ws, st, false);
    if (t.kind == 3) return tile_launch<192, 128, 4, 2, 4, 1, true>(a, 0, 0, false, t.splits, ws, st, false);
    return tile_launch<256, 128, 4, 2, 3, 1, true>(a, 0, 0, false, t.splits, ws, st, false);
}

extern "C" int evo_dense_bf16(int64_t mode, int64_t act, int64_t xblk, const void* x, const void* w, const void* bias, const void* residual, void* y,
                              const float* row_scale, float* sumsq, int64_t ss_ld, int64_t M, int64_t N, int64_t K, int64_t act_cols, int64_t x_rows,
                              int64_t Tm, int64_t row_skip, void* ws, int64_t ws_bytes, void* stream) {
    if (!dense_shape(mode, M, N, K) || act < 0 || act > 3 || act_cols < 0 || act_cols > N || act_cols % 256 != 0) return -1;
    if ((mode == 1 || mode == 2) && (act > 1 || bias || residual || sumsq || xblk)) return -1;
    if (mode == 3 && (act || residual || sumsq || xblk)) return -1;
    if ((row_scale && (residual || sumsq)) || (sumsq && (!residual || ss_ld < (M + 255) / 256 * 256))) return -1;
    if (mode == 0 && act && (residual || row_scale)) return -1;
    if (xblk && (M % 256 != 0 || row_scale || act)) return -1;
    if (mode == 3 && row_scale ? (Tm <= 0 || Tm % 256 != 0 || M % Tm != 0 || row_skip < 0 || row_skip > 0x7fff || x_rows < M + (M / Tm - 1) * row_skip)
                               : (x_rows != 0 || Tm != 0 || row_skip != 0)) return -1;
    // blocks of 128 rows of x lie whole in a tile; the persistent kernel has 32 bits for an operand's bytes, and tokens that are skipped between rows count (256 rows refuse)
    const bool square = xblk || (mode == 3 && row_scale && x_rows * K * 2 >= 0xffffffffll);
    TilePlan plan[2];
    int n = dense_plan(mode, sumsq != nullptr, M, N, K, true, square, plan);
    for (int i = 0; i < n; ++i)
        if (plan[i].splits > 1 && (!ws || ws_bytes < plan[i].splits * plan[i].rows * N * 4)) {
            n = dense_plan(mode, sumsq != nullptr, M, N, K, false, square, plan);
            break;
        }
    // (from 256 rows on the order of k is the persistent kernel's.  us, in step -> in turn: K = 2,048, 4,096 columns 8.5 -> 9.1 at 65 rows, 22,016 24.8 -> 23.4; [W1; W2] as it is
    //  with halves a power of two apart, 8,192 gated columns 37.3 -> 42.7)
    const int turn = M < 256 && K > 2048 && !(mode == 2 && (N & (N - 1)) == 0) ? 1 : 0;
    int64_t m0 = 0;
    for (int i = 0; i < n; ++i) {
        const TilePlan& t = plan[i];
        const unsigned char* xi = (const unsigned char*)x + m0 * K * 2;
        const uint16_t* ri = residual ? (const uint16_t*)residual + m0 * N : nullptr;
        uint16_t* yi = (uint16_t*)y + m0 * (mode == 1 || mode == 2 ? N / 2 : N);
        const float* si = row_scale ? row_scale + m0 : nullptr;
        float* qi = sumsq ? sumsq + m0 : nullptr;
        int rc;
        if (t.kind == T_PERSISTENT) {
            if (mode == 1) rc = gemmr_gate(xi, si, w, yi, t.rows, N / 2, K, act, stream);
            else if (mode == 3) rc = row_scale ? evo_linear_t_mfma_nf_bf16(x, row_scale, w, bias, y, M, N, K, x_rows, Tm, row_skip, stream)
                                               : evo_linear_t_mfma_bf16(x, w, bias, y, M, N, K, stream);
            else if (xblk) rc = evo_linear_xblk_mfma_nf_bf16(xi, w, bias, ri, yi, qi, ss_ld, t.rows, N, K, stream);
            else if (act) rc = evo_linear_act_mfma_bf16(xi, w, bias, yi, t.rows, N, K, act_cols, act, stream);
            else rc = evo_linear_mfma_nf_bf16(xi, w, bias, ri, yi, si, qi, ss_ld, t.rows, N, K, stream);
        } else {
            GemmArgs a;
            a.x = xi; a.w = (const unsigned char*)w; a.bias = (const uint16_t*)bias; a.res = ri; a.y = yi;
            a.M = t.rows; a.N = (int)N; a.K = (int)K;
            a.rs = si; a.ss = qi; a.ss_ld = ss_ld; a.act_cols = act ? (int)act_cols : 0; a.turn = turn;
            if (mode == 2) a.w_rows = N;
            if (mode == 3) {                                     // the rows of the launch are the weight's, its columns the tokens
                a.x = (const unsigned char*)w; a.w = (const unsigned char*)x;
                a.M = N; a.N = (int)M;
                if (row_scale) { a.w_rows = x_rows; a.tm_tiles = (int)(Tm / 256); a.row_skip = (int)row_skip; }
            }
            const int tm = mode == 2 ? 1 : (int)mode, phases = tile_phases(t.kind, tm, xblk != 0, t.splits, a.M, a.N, a.K);
            float* f = (float*)ws;
            hipStream_t st = (hipStream_t)stream;
            if (t.kind >= T_SHORT) rc = t.kind == T_SHORT ? gemmr_rows160(a, tm, (int)act, st) : t.kind == T_SHORT + 1 ? gemmr_rows192(a, tm, (int)act, st) : gemmr_rows224(a, tm, (int)act, st);
            else if (t.kind == 0) rc = tile_launch<64, 64, 2, 2, 5, 2, false>(a, tm, (int)act, xblk != 0, t.splits, f, st);
            else if (t.kind == 1) rc = tile_launch<128, 64, 4, 1, 3, 2, true>(a, tm, (int)act, xblk != 0, t.splits, f, st);
            else if (t.kind == 2) rc = tile_launch<128, 128, 4, 2, 5, 1, true>(a, tm, (int)act, xblk != 0, t.splits, f, st);
            else if (t.kind == 3) rc = tile_launch<192, 128, 4, 2, 4, 1, true>(a, tm, (int)act, xblk != 0, t.splits, f, st);
            else if (t.kind == 4) rc = tile_launch<256, 128, 4, 2, 3, 1, true>(a, tm, (int)act, xblk != 0, t.splits, f, st);
            else if (t.kind == 5) rc = tile_launch<128, 256, 2, 4, 3, 1, true>(a, tm, (int)act, xblk != 0, t.splits, f, st);
            else if (xblk || tm > 1 || (tm == 1 ? t.kind == T_ODD + 2 || t.kind == T_ODD + 3 : t.kind == T_ODD + 1 || t.kind == T_ODD + 4)) rc = -1;
            else if (t.kind == T_ODD + 4) rc = tile_launch_odd<128, 96, 4, 1, 17, 1>(a, (int)act, st);
            else if (tm == 0 && t.kind == T_ODD) rc = phases ? tile_launch_odd<96, 96, 2, 3, 18, 0>(a, (int)act, st) : tile_launch_odd<96, 96, 2, 3, 6, 0>(a, (int)act, st);
            else if (t.kind == T_ODD + 3) rc = tile_launch_odd<64, 96, 2, 2, 7, 0>(a, (int)act, st);
            else if (t.kind == T_ODD) rc = phases ? tile_launch_odd<96, 96, 2, 3, 18, 1>(a, (int)act, st) : tile_launch_odd<96, 96, 2, 3, 6, 1>(a, (int)act, st);
            else if (t.kind == T_ODD + 1) rc = phases ? tile_launch_odd<192, 96, 4, 3, 15, 1>(a, (int)act, st) : tile_launch_odd<192, 96, 4, 3, 4, 1>(a, (int)act, st);
            else rc = tile_launch_odd<96, 48, 3, 1, 8, 0>(a, (int)act, st);
        }
        if (rc != 0) return rc;
        m0 += t.rows;
    }
    return 0;
}
