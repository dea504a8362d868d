// fp32 dense layers on the bf16 matrix cores of gfx950:  y [M, N] = x [M, K] w [N, K]^T (+ bias), all fp32.
//
// Every fp32 value is the exact sum of three bf16 ones, x = h + m + l: h the value rounded to bf16, m the rest rounded to bf16, l what is left (at most
// 8 bits, so exact).  A product is h h' + (h m' + m h') + (h l' + l h' + m m') with fp32 accumulation; what is left out, m l' + l m' + l l', is at most
// 2^-24 of a product, as much as an fp32 multiplication rounds, and 2^-27 in the mean square (with h cut instead of rounded 2^-22).  A lone product is
// within 2^-22.7 (the matrix cores' adders cut; 2^-24.8 in the mean square, fp32 2^-25.2), sums of K >= 256 are nearer to 64 bits than the fp32
// MFMA's (1,024 columns, 40 to 1,290 rows: K = 256 2.4e-7 against 2.9e-7, 4,096 3.5e-7 to 4.1e-7 against 5.7e-7 to 1.1e-6, 11,008 6.0e-7 to 7.0e-7
// against 0.9e-6 to 1.9e-6; unsplit 4,096 1.00e-6 against 1.15e-6).
// Six bf16 MFMAs in place of one fp32 MFMA at 1/16 of their rate.
//
// Workgroup = BM x BN of y, waves of (BM / WGM) x (BN / WGN) in 32 x 32 x 16 MFMAs, computed transposed (A = rows of w, B = rows of x) so that a lane
// holds four neighbouring columns of one row of y.  K is walked in steps of 32: a thread loads 8 neighbouring fp32 of a row, splits them in registers
// and writes the three 16-byte pieces to the planes of an LDS stage; rows of 64 B with the piece index XORed by (row >> 2) & 3: 16 lanes reading one
// piece of 16 rows touch every bank once.  One stage and two barriers per step: the workgroups that share a CU split and multiply in turn (two
// stages and one barrier at 256 x 128 were 1.1 to 1.3 times as slow: one workgroup per CU).
#include "gemm_f32.h"
#include "../../include/evo_mi355x.h"
#define F3_ROWB 64

struct F3Args {
    const float* x; const float* w; const float* bias; float* y; float* parts;
    int64_t M; int N, K, tiles_m, tiles_n, n_tiles, group_m, splits;
};

template <int BM, int BN, int WGM, int WGN, int PER_CU, bool SPLIT>
__global__ __launch_bounds__(64 * WGM * WGN, PER_CU * WGM * WGN / 4) void gemm_f32_kernel(F3Args a) {
    constexpr int NT = 64 * WGM * WGN, TM = BM / WGM / 32, TN = BN / WGN / 32, ROWS = BM + BN, PLANE = ROWS * F3_ROWB, STAGE = 3 * PLANE, NP = ROWS * 4 / NT;
    static_assert(ROWS * 4 % NT == 0, "whole pieces per thread");
    __shared__ __attribute__((aligned(16))) unsigned char smem[STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = lane >> 5, l31 = lane & 31;
    const int wm = wave / WGN, wn = wave % WGN;
    // block b runs on XCD b % 8: every XCD gets a contiguous run of tiles, group_m row tiles next to each other before the next column tile
    int tile, part = 0;
    {
        const int bid = blockIdx.x, q = a.n_tiles >> 3, r = a.n_tiles & 7, xcd = bid & 7, slot = bid >> 3;
        tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
    }
    if (SPLIT) { part = tile % a.splits; tile /= a.splits; }
    const int per = a.group_m * a.tiles_n, g = tile / per, gm0 = g * a.group_m, gsz = min(a.tiles_m - gm0, a.group_m);
    const int tm = gm0 + (tile - g * per) % gsz, tn = (tile - g * per) / gsz;
    const int64_t m0 = (int64_t)tm * BM;
    const int n0 = tn * BN;
    const int nk = a.K / F3_BK, k0 = SPLIT ? (int)((int64_t)nk * part / a.splits) : 0, k1 = SPLIT ? (int)((int64_t)nk * (part + 1) / a.splits) : nk;

    const float* src[NP];
    int dst[NP];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        const int i = p * NT + tid, r = i >> 2, s = i & 3;
        int64_t m = m0 + r;
        int n = n0 + r - BM;
        if (m > a.M - 1) m = a.M - 1;                          // rows past the end: any row that is there (never written)
        if (n > a.N - 1) n = a.N - 1;
        src[p] = (r < BM ? a.x + m * a.K : a.w + (int64_t)n * a.K) + (int64_t)k0 * F3_BK + s * 8;
        dst[p] = r * F3_ROWB + ((s ^ (r >> 2)) & 3) * 16;
    }
    float4 st[NP][2];
    float top[NP];                                             // the largest of this thread's values of each row
#pragma unroll
    for (int p = 0; p < NP; ++p) top[p] = 0.f;
    auto fetch = [&]() {
#pragma unroll
        for (int p = 0; p < NP; ++p) { st[p][0] = *(const float4*)src[p]; st[p][1] = *(const float4*)(src[p] + 4); src[p] += F3_BK; }
    };
    auto put = [&]() {
#pragma unroll
        for (int p = 0; p < NP; ++p) {
            uint4 h, m, l;
            f3_split(st[p][0], st[p][1], h, m, l);
            f3_row_max(top[p], st[p][0], st[p][1]);
            *(uint4*)(smem + dst[p]) = h;
            *(uint4*)(smem + PLANE + dst[p]) = m;
            *(uint4*)(smem + 2 * PLANE + dst[p]) = l;
        }
    };
    int xo[TM][2], wo[TN][2];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
        for (int i = 0; i < TM; ++i) { const int r = wm * (BM / WGM) + i * 32 + l31; xo[i][ks] = r * F3_ROWB + (((2 * ks + half) ^ (r >> 2)) & 3) * 16; }
#pragma unroll
        for (int j = 0; j < TN; ++j) { const int r = BM + wn * (BN / WGN) + j * 32 + l31; wo[j][ks] = r * F3_ROWB + (((2 * ks + half) ^ (r >> 2)) & 3) * 16; }
    }
    f32x16_t acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    auto multiply = [&]() {
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8_t xf[3][TM], wf[3][TN];
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
                for (int i = 0; i < TM; ++i) xf[pl][i] = *(const bf16x8_t*)(smem + pl * PLANE + xo[i][ks]);
#pragma unroll
                for (int j = 0; j < TN; ++j) wf[pl][j] = *(const bf16x8_t*)(smem + pl * PLANE + wo[j][ks]);
            }
            constexpr int PX[6] = {0, 2, 1, 0, 1, 0}, PW[6] = {2, 0, 1, 1, 0, 0};        // the smallest products first
#pragma unroll
            for (int q = 0; q < 6; ++q)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[PW[q]][j], xf[PX[q]][i], acc[i][j], 0, 0, 0);
        }
    };
    fetch();
    for (int k = k0; k < k1; ++k) {
        put();
        __syncthreads();
        if (k + 1 < k1) fetch();
        multiply();
        __syncthreads();
    }
    float* row_max = (float*)smem;                             // (a row of zeros: -inf, which no output is under)
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        top[p] = fmaxf(top[p], dpp_fetch<EVO_DPP_XOR1>(top[p]));
        top[p] = fmaxf(top[p], dpp_fetch<EVO_DPP_XOR2>(top[p]));
        if ((tid & 3) == 0) row_max[(p * NT + tid) >> 2] = top[p] > 0.f ? top[p] : -INFINITY;
    }
    __syncthreads();
    const float least = (float)(k1 - k0) * (F3_BK * 0x1p-98f);
    float wide = 0.f;                                          // the largest of this lane's columns
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const float4 w = *(const float4*)(row_max + BM + wn * (BN / WGN) + j * 32 + q * 8 + half * 4);
            wide = fmaxf(fmaxf(fmaxf(wide, w.x), fmaxf(w.y, w.z)), w.w);
        }
    auto at = [&](int64_t m, int n) { return SPLIT ? a.parts + ((int64_t)part * a.M + m) * a.N + n : a.y + m * a.N + n; };
    bool look = false;                                         // an output may have to be taken again
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int r = wm * (BM / WGM) + i * 32 + l31;
        const int64_t m = m0 + r;
        if (m >= a.M) continue;
        float lo = INFINITY, hi = 0.f;
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float4 v = make_float4(acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]);
                f3_range(lo, hi, v.x, v.y);
                f3_range(lo, hi, v.z, v.w);
                const int n = n0 + wn * (BN / WGN) + j * 32 + q * 8 + half * 4;
                if (n >= a.N) continue;
                if (!SPLIT && a.bias) { const float4 b = *(const float4*)(a.bias + n); v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w; }
                *(float4*)at(m, n) = v;
            }
        look |= !(lo >= fmaf(least, wide, fmaf(least, fmaxf(row_max[r], 0.f), least)) && hi <= 3.402823466e38f);
    }
    f3_again<TM, TN>(acc, look, a.x, a.w, SPLIT ? nullptr : a.bias, m0 + wm * (BM / WGM), a.M, n0 + wn * (BN / WGN), a.N, a.K, k0, k1, row_max + wm * (BM / WGM),
                     row_max + BM + wn * (BN / WGN), at);
}

// the sum of the parts of K
__global__ __launch_bounds__(256) void gemm_f32_parts_kernel(F3Args a) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= a.M * a.N) return;
    const int64_t m = i / a.N;
    const int n = (int)(i - m * a.N);
    float4 v = *(const float4*)(a.parts + i);
    for (int s = 1; s < a.splits; ++s) {
        const float4 p = *(const float4*)(a.parts + (int64_t)s * a.M * a.N + i);
        v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
    }
    if (a.bias) { const float4 b = *(const float4*)(a.bias + n); v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w; }
    *(float4*)(a.y + i) = v;
}

// ---------------------------------------------------------------------------------------------------------------- which tile
// One k-step (32 deep) of the n tiles that share a CU takes `start` + n `each` us (at most `per_cu` share it: LDS and registers), fitted to 33 to 4,000
// rows of eight layers.  The matrix cores bound the larger tiles: 128 x 128 with two on a CU 222 TF, 256 x 256 235 TF (six bf16 products each: 1.4 PF, what a
// large bf16 product reaches).  Against the library's fp32 MFMA layers (us, K = 4,096, MI355X,
// back to back on the GPU, before -> here): 4,096 columns 38 -> 41 at 65 rows, 56 -> 49 at 161, 90 -> 82 at 300, 1,002 -> 627 at 4,000; 22,016 columns
// 160 -> 135, 290 -> 232, 456 -> 359, at 1,500 2,212 -> 1,424; K = 11,008, 4,096 columns 89 -> 92, 140 -> 117, 222 -> 190, at 1,500 1,039 -> 703.  Small layers are left
// to the library (HipOps._f32_layer_pays).  Error against 64 bits (random normal operands,
// 4,096 x 4,096): 1.00e-6 unsplit, 7.1e-7 in two parts, 5.0e-7 in four, 3.5e-7 in eight; library 1.14e-6.
struct F3Kind { int bm, bn, per_cu; double start, each; };
static const F3Kind f3_kinds[] = {{64, 64, 5, 0.29, 0.33}, {64, 128, 4, 0.30, 0.655}, {128, 128, 2, 0.20, 1.11}, {256, 256, 1, 0.10, 4.36}};
struct F3Plan { int kind, splits; double us; };

static F3Plan f3_plan(int64_t M, int64_t N, int64_t K) {
    static const int cus = [] {
        int dev = 0, c = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
        return c < 8 ? 8 : c;
    }();
    F3Plan best = {0, 1, 1e300};
    const double memory = 4.0 * ((double)N * K + (double)M * K) / 4.2e6;
    for (int c = 0; c < 4; ++c) {
        const F3Kind& k = f3_kinds[c];
        const double tiles = (double)((M + k.bm - 1) / k.bm) * (double)((N + k.bn - 1) / k.bn);
        for (int s = 1; s <= 8; ++s) {
            if (s == 5 || s == 7) continue;
            if (s > 1 && (K / F3_BK / s < 8 || tiles * s > 12.0 * cus || (double)s * M * N * 4 > 256e6)) break;
            const double steps = ceil((double)(K / F3_BK) / s), n = ceil(tiles * s / cus), rest = fmod(n, k.per_cu), full = (n - rest) / k.per_cu;
            const double work = steps * (full * (k.start + k.per_cu * k.each) + (rest > 0 ? k.start + rest * k.each : 0.0)) + 5.0;
            double us = work > memory ? work + 0.085 * memory : memory + 0.085 * work;
            if (s > 1) us += 6.0 + (double)s * M * N * 8 / 9.1e6;
            if (us < best.us) best = {c, s, us};
        }
    }
    return best;
}

double f3_tiles_us(int64_t M, int64_t N, int64_t K) { return f3_plan(M, N, K).us; }

template <int BM, int BN, int WGM, int WGN, int PER_CU>
static int f3_launch(F3Args a, hipStream_t st) {
    const int64_t tm = (a.M + BM - 1) / BM, tn = ((int64_t)a.N + BN - 1) / BN;
    if (tm * tn * a.splits > 0x7fffffff) return -1;
    a.tiles_m = (int)tm;
    a.tiles_n = (int)tn;
    a.n_tiles = (int)(tm * tn * a.splits);
    a.group_m = 8;
    const dim3 grid((unsigned)a.n_tiles), block(64 * WGM * WGN);
    if (a.splits == 1) {
        hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WGM, WGN, PER_CU, false>), grid, block, 0, st, a);
        return evo_launch_status();
    }
    hipLaunchKernelGGL((gemm_f32_kernel<BM, BN, WGM, WGN, PER_CU, true>), grid, block, 0, st, a);
    const int rc = evo_launch_status();
    if (rc) return rc;
    hipLaunchKernelGGL(gemm_f32_parts_kernel, dim3((unsigned)((a.M * a.N / 4 + 255) / 256)), dim3(256), 0, st, a);
    return evo_launch_status();
}

static bool f3_ok(int64_t M, int64_t N, int64_t K) {
    return M >= 0 && N > 0 && K >= F3_BK && M <= 0x7fffffff && N <= 0x7fffff00 && K <= 0x7fffff00 && N % 4 == 0 && K % F3_BK == 0 && (double)M * N <= 4e11;
}

extern "C" int evo_linear_f32_ws(int64_t M, int64_t N, int64_t K) {
    if (!f3_ok(M, N, K)) return -1;
    const F3Plan p = f3_plan(M, N, K);
    return p.splits > 1 ? p.splits : 0;
}

extern "C" int evo_linear_f32_plan(int64_t M, int64_t N, int64_t K, int64_t* out) {
    if (!f3_ok(M, N, K) || !out) return -1;
    const F3Plan p = f3_plan(M, N, K);
    out[0] = f3_kinds[p.kind].bm;
    out[1] = f3_kinds[p.kind].bn;
    out[2] = p.splits;
    return 0;
}

extern "C" int evo_linear_f32(const float* x, const float* w, const float* bias, float* y, int64_t M, int64_t N, int64_t K, float* ws, int64_t ws_bytes, void* stream) {
    if (!f3_ok(M, N, K)) return -1;
    if (M == 0) return 0;
    if (!x || !w || !y || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)y | (uintptr_t)ws) & 15)) return -1;
    F3Plan p = f3_plan(M, N, K);
    if (p.splits > 1 && (!ws || ws_bytes < p.splits * M * N * 4)) p.splits = 1;
    F3Args a = {x, w, bias, y, ws, M, (int)N, (int)K, 0, 0, 0, 0, p.splits};
    hipStream_t st = (hipStream_t)stream;
    switch (p.kind) {
        case 0: return f3_launch<64, 64, 2, 2, 5>(a, st);
        case 1: return f3_launch<64, 128, 2, 2, 4>(a, st);
        case 2: return f3_launch<128, 128, 2, 2, 2>(a, st);
        default: return f3_launch<256, 256, 2, 4, 1>(a, st);
    }
}
