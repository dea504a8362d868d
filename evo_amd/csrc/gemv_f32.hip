// fp32 dense layers of up to four rows:  y [M, N] = x [M, K] w [N, K]^T (+ bias), all fp32: a decoding step of an fp32 model.
//
// The weight's bytes bound it (a copy reaches 4.8 TB/s, reads alone 6.3).  Every CU takes a contiguous run of rows of w, one workgroup each: a wave owns an eighth of K
// and keeps its part of x in registers, so that nothing but w moves, in whole lines of 1 KiB a request, 8 to 16 of them out per wave, each register filled again as
// soon as its products are taken.  Sums over lanes are taken for a batch of rows at once, sums over waves once at the end.  us, library -> here, 1 / 4 rows (MI355X):
// 22,016 x 4,096 72 -> 57 / 75 -> 63 (6.3 / 5.7 TB/s), 16,384 x 4,096 53 -> 42 / 53 -> 44, 4,096 x 16,384 50 -> 43 / 50 -> 44, 4,096 x 11,008 42 -> 30 / 42 -> 32, 4,096 x 4,096 16.5 ->
// 12.6 / 16.5 -> 13.8, 512 x 4,096 10 -> 4 / 10 -> 5.  Error against 64 bits at K = 4,096 5.8e-7 -> 1.0e-7, at 16,384 1.2e-6 -> 1.3e-7.
// Tried: lane sums one value after the other (6 steps each, two through LDS: 71 us for 22,016 x 4,096 at 4 rows); more rows out per wave (4 rows of 22 KB requests
// a wave spill at 4 rows of x: 57 us for 4,096 x 11,008), fewer (5 % slower up to K = 6,144).
#include "common.h"
#include "../../include/evo_mi355x.h"

#define FV_WAVES 8                           // a wave per eighth of K
#define FV_ROWS 512                          // rows of w that a workgroup can take (64 KB of sums)

struct FvArgs { const float* x; const float* w; const float* bias; float* y; int64_t N; int K; };

// Workgroup = a contiguous run of rows of w; wave = an eighth of K, its part of x in registers; NCH requests of 1 KiB a row, RB rows of them out at a time, each
// register refilled as soon as its products are taken.  (RB: 8 to 16 requests out where the registers hold them, see the sizes above.)
template <int M, int NCH, int RB>
__global__ __launch_bounds__(64 * FV_WAVES, 2) void gemv_f32_kernel(FvArgs a) {
    extern __shared__ __attribute__((aligned(16))) float part[];        // [rows][M][waves]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n0 = a.N * blockIdx.x / gridDim.x;
    const int rows = (int)(a.N * (blockIdx.x + 1) / gridDim.x - n0), slice = a.K / FV_WAVES;
    const int k0 = wave * slice + lane * 4;
    const bool last = (NCH - 1) * 256 + lane * 4 < slice;        // (the last request may not reach every lane)
    f32x4_t xr[M][NCH];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            xr[m][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if (c + 1 < NCH || last) xr[m][c] = *(const f32x4_t*)(a.x + (int64_t)m * a.K + k0 + c * 256);
        }
    const float* w = a.w + n0 * a.K + k0;
    f32x4_t wr[RB][NCH];
    auto fetch = [&](int row, int c, f32x4_t& d) {
        const float* p = w + (int64_t)min(row, rows - 1) * a.K + c * 256;
        if (c + 1 < NCH) d = __builtin_nontemporal_load((const f32x4_t*)p);
        else if (last) d = __builtin_nontemporal_load((const f32x4_t*)p);
    };
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            wr[r][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};              // (lanes that the last request does not reach)
            fetch(r, c, wr[r][c]);
        }
    // sums over the wave of a batch's RB x M values: the halves of two values change places, then the rows of 16 lanes, then four steps inside a row: 2.5 steps a
    // value where one after the other takes six, two of them through LDS
    constexpr int V = (RB * M + 3) / 4 * 4;
    auto batch = [&](int base, bool more) {
        float sum[V];
#pragma unroll
        for (int i = 0; i < V; ++i) sum[i] = 0.f;
#pragma unroll
        for (int r = 0; r < RB; ++r)
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
#pragma unroll
                for (int m = 0; m < M; ++m)
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[r * M + m] = fmaf(wr[r][c][e], xr[m][c][e], sum[r * M + m]);
                if (more) fetch(base + RB + r, c, wr[r][c]);
            }
#pragma unroll
        for (int i = 0; i < V / 4; ++i) {
            float u[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(sum[4 * i + 2 * h]), __float_as_uint(sum[4 * i + 2 * h + 1]), false, false);
                u[h] = __uint_as_float(t[0]) + __uint_as_float(t[1]);
            }
            const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(u[0]), __float_as_uint(u[1]), false, false);
            float v = __uint_as_float(t[0]) + __uint_as_float(t[1]);     // row q of 16 lanes: value 4 i + (q >> 1) + 2 (q & 1)
            v += dpp_fetch<EVO_DPP_XOR1>(v);
            v += dpp_fetch<EVO_DPP_XOR2>(v);
            v += dpp_fetch<EVO_DPP_HALF_MIRROR>(v);
            v += dpp_fetch<EVO_DPP_MIRROR>(v);
            const int j = 4 * i + (lane >> 5) + 2 * ((lane >> 4) & 1);
            if ((lane & 15) == 0 && j < RB * M && base * M + j < rows * M) part[(base * M + j) * FV_WAVES + wave] = v;
        }
    };
    int base = 0;
    for (; base + RB < rows; base += RB) batch(base, true);
    batch(base, false);
    __syncthreads();
    for (int i = threadIdx.x; i < rows * M; i += 64 * FV_WAVES) {
        const int r = i / M, m = i - r * M;
        const f32x4_t u = *(const f32x4_t*)(part + i * FV_WAVES), v = *(const f32x4_t*)(part + i * FV_WAVES + 4);
        const float s = ((u[0] + u[1]) + (u[2] + u[3])) + ((v[0] + v[1]) + (v[2] + v[3]));
        a.y[m * a.N + n0 + r] = a.bias ? s + a.bias[n0 + r] : s;
    }
}

template <int M>
static int fv_launch(const FvArgs& a, int blocks, size_t lds, hipStream_t st) {
    const int nch = (a.K / FV_WAVES + 255) / 256;
#define FV_GO(NCH, RB) case NCH: hipLaunchKernelGGL((gemv_f32_kernel<M, NCH, RB>), dim3(blocks), dim3(64 * FV_WAVES), lds, st, a); break
    switch (nch) {
        FV_GO(1, 4); FV_GO(2, 4); FV_GO(3, 4); FV_GO(4, 2); FV_GO(5, 2); FV_GO(6, 2); FV_GO(7, 1); FV_GO(8, 1);
        default: return -1;
    }
#undef FV_GO
    return evo_launch_status();
}

extern "C" int evo_linear_few_f32(const float* x, const float* w, const float* bias, float* y, int64_t M, int64_t N, int64_t K, void* stream) {
    if (M < 1 || M > 4 || N < 1 || K < 32 || K % 32 != 0 || K > 16384 || N > 0x3fffffff) return -1;
    if (!x || !w || !y || (((uintptr_t)x | (uintptr_t)w) & 15) || (((uintptr_t)bias | (uintptr_t)y) & 3)) return -1;
    static const int cus = [] {
        int dev = 0, c = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
        return c < 8 ? 8 : c;
    }();
    int64_t blocks = N < cus ? N : cus;
    if ((N + blocks - 1) / blocks > FV_ROWS) blocks = (N + FV_ROWS - 1) / FV_ROWS;
    const FvArgs a = {x, w, bias, y, N, (int)K};
    const size_t lds = (size_t)((N + blocks - 1) / blocks) * M * FV_WAVES * 4;
    hipStream_t st = (hipStream_t)stream;
    switch (M) {
        case 1: return fv_launch<1>(a, (int)blocks, lds, st);
        case 2: return fv_launch<2>(a, (int)blocks, lds, st);
        case 3: return fv_launch<3>(a, (int)blocks, lds, st);
        default: return fv_launch<4>(a, (int)blocks, lds, st);
    }
}
