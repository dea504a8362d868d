// Skinny dense layer for decoding: y[M,N] = x[M,K] . W[N,K]^T (+ bias[N]) (+ residual[M,N]), M <= 16.
//
// Two kernels.  gemv_kernel (M <= 4, or any K % 8 == 0 shape): dot2 on the VALU, below.  skinny_mfma_kernel
// (5 <= M <= 16, K % 32 == 0): the batch rows become the N side of v_mfma_f32_16x16x32_bf16 -- with 5+ rows the VALU
// form spends more on re-reading x from L2 (M loads per R weight loads) than on the weights; here one 1-KiB x
// fragment meets one 1-KiB weight fragment per MFMA and the math is free.
//
// At batch 1-8 a decode step streams all 12.9 GB of weights once and is bound by HBM, not by MFMA: through
// hipBLASLt's tile GEMM it ran at ~2.5 TB/s (5.2 ms/token).  This kernel is the weight-streaming form: one wave
// owns R consecutive output rows, its lanes stride over K with 16-byte non-temporal loads straight into
// VGPRs (no LDS round trip -- the operand is streamed once and shared with nobody), accumulates with
// v_dot2c_f32_bf16 (two bf16 MACs per lane-op, fp32 accumulate, no unpack), and reduces across the wave at
// the end.  x (<= 8 x K bf16) is re-read by every wave and lives in L2.
// Entry point and reference citation: include/evo_mi355x.h.
#include "common.h"
#include "../../include/evo_mi355x.h"

typedef __bf16 dot_bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot8(const uint4& a, const uint4& b, float acc) {
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dot_bf16x2, a.x), __builtin_bit_cast(dot_bf16x2, b.x), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dot_bf16x2, a.y), __builtin_bit_cast(dot_bf16x2, b.y), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dot_bf16x2, a.z), __builtin_bit_cast(dot_bf16x2, b.z), acc, false);
    acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(dot_bf16x2, a.w), __builtin_bit_cast(dot_bf16x2, b.w), acc, false);
    return acc;
}

__device__ __forceinline__ uint4 ld_stream(const uint4* p) {
    typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
    u32x4 v = __builtin_nontemporal_load((const u32x4*)p);
    return make_uint4(v[0], v[1], v[2], v[3]);
}

// SPLIT: the four waves of a workgroup share the SAME R rows and each takes every fourth 64-vector slice of K (the
// partial sums meet in LDS).  Used for the narrow layers (N <= 4096: out_filter_dense, out_proj, l3), where one wave
// per R rows leaves the chip with too few loads in flight: 3.3 -> see tools/bench_gemv.py.
// an ungated feed-forward's activation on the way out: act 3 = square of relu, else none
__device__ __forceinline__ float out_act(float o, int act) {
    const float z = fmaxf(o, 0.f);
    return act == 3 ? z * z : o;
}

template <int M, int R, bool SPLIT>
__global__ __launch_bounds__(256) void gemv_kernel(const uint4* __restrict__ x, const uint4* __restrict__ w,
                                                   const uint16_t* __restrict__ bias, const uint16_t* res,
                                                   uint16_t* y, int N, int nvec, int act) {   // res may alias y
    __shared__ float part[SPLIT ? 4 * R * M : 1];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n0 = SPLIT ? (int64_t)blockIdx.x * R : ((int64_t)blockIdx.x * 4 + wave) * R;
    if (n0 >= N) return;                                     // (workgroup-uniform when SPLIT)
    const uint4* wrow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t n = n0 + r < N ? n0 + r : N - 1;            // rows past the end are computed on a clamp, not stored
        wrow[r] = w + n * nvec;
    }
    // the storing lane requests its bias / residual values NOW: fetched after the reduction they were a dependent ~1 us tail on
    // a launch whose whole stream is 5-17 us (out_filter_dense, out_proj, l3)
    const bool ep_lane = lane == 0 && (!SPLIT || wave == 0);
    uint16_t pf_b[R], pf_r[R][M];
    if (ep_lane) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t n = n0 + r < N ? n0 + r : N - 1;
            pf_b[r] = bias ? bias[n] : (uint16_t)0;
#pragma unroll
            for (int m = 0; m < M; ++m) pf_r[r][m] = res ? res[(int64_t)m * N + n] : (uint16_t)0;
        }
    }
    float acc[R][M];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.f;

    constexpr int ST = SPLIT ? 256 : 64;                     // slice stride of this wave
    int v = SPLIT ? wave * 64 + lane : lane;
    for (; v + ST < nvec; v += 2 * ST) {                     // two k-slices per trip: 2R weight loads in flight
        uint4 w0[R], w1[R];
#pragma unroll
        for (int r = 0; r < R; ++r) { w0[r] = ld_stream(wrow[r] + v); w1[r] = ld_stream(wrow[r] + v + ST); }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint4 x0 = x[(int64_t)m * nvec + v], x1 = x[(int64_t)m * nvec + v + ST];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r][m] = dot8(w1[r], x1, dot8(w0[r], x0, acc[r][m]));
        }
    }
    for (; v < nvec; v += ST) {
        uint4 w0[R];
#pragma unroll
        for (int r = 0; r < R; ++r) w0[r] = ld_stream(wrow[r] + v);
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint4 x0 = x[(int64_t)m * nvec + v];
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r][m] = dot8(w0[r], x0, acc[r][m]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = wave_sum(acc[r][m]);
    if (SPLIT) {
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int m = 0; m < M; ++m) part[(wave * R + r) * M + m] = acc[r][m];
        }
        __syncthreads();
        if (wave != 0) return;
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int m = 0; m < M; ++m)
                acc[r][m] = part[r * M + m] + part[(R + r) * M + m] + part[(2 * R + r) * M + m] + part[(3 * R + r) * M + m];
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t n = n0 + r;
            if (n < N) {
                const float b = bias ? bf_to_f(pf_b[r]) : 0.f;
#pragma unroll
                for (int m = 0; m < M; ++m) {
                    float o = acc[r][m] + b;
                    if (res) o += bf_to_f(pf_r[r][m]);
                    y[(int64_t)m * N + n] = f_to_bf(out_act(o, act));
                }
            }
        }
    }
}

// STAGE: wave m of the workgroup normalises batch row m (and m + 4 when M > 4) ONCE into LDS and every wave's trips read it from there.
// Two things were wrong with every wave rebuilding the normalised slices itself: the sum of squares was a loop of one 16-byte
// load + s_waitcnt vmcnt(0) per 64-vector slice -- eight dependent L2 round trips per row, queued BEHIND the weight prefetch
// (vmcnt retires in order), ~6 us of every wave's life at M = 1 -- and at M >= 2 the per-trip re-normalisation made the
// launches VALU-bound (fused Hyena step 22 / 26 / 43 us at M = 1 / 2 / 4 against 20-22 us for the plain GEMV of the matrix).
// Here the staging wave requests its row's 2 x 8 vectors at once, AHEAD of its weight prefetch, reduces in rmsnorm_kernel's
// order (lane-strided sequential fp32, wave butterfly) and stores the normalised row: bit-identical values, one L2 round trip.
#define GV_WG_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")   // orders LDS only: weight loads stay in flight
extern __shared__ uint4 gv_xn[];                                                          // [M][nvec] normalised rows (STAGE)

__device__ __forceinline__ uint4 gv_norm8(const uint4& xv, const uint4& sv, float inv) {
    uint4 o;
    o.x = pack_bf2(bf_lo(sv.x) * (bf_lo(xv.x) * inv), bf_hi(sv.x) * (bf_hi(xv.x) * inv));
    o.y = pack_bf2(bf_lo(sv.y) * (bf_lo(xv.y) * inv), bf_hi(sv.y) * (bf_hi(xv.y) * inv));
    o.z = pack_bf2(bf_lo(sv.z) * (bf_lo(xv.z) * inv), bf_hi(sv.z) * (bf_hi(xv.z) * inv));
    o.w = pack_bf2(bf_lo(sv.w) * (bf_lo(xv.w) * inv), bf_hi(sv.w) * (bf_hi(xv.w) * inv));
    return o;
}
__device__ __forceinline__ float gv_sumsq8(const uint4& xv, float ss) {
    const float f[8] = {bf_lo(xv.x), bf_hi(xv.x), bf_lo(xv.y), bf_hi(xv.y), bf_lo(xv.z), bf_hi(xv.z), bf_lo(xv.w), bf_hi(xv.w)};
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
    return ss;
}
// rows of up to 512 vectors (the host stages K = 4096 only; other widths take the unstaged kernels): request everything (slices
// past the row end re-read the lane's first vector, unused)
__device__ __forceinline__ void gv_stage_load(const uint4* xr, const uint4* scale, int nvec, int lane, uint4 (&sx)[8], uint4 (&sc)[8]) {
    const int v0 = lane < nvec ? lane : 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int v = lane + 64 * i, vc = v < nvec ? v : v0;
        sx[i] = xr[vc];
        sc[i] = scale[vc];
    }
}
__device__ __forceinline__ void gv_stage_finish(uint4* dst, int nvec, int lane, float eps, float inv_sqrt_d, const uint4 (&sx)[8],
                                                const uint4 (&sc)[8]) {
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (lane + 64 * i < nvec) ss = gv_sumsq8(sx[i], ss);
    ss = wave_sum(ss);
    const float inv = 1.0f / (sqrtf(ss) * inv_sqrt_d + eps);
    uint4 px[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {                            // (opaque copy: otherwise the 64 unpacked fp32 values of the reduction are
        px[i] = sx[i];                                       //  kept alive across it for the normalisation, +64 VGPRs on every wave)
        asm volatile("" : "+v"(px[i].x), "+v"(px[i].y), "+v"(px[i].z), "+v"(px[i].w));
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
        if (lane + 64 * i < nvec) dst[lane + 64 * i] = gv_norm8(px[i], sc[i], inv);
}
// K = 4096 (nvec = 512: every decode layer behind a norm) written out as four trips with a two-deep register pipeline: the
// generic loop below ends each trip by copying the next trip's registers over the current ones, which makes the compiler wait
// for the loads it has just issued -- one trip in flight per wave.  Same operations in the same order.
#define GV_TRIP_LOAD(BUF, T)                                                                                          \
    _Pragma("unroll") for (int r = 0; r < GV_R; ++r) {                                                                \
        BUF[r] = ld_stream(wrow[r] + lane + 128 * (T));                                                               \
        BUF[GV_R + r] = ld_stream(wrow[r] + lane + 128 * (T) + 64);                                                   \
    }
#define GV_TRIP_DOT(BUF, T, XF)                                                                                       \
    _Pragma("unroll") for (int m = 0; m < M; ++m) {                                                                   \
        const uint4 x0 = XF(m, lane + 128 * (T)), x1 = XF(m, lane + 128 * (T) + 64);                                  \
        _Pragma("unroll") for (int r = 0; r < GV_R; ++r) acc[r][m] = dot8(BUF[GV_R + r], x1, dot8(BUF[r], x0, acc[r][m])); \
    }
#define GV_FOUR_TRIPS(XF)                                                                                             \
    {                                                                                                                 \
        uint4 wb[2 * GV_R];                                                                                           \
        GV_TRIP_LOAD(wb, 1)                                                                                           \
        GV_TRIP_DOT(wa, 0, XF)                                                                                        \
        __builtin_amdgcn_sched_barrier(0); /* (trips stay in program order: requests retire in issue order) */        \
        GV_TRIP_LOAD(wa, 2)                                                                                           \
        GV_TRIP_DOT(wb, 1, XF)                                                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                                            \
        GV_TRIP_LOAD(wb, 3)                                                                                           \
        GV_TRIP_DOT(wa, 2, XF)                                                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                                            \
        GV_TRIP_DOT(wb, 3, XF)                                                                                        \
    }

// ---- RMSNorm folded into the layer that consumes it (decode form): y = bf16(scale * x / (rms(x) + eps)) . W^T + bias.
// Every wave first reduces sum(x^2) with the rmsnorm kernel's own lane -> element mapping and summation order (so the
// normalised row is bit-identical to what that kernel would have stored), then streams its R rows of W while it
// rebuilds the normalised x slice by slice in registers -- one launch instead of two per block.  That is the STAGE = false
// form (any K); at K = 4096 the launches take STAGE = true (above): rows normalised once into LDS, four pipelined trips.
template <int M, int R, bool STAGE>
__global__ __launch_bounds__(256) void gemv_norm_kernel(const uint4* __restrict__ x, const uint4* __restrict__ scale,
                                                        const uint4* __restrict__ w, const uint16_t* __restrict__ bias,
                                                        uint16_t* __restrict__ y, int N, int nvec, float eps, float inv_sqrt_d) {
    constexpr int GV_R = R;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * R;
    if (!STAGE && n0 >= N) return;                           // (STAGE: every wave helps to stage x, then leaves)
    const uint4* wrow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        int64_t n = n0 + r < N ? n0 + r : N - 1;
        wrow[r] = w + n * nvec;
    }
    // (STAGE) the staging wave's x / scale requests go out first, so they come back first
    uint4 st_x[8], st_s[8];
    const bool stager = STAGE && wave < M;                   // (M > 4: waves 0-3 take rows 4-7 in a second round)
    if (stager) gv_stage_load(x + (int64_t)wave * nvec, scale, nvec, lane, st_x, st_s);
    __builtin_amdgcn_sched_barrier(0);                       // (requests retire in issue order: keep these ahead of the weights)
    // the first trip's weights are requested BEFORE the norm pass (which only touches x, in L2): the HBM stream starts at
    // once instead of after a ~1.5 us reduction, and every later trip's loads are issued ahead of the trip that consumes
    // the previous ones (same arithmetic in the same order: results are bit-identical to the single-buffered loop)
    uint4 wa[2 * GV_R];
    const bool gv_any = lane + 64 < nvec;
    if (gv_any) {
#pragma unroll
        for (int r = 0; r < GV_R; ++r) { wa[r] = ld_stream(wrow[r] + lane); wa[GV_R + r] = ld_stream(wrow[r] + lane + 64); }
    }
    float inv[M];
#pragma unroll
    for (int m = 0; m < M; ++m) inv[m] = 0.f;
    if (!STAGE) {                                            // rows too long for LDS: every wave reduces every row itself
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float ss = 0.f;
            for (int v = lane; v < nvec; v += 64) ss = gv_sumsq8(x[(int64_t)m * nvec + v], ss);
            ss = wave_sum(ss);
            inv[m] = 1.0f / (sqrtf(ss) * inv_sqrt_d + eps);
        }
    }
    auto normed_calc = [&](int m, int v) {
        const uint4 xv = x[(int64_t)m * nvec + v], sv = scale[v];
        uint4 o;
        o.x = pack_bf2(bf_lo(sv.x) * (bf_lo(xv.x) * inv[m]), bf_hi(sv.x) * (bf_hi(xv.x) * inv[m]));
        o.y = pack_bf2(bf_lo(sv.y) * (bf_lo(xv.y) * inv[m]), bf_hi(sv.y) * (bf_hi(xv.y) * inv[m]));
        o.z = pack_bf2(bf_lo(sv.z) * (bf_lo(xv.z) * inv[m]), bf_hi(sv.z) * (bf_hi(xv.z) * inv[m]));
        o.w = pack_bf2(bf_lo(sv.w) * (bf_lo(xv.w) * inv[m]), bf_hi(sv.w) * (bf_hi(xv.w) * inv[m]));
        return o;
    };
    if (STAGE) {
        if (stager) gv_stage_finish(gv_xn + wave * nvec, nvec, lane, eps, inv_sqrt_d, st_x, st_s);
        if (M > 4) {                                         // batch rows 4-7: a second round for the same waves
            for (int r = wave + 4; r < M; r += 4) {
                gv_stage_load(x + (int64_t)r * nvec, scale, nvec, lane, st_x, st_s);
                gv_stage_finish(gv_xn + r * nvec, nvec, lane, eps, inv_sqrt_d, st_x, st_s);
            }
        }
        GV_WG_BARRIER();
        if (n0 >= N) return;
        __builtin_amdgcn_sched_barrier(0);                   // (the second trip's requests stay below the staging: its registers are free now)
    }
    auto normed = [&](int m, int v) { return STAGE ? gv_xn[m * nvec + v] : normed_calc(m, v); };
    float acc[R][M];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
    if constexpr (STAGE) {                                   // (STAGE launches have nvec == 512: the host checks)
        GV_FOUR_TRIPS(normed)
    } else {
        int v = lane;
        for (; v + 64 < nvec; v += 128) {
            uint4 wb[2 * GV_R];
            const bool more = v + 128 + 64 < nvec;
            if (more) {
#pragma unroll
                for (int r = 0; r < GV_R; ++r) { wb[r] = ld_stream(wrow[r] + v + 128); wb[GV_R + r] = ld_stream(wrow[r] + v + 192); }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 x0 = normed(m, v), x1 = normed(m, v + 64);
#pragma unroll
                for (int r = 0; r < GV_R; ++r) acc[r][m] = dot8(wa[GV_R + r], x1, dot8(wa[r], x0, acc[r][m]));
            }
            if (more) {
#pragma unroll
                for (int r = 0; r < 2 * GV_R; ++r) wa[r] = wb[r];
            }
        }
        for (; v < nvec; v += 64) {
            uint4 w0[R];
#pragma unroll
            for (int r = 0; r < R; ++r) w0[r] = ld_stream(wrow[r] + v);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 x0 = normed(m, v);
#pragma unroll
                for (int r = 0; r < R; ++r) acc[r][m] = dot8(w0[r], x0, acc[r][m]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = wave_sum(acc[r][m]);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int64_t n = n0 + r;
            if (n < N) {
                const float b = bias ? bf_to_f(bias[n]) : 0.f;
#pragma unroll
                for (int m = 0; m < M; ++m) y[(int64_t)m * N + n] = f_to_bf(acc[r][m] + b);
            }
        }
    }
}

// ---- the whole Hyena mixer input of a decode step in one launch: pre-norm + projection + FIR/modal step + gate.
// A wave owns CPW (one or two) adjacent channels of one head = 3 CPW rows of the projection weight (x2, x1, v thirds), streams
// them like gemv_norm_kernel, and then its first CPW * M lanes (one per channel x batch row) run evo_hyena_step's arithmetic
// on the dot products -- same operations in the same order, so outputs and carried states are bit-identical to
// evo_norm_linear_small_m_bf16 followed by evo_hyena_step.
template <int M, int CPW, bool STAGE>
__global__ __launch_bounds__(256) void gemv_norm_hyena_kernel(
    const uint4* __restrict__ x, const uint4* __restrict__ scale, const uint4* __restrict__ w,
    const uint16_t* __restrict__ bias, uint16_t* __restrict__ fir_state, float* __restrict__ iir_state,
    const uint16_t* __restrict__ fir_w, const uint16_t* __restrict__ fir_b, const float* __restrict__ poles,
    const float* __restrict__ residues, const uint16_t* __restrict__ dskip, uint16_t* __restrict__ y, int D, int nvec,
    float eps, float inv_sqrt_d) {
    constexpr int HDc = 128, NSc = 8, GV_R = 3 * CPW;      // CPW channels per wave (1 or 2)
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int unit = blockIdx.x * 4 + wave;                     // channel (pair) index over D / CPW
    if (!STAGE && unit >= D / CPW) return;
    const int unit_c = unit < D / CPW ? unit : D / CPW - 1;      // (STAGE: a wave past the end stages x with the others, then leaves)
    const int h = unit_c / (HDc / CPW), j0 = CPW * (unit_c - h * (HDc / CPW));
    const uint4* wrow[GV_R];
#pragma unroll
    for (int r = 0; r < GV_R; ++r) wrow[r] = w + (int64_t)(h * 3 * HDc + (r / CPW) * HDc + j0 + (r % CPW)) * nvec;
    // (STAGE) the staging wave's x / scale requests go out first, so they come back first
    uint4 st_x[8], st_s[8];
    const bool stager = STAGE && wave < M;                   // (M > 4: waves 0-3 take rows 4-7 in a second round)
    if (stager) gv_stage_load(x + (int64_t)wave * nvec, scale, nvec, lane, st_x, st_s);
    __builtin_amdgcn_sched_barrier(0);                       // (requests retire in issue order: keep these ahead of the weights)
    // the first trip's weights are requested BEFORE the norm pass (which only touches x, in L2): the HBM stream starts at
    // once instead of after a ~1.5 us reduction, and every later trip's loads are issued ahead of the trip that consumes
    // the previous ones (same arithmetic in the same order: results are bit-identical to the single-buffered loop)
    uint4 wa[2 * GV_R];
    const bool gv_any = lane + 64 < nvec;
    if (gv_any) {
#pragma unroll
        for (int r = 0; r < GV_R; ++r) { wa[r] = ld_stream(wrow[r] + lane); wa[GV_R + r] = ld_stream(wrow[r] + lane + 64); }
    }
    float inv[M];
#pragma unroll
    for (int m = 0; m < M; ++m) inv[m] = 0.f;
    if (!STAGE) {                                            // rows too long for LDS: every wave reduces every row itself
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float ss = 0.f;
            for (int v = lane; v < nvec; v += 64) ss = gv_sumsq8(x[(int64_t)m * nvec + v], ss);
            ss = wave_sum(ss);
            inv[m] = 1.0f / (sqrtf(ss) * inv_sqrt_d + eps);
        }
    }
    auto normed_calc = [&](int m, int v) {
        const uint4 xv = x[(int64_t)m * nvec + v], sv = scale[v];
        uint4 o;
        o.x = pack_bf2(bf_lo(sv.x) * (bf_lo(xv.x) * inv[m]), bf_hi(sv.x) * (bf_hi(xv.x) * inv[m]));
        o.y = pack_bf2(bf_lo(sv.y) * (bf_lo(xv.y) * inv[m]), bf_hi(sv.y) * (bf_hi(xv.y) * inv[m]));
        o.z = pack_bf2(bf_lo(sv.z) * (bf_lo(xv.z) * inv[m]), bf_hi(sv.z) * (bf_hi(xv.z) * inv[m]));
        o.w = pack_bf2(bf_lo(sv.w) * (bf_lo(xv.w) * inv[m]), bf_hi(sv.w) * (bf_hi(xv.w) * inv[m]));
        return o;
    };
    if (STAGE) {
        if (stager) gv_stage_finish(gv_xn + wave * nvec, nvec, lane, eps, inv_sqrt_d, st_x, st_s);
        if (M > 4) {                                         // batch rows 4-7: a second round for the same waves
            for (int r = wave + 4; r < M; r += 4) {
                gv_stage_load(x + (int64_t)r * nvec, scale, nvec, lane, st_x, st_s);
                gv_stage_finish(gv_xn + r * nvec, nvec, lane, eps, inv_sqrt_d, st_x, st_s);
            }
        }
        GV_WG_BARRIER();
        if (unit >= D / CPW) return;
        __builtin_amdgcn_sched_barrier(0);                   // (the second trip's requests stay below the staging: its registers are free now)
    }
    // the epilogue's operands (this lane's channel x batch row: FIR taps / state / bias of x2, x1, v, the 8 poles, residues and
    // modal states, D) are requested NOW (after the staging, whose registers they reuse), behind the first weight trip: they do not depend on the dot products, and fetched
    // at the end they were a ~2 us dependent-latency tail per wave with nothing left to overlap it
    const bool ep_lane = lane < CPW * M;
    const int ep_e = lane % CPW, ep_m = ep_lane ? lane / CPW : 0;
    const int ep_dch = h * HDc + j0 + ep_e;
    uint16_t pf_bias[3], pf_fw[3][3], pf_fb[3], pf_fs[3][2], pf_dk = 0;
    float2 pf_p[NSc], pf_r[NSc], pf_s[NSc];
    if (ep_lane) {
#pragma unroll
        for (int g = 0; g < 3; ++g) {
            const int c = h * 3 * HDc + g * HDc + j0 + ep_e;
            pf_bias[g] = bias[c];
            pf_fw[g][0] = fir_w[c * 3]; pf_fw[g][1] = fir_w[c * 3 + 1]; pf_fw[g][2] = fir_w[c * 3 + 2];
            pf_fb[g] = fir_b[c];
            const uint16_t* fs = fir_state + ((int64_t)ep_m * 3 * D + c) * 2;
            pf_fs[g][0] = fs[0]; pf_fs[g][1] = fs[1];
        }
        const float2* st = (const float2*)iir_state + ((int64_t)ep_m * D + ep_dch) * NSc;
        const float2* pp = (const float2*)poles + (int64_t)ep_dch * NSc;
        const float2* rp = (const float2*)residues + (int64_t)ep_dch * NSc;
#pragma unroll
        for (int sI = 0; sI < NSc; ++sI) { pf_p[sI] = pp[sI]; pf_r[sI] = rp[sI]; pf_s[sI] = st[sI]; }
        pf_dk = dskip[ep_dch];
    }
    auto normed = [&](int m, int v) { return STAGE ? gv_xn[m * nvec + v] : normed_calc(m, v); };
    float acc[GV_R][M];
#pragma unroll
    for (int r = 0; r < GV_R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
    if constexpr (STAGE) {                                   // (STAGE launches have nvec == 512: the host checks)
        GV_FOUR_TRIPS(normed)
    } else {
        int v = lane;
        for (; v + 64 < nvec; v += 128) {
            uint4 wb[2 * GV_R];
            const bool more = v + 128 + 64 < nvec;
            if (more) {
#pragma unroll
                for (int r = 0; r < GV_R; ++r) { wb[r] = ld_stream(wrow[r] + v + 128); wb[GV_R + r] = ld_stream(wrow[r] + v + 192); }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 x0 = normed(m, v), x1 = normed(m, v + 64);
#pragma unroll
                for (int r = 0; r < GV_R; ++r) acc[r][m] = dot8(wa[GV_R + r], x1, dot8(wa[r], x0, acc[r][m]));
            }
            if (more) {
#pragma unroll
                for (int r = 0; r < 2 * GV_R; ++r) wa[r] = wb[r];
            }
        }
        for (; v < nvec; v += 64) {
            uint4 w0[GV_R];
#pragma unroll
            for (int r = 0; r < GV_R; ++r) w0[r] = ld_stream(wrow[r] + v);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 x0 = normed(m, v);
#pragma unroll
                for (int r = 0; r < GV_R; ++r) acc[r][m] = dot8(w0[r], x0, acc[r][m]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < GV_R; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = wave_sum(acc[r][m]);
    if (!ep_lane) return;
    const int e = ep_e, m = ep_m;                                // this lane: channel j0 + e of batch row m
    float f[3];
#pragma unroll
    for (int g = 0; g < 3; ++g) {
        float d = 0.f;
#pragma unroll
        for (int mm = 0; mm < M; ++mm)
#pragma unroll
            for (int ee = 0; ee < CPW; ++ee) d = (m == mm && e == ee) ? acc[CPW * g + ee][mm] : d;
        const int c = h * 3 * HDc + g * HDc + j0 + e;            // channel in the 3D row
        const uint16_t zraw = f_to_bf(d + bf_to_f(pf_bias[g]));  // what the unfused projection stores
        uint16_t* fs = fir_state + ((int64_t)m * 3 * D + c) * 2;
        const float o0 = bf_to_f(pf_fs[g][0]), o1 = bf_to_f(pf_fs[g][1]);
        f[g] = fmaf(bf_to_f(pf_fw[g][2]), bf_to_f(zraw),
                    fmaf(bf_to_f(pf_fw[g][1]), o1, fmaf(bf_to_f(pf_fw[g][0]), o0, bf_to_f(pf_fb[g]))));
        fs[0] = pf_fs[g][1];
        fs[1] = zraw;
    }
    const int dch = ep_dch;
    const float xv = f[1] * f[2];
    float2* st = (float2*)iir_state + ((int64_t)m * D + dch) * NSc;
    float accy = 0.f;
#pragma unroll
    for (int s = 0; s < NSc; ++s) {
        const float2 p = pf_p[s], r = pf_r[s], sv = pf_s[s];
        const float nr = fmaf(p.x, sv.x, fmaf(-p.y, sv.y, xv));
        const float ni = fmaf(p.x, sv.y, p.y * sv.x);
        st[s] = make_float2(nr, ni);
        accy = fmaf(r.x, nr, fmaf(-r.y, ni, accy));
    }
    y[(int64_t)m * D + dch] = f_to_bf(fmaf(xv, bf_to_f(pf_dk), accy) * f[0]);
}

// ---- gated MLP input, decode form: a[m][n] = gelu(x_m . W1_n) * (x_m . W2_n) with W12 = [W1; W2] ([2I, K]).  Same
// streaming loop as gemv_kernel; a wave owns 2 output columns = rows (n, n+1) of W1 and (I+n, I+n+1) of W2, rounds both
// dot products to bf16 (what the unfused GEMM stores) and applies the gate -- one launch instead of two per block.
// NORM: x is the un-normalised residual row and `scale` the RMSNorm weight (same fold as gemv_norm_kernel).
template <int M, bool NORM, bool STAGE>
__global__ __launch_bounds__(256) void gemv_gate_kernel(const uint4* __restrict__ x, const uint4* __restrict__ scale,
                                                        const uint4* __restrict__ w, uint16_t* __restrict__ a, int I,
                                                        int nvec, float eps, float inv_sqrt_d, int grouped, int act) {
    constexpr int GV_R = 4;                                  // rows per wave: (n, n+1) of W1 and of W2
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * 2;
    if (!STAGE && n0 >= I) return;
    const uint4* wrow[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        int64_t n = n0 + (r & 1) < I ? n0 + (r & 1) : I - 1;
        // plain [W1; W2]: row (r >> 1) I + n.  grouped (HipOps.pack_gate_weights: blocks of [32 rows of W1 | the same 32 rows of W2], the
        // order the gated MFMA launch reads -- ONE copy of l1 | l2 serves prefill and decode): row 64 (n / 32) + 32 (r >> 1) + n % 32
        const int64_t row = grouped ? 64 * (n >> 5) + 32 * (r >> 1) + (n & 31) : (r >> 1) * (int64_t)I + n;
        wrow[r] = w + row * nvec;
    }
    // (STAGE) the staging wave's x / scale requests go out first, so they come back first
    uint4 st_x[8], st_s[8];
    const bool stager = STAGE && wave < M;                   // (M > 4: waves 0-3 take rows 4-7 in a second round)
    if (stager) gv_stage_load(x + (int64_t)wave * nvec, scale, nvec, lane, st_x, st_s);
    __builtin_amdgcn_sched_barrier(0);                       // (requests retire in issue order: keep these ahead of the weights)
    // first trip's weights before the norm pass, every later trip one ahead (see gemv_norm_kernel)
    uint4 wa[8];
    if (lane + 64 < nvec) {
#pragma unroll
        for (int r = 0; r < 4; ++r) { wa[r] = ld_stream(wrow[r] + lane); wa[4 + r] = ld_stream(wrow[r] + lane + 64); }
    }
    float inv[M];
#pragma unroll
    for (int m = 0; m < M; ++m) inv[m] = 0.f;
    if (NORM && !STAGE) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            float ss = 0.f;
            for (int v = lane; v < nvec; v += 64) ss = gv_sumsq8(x[(int64_t)m * nvec + v], ss);
            ss = wave_sum(ss);
            inv[m] = 1.0f / (sqrtf(ss) * inv_sqrt_d + eps);
        }
    }
    auto xin_calc = [&](int m, int v) {
        const uint4 xv = x[(int64_t)m * nvec + v];
        if (!NORM) return xv;
        const uint4 sv = scale[v];
        uint4 o;
        o.x = pack_bf2(bf_lo(sv.x) * (bf_lo(xv.x) * inv[m]), bf_hi(sv.x) * (bf_hi(xv.x) * inv[m]));
        o.y = pack_bf2(bf_lo(sv.y) * (bf_lo(xv.y) * inv[m]), bf_hi(sv.y) * (bf_hi(xv.y) * inv[m]));
        o.z = pack_bf2(bf_lo(sv.z) * (bf_lo(xv.z) * inv[m]), bf_hi(sv.z) * (bf_hi(xv.z) * inv[m]));
        o.w = pack_bf2(bf_lo(sv.w) * (bf_lo(xv.w) * inv[m]), bf_hi(sv.w) * (bf_hi(xv.w) * inv[m]));
        return o;
    };
    if (STAGE) {
        if (stager) gv_stage_finish(gv_xn + wave * nvec, nvec, lane, eps, inv_sqrt_d, st_x, st_s);
        if (M > 4) {                                         // batch rows 4-7: a second round for the same waves
            for (int r = wave + 4; r < M; r += 4) {
                gv_stage_load(x + (int64_t)r * nvec, scale, nvec, lane, st_x, st_s);
                gv_stage_finish(gv_xn + r * nvec, nvec, lane, eps, inv_sqrt_d, st_x, st_s);
            }
        }
        GV_WG_BARRIER();
        if (n0 >= I) return;
        __builtin_amdgcn_sched_barrier(0);                   // (the second trip's requests stay below the staging: its registers are free now)
    }
    auto xin = [&](int m, int v) { return STAGE ? gv_xn[m * nvec + v] : xin_calc(m, v); };
    float acc[4][M];
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
    if constexpr (STAGE) {                                   // (STAGE launches have nvec == 512: the host checks)
        GV_FOUR_TRIPS(xin)
    } else {
        int v = lane;
        for (; v + 64 < nvec; v += 128) {
            uint4 wb[8];
            const bool more = v + 128 + 64 < nvec;
            if (more) {
#pragma unroll
                for (int r = 0; r < 4; ++r) { wb[r] = ld_stream(wrow[r] + v + 128); wb[4 + r] = ld_stream(wrow[r] + v + 192); }
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 x0 = xin(m, v), x1 = xin(m, v + 64);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r][m] = dot8(wa[4 + r], x1, dot8(wa[r], x0, acc[r][m]));
            }
            if (more) {
#pragma unroll
                for (int r = 0; r < 8; ++r) wa[r] = wb[r];
            }
        }
        for (; v < nvec; v += 64) {
            uint4 w0[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) w0[r] = ld_stream(wrow[r] + v);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const uint4 x0 = xin(m, v);
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r][m] = dot8(w0[r], x0, acc[r][m]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int m = 0; m < M; ++m) acc[r][m] = wave_sum(acc[r][m]);
    if (lane == 0) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const f32x2_t u = {round_bf(acc[0][m]), round_bf(acc[1][m])}, g = {round_bf(acc[2][m]), round_bf(acc[3][m])};
            const f32x2_t o = act_gate2(u, g, act);
            if (n0 + 1 < I) *(uint32_t*)(a + (int64_t)m * I + n0) = pack_bf2(o[0], o[1]);
            else a[(int64_t)m * I + n0] = f_to_bf(o[0]);
        }
    }
}

// ---- a sublayer's closing norm folded into the next one's first layer (decode form of models with an fp32 residual stream):
//   x' = x + y / sqrt(mean(y^2) + eps) * (off + g)       (rows of the stream; workgroup 0 also stores them)
//   SUM: x' = t / sqrt(mean(t^2) + eps) * (off + g), t = alpha x + y
//   plain: z = bf16(x') . W^T (act 3: through the square of relu)         gated: a = act(bf16(x') . W1^T) * (bf16(x') . W2^T), w = [W1; W2] or its grouped order
// Every workgroup rebuilds the row -- 8 bytes per element from L2 -- into LDS while its first weight requests are under way.  One row: with more the norm's own launch is
// ahead (what both take: MixerOps.fuse_postnorm_ok).
template <bool GATE, bool SUM>
__global__ __launch_bounds__(256) void postnorm_gemv_kernel(const uint4* __restrict__ y, const uint4* __restrict__ g, const float4* __restrict__ x,
                                                            float4* __restrict__ x_out, const uint4* __restrict__ w, uint16_t* __restrict__ out, int N,
                                                            int nvec, float alpha, float eps, float off, int grouped, int act) {
    extern __shared__ uint4 pn_x[];                              // [nvec]
    __shared__ float red[4];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * (GATE ? 2 : 4);     // first output column of this wave
    const int I = N;                                             // (GATE: N gated columns, 2 N weight rows)
    const uint4* wrow[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (GATE) {
            const int64_t n = n0 + (r & 1) < I ? n0 + (r & 1) : I - 1;
            wrow[r] = w + (grouped ? 64 * (n >> 5) + 32 * (r >> 1) + (n & 31) : (r >> 1) * (int64_t)I + n) * nvec;
        } else wrow[r] = w + (n0 + r < N ? n0 + r : N - 1) * nvec;
    }
    uint4 wa[8];
#pragma unroll
    for (int r = 0; r < 4; ++r) {                                // (rows shorter than two requests repeat their last vector: not used)
        wa[r] = ld_stream(wrow[r] + (lane < nvec ? lane : nvec - 1));
        wa[4 + r] = ld_stream(wrow[r] + (lane + 64 < nvec ? lane + 64 : nvec - 1));
    }
    float ss = 0.f;
    for (int v = tid; v < nvec; v += 256) {
        const uint4 yv = y[v];
        if (SUM) {
            const float4 a = x[v * 2], b = x[v * 2 + 1];
            const float t[8] = {fmaf(alpha, a.x, bf_lo(yv.x)), fmaf(alpha, a.y, bf_hi(yv.x)), fmaf(alpha, a.z, bf_lo(yv.y)), fmaf(alpha, a.w, bf_hi(yv.y)),
                                fmaf(alpha, b.x, bf_lo(yv.z)), fmaf(alpha, b.y, bf_hi(yv.z)), fmaf(alpha, b.z, bf_lo(yv.w)), fmaf(alpha, b.w, bf_hi(yv.w))};
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(t[e], t[e], ss);
        } else ss = gv_sumsq8(yv, ss);
    }
    ss = wave_sum(ss);
    if (lane == 0) red[wave] = ss;
    __syncthreads();
    const float inv = 1.0f / sqrtf((red[0] + red[1] + red[2] + red[3]) / (float)(nvec * 8) + eps);
    for (int v = tid; v < nvec; v += 256) {
        const uint4 yv = y[v], gv = g[v];
        float4 a = x[v * 2], b = x[v * 2 + 1];
        if (SUM) {
            a.x = fmaf(alpha, a.x, bf_lo(yv.x)) * inv * (off + bf_lo(gv.x)); a.y = fmaf(alpha, a.y, bf_hi(yv.x)) * inv * (off + bf_hi(gv.x));
            a.z = fmaf(alpha, a.z, bf_lo(yv.y)) * inv * (off + bf_lo(gv.y)); a.w = fmaf(alpha, a.w, bf_hi(yv.y)) * inv * (off + bf_hi(gv.y));
            b.x = fmaf(alpha, b.x, bf_lo(yv.z)) * inv * (off + bf_lo(gv.z)); b.y = fmaf(alpha, b.y, bf_hi(yv.z)) * inv * (off + bf_hi(gv.z));
            b.z = fmaf(alpha, b.z, bf_lo(yv.w)) * inv * (off + bf_lo(gv.w)); b.w = fmaf(alpha, b.w, bf_hi(yv.w)) * inv * (off + bf_hi(gv.w));
        } else {
            a.x += bf_lo(yv.x) * inv * (off + bf_lo(gv.x)); a.y += bf_hi(yv.x) * inv * (off + bf_hi(gv.x));
            a.z += bf_lo(yv.y) * inv * (off + bf_lo(gv.y)); a.w += bf_hi(yv.y) * inv * (off + bf_hi(gv.y));
            b.x += bf_lo(yv.z) * inv * (off + bf_lo(gv.z)); b.y += bf_hi(yv.z) * inv * (off + bf_hi(gv.z));
            b.z += bf_lo(yv.w) * inv * (off + bf_lo(gv.w)); b.w += bf_hi(yv.w) * inv * (off + bf_hi(gv.w));
        }
        pn_x[v] = make_uint4(pack_bf2(a.x, a.y), pack_bf2(a.z, a.w), pack_bf2(b.x, b.y), pack_bf2(b.z, b.w));
        if (blockIdx.x == 0) {
            x_out[v * 2] = a;
            x_out[v * 2 + 1] = b;
        }
    }
    __syncthreads();
    if (n0 >= N) return;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    int v = lane;
    for (; v + 64 < nvec; v += 128) {
        uint4 wb[8];
        const bool more = v + 128 < nvec;
        if (more) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                wb[r] = ld_stream(wrow[r] + v + 128);
                wb[4 + r] = ld_stream(wrow[r] + (v + 192 < nvec ? v + 192 : nvec - 1));
            }
        }
        const uint4 x0 = pn_x[v], x1 = pn_x[v + 64];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = dot8(wa[4 + r], x1, dot8(wa[r], x0, acc[r]));
        if (more) {
#pragma unroll
            for (int r = 0; r < 8; ++r) wa[r] = wb[r];
        }
    }
    if (v < nvec) {                                              // one vector left for this lane: its request is in wa already
        const uint4 x0 = pn_x[v];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = dot8(wa[r], x0, acc[r]);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = wave_sum(acc[r]);
    if (lane == 0) {
        if (GATE) {
            const f32x2_t u = {round_bf(acc[0]), round_bf(acc[1])}, z = {round_bf(acc[2]), round_bf(acc[3])};
            const f32x2_t o = act_gate2(u, z, act);
            out[n0] = f_to_bf(o[0]);
            if (n0 + 1 < N) out[n0 + 1] = f_to_bf(o[1]);
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (n0 + r < N) {
                    const float z = act ? fmaxf(acc[r], 0.f) : acc[r];
                    out[n0 + r] = f_to_bf(act ? z * z : z);
                }
        }
    }
}

static int postnorm_gemv_launch(const void* y, const void* g, const float* x, float* x_out, const void* w, void* out, int64_t M, int64_t N, int64_t K,
                                float alpha, bool sum, float eps, float off, bool gate, int64_t grouped, int64_t act, void* stream) {
    if (M < 1 || M > 4 || N <= 0 || N > 0x3fffffff || K <= 0 || K % 8 != 0 || K > 8192 || !y || !g || !x || !x_out || !w || !out || x == x_out) return -1;
    if (gate ? ((act != 0 && act != 1) || (grouped && N % 32 != 0)) : (act != 0 && act != 3)) return -1;
    const dim3 grid((unsigned)((N + (gate ? 7 : 15)) / (gate ? 8 : 16))), block(256);
    const size_t lds = (size_t)K * 2;                            // (<= 16 KB)
#define EVO_PN(G, S) hipLaunchKernelGGL((postnorm_gemv_kernel<G, S>), grid, block, lds, (hipStream_t)stream, (const uint4*)y + m * (K / 8), (const uint4*)g,    \
                                        (const float4*)x + m * (K / 4), (float4*)x_out + m * (K / 4), (const uint4*)w, (uint16_t*)out + m * N, (int)N, (int)(K / 8), \
                                        alpha, eps, off, grouped ? 1 : 0, (int)act)
    for (int64_t m = 0; m < M; ++m) {
        if (gate) { if (sum) EVO_PN(true, true); else EVO_PN(true, false); }
        else { if (sum) EVO_PN(false, true); else EVO_PN(false, false); }
    }
#undef EVO_PN
    return evo_launch_status();
}

extern "C" int evo_postnorm_linear_small_m_bf16(const void* y, const void* g, const float* x, float* x_out, const void* w, void* z, int64_t M, int64_t N,
                                                int64_t K, float alpha, int64_t sum, float eps, float w_offset, int64_t act, void* stream) {
    return postnorm_gemv_launch(y, g, x, x_out, w, z, M, N, K, alpha, sum != 0, eps, w_offset, false, 0, act, stream);
}

extern "C" int evo_postnorm_mlp_gate_small_m_bf16(const void* y, const void* g, const float* x, float* x_out, const void* w12, void* a, int64_t M,
                                                  int64_t I, int64_t K, float alpha, int64_t sum, float eps, float w_offset, int64_t grouped,
                                                  int64_t act, void* stream) {
    return postnorm_gemv_launch(y, g, x, x_out, w12, a, M, I, K, alpha, sum != 0, eps, w_offset, true, grouped, act, stream);
}

// ---- 5 <= M <= 16: MFMA form.  Workgroup = 8 waves = 16 output rows; wave w streams its eighth of K:
//   A operand = W rows   (lane: row n = lane & 15, k-block = lane >> 4 -> 16 B = 8 bf16, non-temporal, straight to VGPRs)
//   B operand = x rows   (lane: row m = lane & 15, same k-block; rows >= M re-read row M-1 and are never stored)
//   D[n][m]: lane holds n = 4 (lane >> 4) + r, m = lane & 15.
// The eight partial tiles meet in LDS; wave 0 adds bias / residual and stores (one rounding).
typedef float gv_f32x4 __attribute__((ext_vector_type(4)));
// MT (round 6): m tiles of 16 batch rows per weight pass -- 17 <= M <= 64 rows (the pooled decode step at 17-64 live slots; small prefill
// batches) stream the weights ONCE with MT MFMAs per weight fragment.  Until round 5 those batches ran the persistent 256 x 256 GEMM:
// N / 256 of the 256 CUs busy, 0.5-1.3 TB/s of weights (profiles/r06_pool32_kernel_stats.txt: 80 % of a 32-slot pooled step).
// NT (round 6): n tiles of 16 weight rows per workgroup sharing every x fragment -- at 17-64 batch rows a weight fragment (1 KiB per wave) pulled
// MT x fragments of the same size through L2 / L1 (2.1 TB/s of weights at 32 rows, 1.5 at 64: tools/bench_gemv.py); two n tiles halve that.
template <int MT, int NT>
__global__ __launch_bounds__(512) void skinny_mfma_kernel(const uint4* __restrict__ x, const uint4* __restrict__ w,
                                                          const uint16_t* __restrict__ bias, const uint16_t* res,
                                                          uint16_t* y, int M, int N, int nvec, int act) {   // res may alias y
    static_assert(MT * NT <= 8, "one reducing wave per (n tile, m tile)");
    __shared__ gv_f32x4 part[NT * MT][8][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kb = lane >> 4;
    const int n0 = blockIdx.x * 16 * NT;
    const int nsteps = nvec >> 2;                                // 32 k per MFMA = 4 vectors of 8
    const int s0 = (int)((int64_t)nsteps * wave / 8), s1 = (int)((int64_t)nsteps * (wave + 1) / 8);
    const uint4* wp[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
        const int nrow = n0 + 16 * j + r16 < N ? n0 + 16 * j + r16 : N - 1;
        wp[j] = w + (int64_t)nrow * nvec + kb;
    }
    const uint4* xp[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) {
        const int mrow = 16 * t + r16 < M ? 16 * t + r16 : M - 1;
        xp[t] = x + (int64_t)mrow * nvec + kb;
    }
    gv_f32x4 acc[NT][MT];
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[j][t] = gv_f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int U = NT * MT == 1 ? 8 : (NT + MT <= 4 ? 4 : 2);     // steps per trip: U * (NT weight + MT x) fragments requested together
    int s = s0;
    for (; s + U <= s1; s += U) {
        uint4 wf[NT][U], xf[MT][U];
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int u = 0; u < U; ++u) wf[j][u] = ld_stream(wp[j] + 4 * (s + u));
#pragma unroll
        for (int t = 0; t < MT; ++t)
#pragma unroll
            for (int u = 0; u < U; ++u) xf[t][u] = xp[t][4 * (s + u)];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[j][u]), __builtin_bit_cast(bf16x8_t, xf[t][u]),
                                                                        acc[j][t], 0, 0, 0);
    }
    for (; s < s1; ++s) {
        uint4 xv[MT];
#pragma unroll
        for (int t = 0; t < MT; ++t) xv[t] = xp[t][4 * s];
#pragma unroll
        for (int j = 0; j < NT; ++j) {
            const uint4 wv = ld_stream(wp[j] + 4 * s);
#pragma unroll
            for (int t = 0; t < MT; ++t)
                acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wv), __builtin_bit_cast(bf16x8_t, xv[t]), acc[j][t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int t = 0; t < MT; ++t) part[j * MT + t][wave][lane] = acc[j][t];
    __syncthreads();
    // the eight partial tiles of (n tile j, m tile t) meet in wave j MT + t: bias / residual added in fp32, one rounding
    if (wave < NT * MT) {
        gv_f32x4 a_ = part[wave][0][lane];
#pragma unroll
        for (int q = 1; q < 8; ++q) a_ += part[wave][q][lane];
        const int jt = wave / MT, tt = wave - jt * MT;
        const int m = 16 * tt + r16;
        if (m < M) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int n = n0 + 16 * jt + 4 * kb + r;
                if (n < N) {
                    float o = a_[r] + (bias ? bf_to_f(bias[n]) : 0.f);
                    if (res) o += bf_to_f(res[(int64_t)m * N + n]);
                    y[(int64_t)m * N + n] = f_to_bf(out_act(o, act));
                }
            }
        }
    }
}

// ---- 3 to 32 rows on the narrow layers (N <= 4096: a workgroup per 16 columns is about one per CU): the k-split form with whole row pieces.  A workgroup =
// 16 weight rows; its waves take every WAVES-th chunk of CH k and park weight and batch rows of a chunk in a PRIVATE part of LDS (asynchronous loads of
// 1 KiB = whole row pieces of 2 CH bytes, no registers, no barrier), NB chunks in flight; the WAVES partial tiles meet in LDS at the end.  Granule g of a
// row sits at slot g ^ (row & 15): a fragment read meets no bank twice.
// Bound by the weight stream and, at K = 4,096, by a launch's ramp (us at 8 / 16 / 32 rows, a plain read of the matrix in brackets; all workgroups from K = 0 on ->
// three chunks apart by turns, four waves): 4,096 x 4,096 [6.5] 8.0 / 8.9 / 10.6 -> 7.6 / 8.2 / 9.8; K = 11,008 [14.1] 18.6 / 20.1 / 23.3 -> 16.1 / 17.6 / 21.8;
// K = 16,384 [22.0] 28.5 / 29.9 / 33.3 -> 22.8 / 22.3 / 29.3.
// XR: batch rows loaded (8, 16 or 32; rows behind M read as zero or are a repeated row, and are never stored).
#define KW_WAIT(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")
template <int XR, int WAVES, int CH, int NB, int EP>
__global__ __launch_bounds__(64 * WAVES) void skinny_kw_kernel(const unsigned char* __restrict__ x, const unsigned char* __restrict__ w,
                                                               const uint16_t* __restrict__ bias, const uint16_t* res, uint16_t* y, int M, int N, int K,
                                                               int act, const uint16_t* __restrict__ scale, uint16_t* __restrict__ xg, float* __restrict__ ss) {   // res may alias y
    constexpr int MT = XR > 16 ? 2 : 1, ROW = 2 * CH, RPI = 1024 / ROW, GR = ROW / 16;      // bytes of a row piece, rows per request, granules per row piece
    constexpr int PW = 16 / RPI, PX = XR / RPI, P = PW + PX, BUF = (16 + XR) * ROW;
    extern __shared__ __attribute__((aligned(16))) unsigned char kw_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kb = lane >> 4;
    const int n0 = blockIdx.x * 16;
    const uint32_t rowb = (uint32_t)K * 2;
    const uint64_t wa = (uint64_t)w + (uint64_t)n0 * rowb, xa = (uint64_t)x;
    const uint32_t wn = (uint32_t)(N - n0 < 16 ? N - n0 : 16);
    typedef uint32_t kw_u32x4 __attribute__((ext_vector_type(4)));
    const kw_u32x4 rw = {(uint32_t)wa, (uint32_t)(wa >> 32) & 0xffffu, wn * rowb, 0x00020000u};
    const kw_u32x4 rx = {(uint32_t)xa, (uint32_t)(xa >> 32) & 0xffffu, (uint32_t)M * rowb, 0x00020000u};
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)kw_lds + wave * (NB * BUF);
    uint32_t off[PX > PW ? PX : PW];
#pragma unroll
    for (int i = 0; i < (PX > PW ? PX : PW); ++i) {
        const int r = i * RPI + lane / GR;
        off[i] = (uint32_t)r * rowb + (uint32_t)((lane % GR) ^ (r & 15 & (GR - 1))) * 16u;
    }
    // EP: bias and residual values of the waves that end with results, requested ahead of everything (from places that are there; `EP` 2: four at a time) and looked at behind the
    // last product: asked for there they were a memory latency of their own at the end (4,096 x 4,096 with both, 5 / 16 / 32 rows 8.4 / 9.3 / 11.4 -> 7.5 / 8.1 / 10.0 us, K = 11,008
    // 17.8 / 18.9 -> 16.7 / 17.7; one value a request 7.7 / 8.4 / 10.3, behind the first chunks 8.1 / 9.0 / 10.8).  Without either they are not in the code: 7.25 -> 7.1.
    // EP 3 (N % 16 == 0): for the norm behind the layer, whose scale this is: xg = the new value times scale, and ss [M][N / 16], a row's sum of squares by workgroups.  What takes the
    // norm multiplies xg by its weights and the sums by 1 / (rms + eps) (skinny_ring_kernel, RS).
    uint2 pb = {}, pr = {}, pg = {};
    if (EP && wave < MT) {
        const int m = 16 * wave + r16, nq = n0 + 4 * kb;
        const uint16_t* from = res + (int64_t)(m < M ? m : M - 1) * N;
        auto four = [&](const uint16_t* p) {
            if constexpr (EP >= 2) return *(const uint2*)(p + (nq < N ? nq : 0));
            uint32_t v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = p[nq + r < N ? nq + r : N - 1];
            return make_uint2(v[0] | v[1] << 16, v[2] | v[3] << 16);
        };
        if (bias) pb = four(bias);
        if (res) pr = four(from);
        if constexpr (EP == 3) pg = four(scale);
    }
    const int chunks = K / CH, mine = (chunks - wave + WAVES - 1) / WAVES;
    const int start = mine > 4 && gridDim.x >= 128 ? (int)(blockIdx.x >> 3) * 3 % mine : 0;       // (workgroups of an XCD don't walk K in step: skinny_ring_kernel)
    auto fetch = [&](int i, uint32_t buf) {
        i = start + i >= mine ? start + i - mine : start + i;
        const uint32_t so = (uint32_t)(wave + WAVES * i) * ROW;
#pragma unroll
        for (int j = 0; j < PW; ++j)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(buf + j * 1024), "v"(off[j]), "s"(rw), "s"(so) : "memory", "m0");
#pragma unroll
        for (int j = 0; j < PX; ++j)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(buf + 16 * ROW + j * 1024), "v"(off[j]), "s"(rx), "s"(so) : "memory", "m0");
    };
    gv_f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = gv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NB; ++i)
        if (i < mine) fetch(i, lds0 + i * BUF);
    uint32_t buf = lds0;
    const uint32_t wrd = (uint32_t)r16 * ROW;
    uint32_t xrd[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) xrd[t] = 16u * ROW + (uint32_t)((16 * t + r16) & (XR - 1)) * ROW;
    for (int i = 0; i < mine; ++i) {
        if (i + NB <= mine) KW_WAIT((NB - 1) * P); else KW_WAIT(0);      // this chunk has landed (the last ones: all of them)
#pragma unroll
        for (int h = 0; h < CH / 32; h += 4) {                   // four fragments of 32 k at a time
            kw_u32x4 wf[4], xf[4][MT];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t g = (uint32_t)((4 * (h + u) + kb) ^ (r16 & (GR - 1))) * 16u;
                asm volatile("ds_read_b128 %0, %1" : "=v"(wf[u]) : "v"(buf + wrd + g));
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const uint32_t gx = (uint32_t)((4 * (h + u) + kb) ^ (((16 * t + r16) & (XR - 1)) & 15 & (GR - 1))) * 16u;
                    asm volatile("ds_read_b128 %0, %1" : "=v"(xf[u][t]) : "v"(buf + xrd[t] + gx));
                }
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                asm volatile("" : "+v"(wf[u]));
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    asm volatile("" : "+v"(xf[u][t]));
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[u]), __builtin_bit_cast(bf16x8_t, xf[u][t]), acc[t], 0, 0, 0);
                }
            }
        }
        if (i + NB < mine) fetch(i + NB, buf);                   // (the chunk has been read: its place takes the next but NB)
        buf = buf + BUF == lds0 + NB * BUF ? lds0 : buf + BUF;
    }
    __syncthreads();                                             // (every wave's loads have landed and been read: the partial tiles go over them)
    gv_f32x4* part = (gv_f32x4*)kw_lds;
#pragma unroll
    for (int t = 0; t < MT; ++t) part[(t * WAVES + wave) * 64 + lane] = acc[t];
    __syncthreads();
    if (wave < MT) {
        gv_f32x4 a_ = part[wave * WAVES * 64 + lane];
#pragma unroll
        for (int q = 1; q < WAVES; ++q) a_ += part[(wave * WAVES + q) * 64 + lane];
        const int m = 16 * wave + r16;
        if constexpr (EP == 3) {
            float o[4], q = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                auto one = [&](uint2 v) { const uint32_t h = r < 2 ? v.x : v.y; return r & 1 ? bf_hi(h) : bf_lo(h); };
                o[r] = a_[r] + (bias ? one(pb) : 0.f);
                o[r] = round_bf(o[r] + one(pr));
                q = fmaf(o[r], o[r], q);
            }
            q += __shfl_xor(q, 16, 64);
            q += __shfl_xor(q, 32, 64);
            if (m < M) {
                const int64_t at = (int64_t)m * N + n0 + 4 * kb;
                *(uint2*)(y + at) = make_uint2(pack_bf2(o[0], o[1]), pack_bf2(o[2], o[3]));
                *(uint2*)(xg + at) = make_uint2(pack_bf2(o[0] * bf_lo(pg.x), o[1] * bf_hi(pg.x)), pack_bf2(o[2] * bf_lo(pg.y), o[3] * bf_hi(pg.y)));
                if (kb == 0) ss[(int64_t)m * gridDim.x + blockIdx.x] = q;
            }
            return;
        }
        if (m < M) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int n = n0 + 4 * kb + r;
                if (n < N) {
                    auto one = [&](uint2 v) { const uint32_t h = r < 2 ? v.x : v.y; return r & 1 ? bf_hi(h) : bf_lo(h); };
                    float o = a_[r] + (EP && bias ? one(pb) : 0.f);
                    if (EP && res) o += one(pr);
                    y[(int64_t)m * N + n] = f_to_bf(out_act(o, act));
                }
            }
        }
    }
}

template <int XR, int WAVES, int CH, int NB, int EP>
static int kw_go(const void* x, const void* w, const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t K, int act, hipStream_t s,
                 const void* scale = nullptr, void* xg = nullptr, float* ss = nullptr) {
    constexpr size_t lds = (size_t)WAVES * NB * (16 + XR) * 2 * CH;
    static_assert(lds <= 160 * 1024, "the CU's LDS");
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)skinny_kw_kernel<XR, WAVES, CH, NB, EP>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((skinny_kw_kernel<XR, WAVES, CH, NB, EP>), dim3((unsigned)((N + 15) / 16)), dim3(64 * WAVES), lds, s, (const unsigned char*)x,
                       (const unsigned char*)w, (const uint16_t*)bias, (const uint16_t*)residual, (uint16_t*)y, (int)M, (int)N, (int)K, act, (const uint16_t*)scale, (uint16_t*)xg, ss);
    return evo_launch_status();
}
// (a form of its own for layers without bias and residual: the requests in front of their loop cost 0.2 to 0.3 us there)
template <int XR, int WAVES, int CH, int NB>
static int kw_launch(const void* x, const void* w, const void* bias, const void* residual, void* y, int64_t M, int64_t N, int64_t K, int act, hipStream_t s) {
    if (!bias && !residual) return kw_go<XR, WAVES, CH, NB, 0>(x, w, bias, residual, y, M, N, K, act, s);
    if (N % 4 == 0 && (((uintptr_t)bias | (uintptr_t)residual) & 7) == 0) return kw_go<XR, WAVES, CH, NB, 2>(x, w, bias, residual, y, M, N, K, act, s);
    return kw_go<XR, WAVES, CH, NB, 1>(x, w, bias, residual, y, M, N, K, act, s);
}

// ---- 3 to 64 rows on the wide layers (and, with parts of K, on those of up to 8,192 columns from 17 rows on): a workgroup owns N / gridDim.x weight rows (any number up to
// 16 T, a wave per 16 of them) and walks K in chunks of 128; weight and batch rows of a chunk arrive in LDS by asynchronous loads (no registers) into a ring
// of NB stages, NB - 1 of them under way, one barrier per chunk.  LDS rows of 256 B, granule g of row r at slot g ^ (r & 15): a fragment read meets no bank twice.
// What bounds it is the weight stream, under three conditions that decide the layout (us, MI355X, launches back to back; a plain read of the matrix in brackets):
//  * every CU has the same number of rows: 22,016 x 4,096 [26.3] at 16 rows takes 28.6 in 256 x 86 rows, 36.2 in 344 x 64;
//  * workgroups of one XCD don't walk K in step: rows lie a power of two apart, so equal places of K are the same L2 channels.  Starts one chunk apart by turns
//    took 16,384 x 4,096 [22.0] at 16 rows from 34.8 to 21.4 (32 rows a workgroup), 8,192 x 28,672 [69] from 107 to 69;
//  * the batch rows, read once per workgroup, are few against its weight rows.
// At 8 / 16 / 32 / 64 rows: 22,016 x 4,096 32.6 / 33.4 / 36.6 / 46.4 (register-staged chunks, 64 rows a workgroup, all from K = 0 on) -> 28.4 / 28.6 / 29.4 / 32.5;
// 16,384 x 4,096 26.1 / 26.3 / 29.2 / 36.3 -> 22.1 / 22.3 / 23.2 / 26.0; 12,288 x 4,096 [16.0] 20.8 / 21.4 / 22.4 / 34.0 -> 17.1 / 17.1 / 17.6 / 21.8;
// 8,192 x 4,096 [11.4] 20.4 / 20.4 / 21.1 / 30.6 -> 12.1 / 12.3 / 13.8 / 17.5.
// MODE 0: y = x w^T (+ bias, + residual, activation).  MODE 1: the gated MLP's first half [REF stripedhyena/layers.py ParallelGatedMLP: gelu(l1 x) * l2 x]: a wave's 16
// rows are 8 of W1 and the same 8 of W2 (`layout` 1: HipOps.pack_gate_weights' blocks of 32 + 32 rows, 2: plain [W1; W2]), z2 crosses by one lane exchange, both are
// rounded to bf16 (the dense layer's outputs), the gate is evaluated in fp32 and rounded once; N = 2 I, y = a [M, I].  A column's first chunk follows its place:
// where N >= 16,384 is no multiple of 4,096 workgroup b of MODE 1 starts where b / 2 and b / 2 + half of MODE 0 do, which hold its columns of plain [W1; W2]: both
// give the same bits there.
// MODE 2: blockIdx.y is a part of K, fp32 partial sums to ws [parts][M][N] (skinny_reduce_kernel adds them in order).
typedef uint32_t rg_u32x4 __attribute__((ext_vector_type(4)));
#define RG_WAIT(N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory")
#define RG_ROWB 256                          // bytes of a row's piece of a chunk
#define RG_NONE 0xf0000000u                  // behind every buffer: nothing is read, zero arrives
// first of the columns of workgroup `b` (b = groups: behind the last): floor(b cols / groups).  b * more has 32 bits up to 65,536 workgroups only (6.3 M columns).
static __host__ __device__ __forceinline__ uint32_t ring_edge(uint32_t cols, uint32_t groups, uint32_t b) {
    const uint32_t each = cols / groups, more = cols % groups;
    return b * each + (groups <= 0x10000 ? b * more / groups : (uint32_t)((uint64_t)b * more / groups));
}
// RS: x is a row times the scale of its norm, and its products are taken times 1 / (rms + eps) of the row, from the sums of squares ss [M][strips] (skinny_kw_kernel, EP 3): the norm
// between two layers without a launch.  The sums are asked for ahead of the stream and added up behind it, 0.3 us; the launch was 2.6.  Pools of 5 / 8 / 16 / 24 / 32
// short prompts, four layers, 32 steps (seven norms a step; three from 17 rows on, whose l3 is summed in parts): 12.88 / 13.46 / 15.11 / 16.88 / 18.33 -> 12.53 / 12.98 / 14.54 / 16.58 /
// 18.03 ms, logits as far from 64 bits as before (7.9e-3 -> 7.8e-3 to 7.9e-3).
template <int XR, int T, int NB, int MODE, bool RS = false>
__global__ __launch_bounds__(64 * T) void skinny_ring_kernel(const unsigned char* __restrict__ x, const unsigned char* __restrict__ w, const uint16_t* __restrict__ bias,
                                                             const uint16_t* res, uint16_t* y, int M, int N, int K, int act, int layout, float* __restrict__ ws,
                                                             const float* __restrict__ ss, int strips, float eps, float inv_sqrt_d) {   // res may alias y
    constexpr int MT = XR / 16, PX = (XR / 4 + T - 1) / T, PW = 4, P = PX + PW;      // requests of 1 KiB (4 rows) per wave and chunk
    constexpr int XOFF = T * 16 * RG_ROWB, BUF = XOFF + T * PX * 1024;
    static_assert(XR % 16 == 0 && NB >= 2 && (NB - 2) * P < 64, "the wait counter has six bits");
    extern __shared__ __attribute__((aligned(16))) unsigned char rg_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kb = lane >> 4;
    const uint32_t rowb = (uint32_t)K * 2;
    const int cols = MODE == 1 ? N >> 1 : N;                     // result columns; this workgroup's: lo .. hi - 1
    const int lo = (int)ring_edge(cols, gridDim.x, blockIdx.x), hi = (int)ring_edge(cols, gridDim.x, blockIdx.x + 1);
    // weight rows: four requests of four rows; of MODE 1 the first two from W1, the others from W2
    rg_u32x4 rw[2];
    uint32_t ow[PW];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const bool grouped = MODE == 1 && layout == 1;
        const int64_t first = MODE != 1 ? lo : (grouped ? 64 * (int64_t)(lo >> 5) + 32 * h : (int64_t)h * cols + lo);
        const uint64_t a = (uint64_t)w + (uint64_t)first * rowb;
        const uint32_t rows = grouped ? 64 * (((hi - 1) >> 5) - (lo >> 5)) + 32 : hi - lo;
        rw[h] = rg_u32x4{(uint32_t)a, (uint32_t)(a >> 32) & 0xffffu, rows * rowb, 0x00020000u};
    }
#pragma unroll
    for (int i = 0; i < PW; ++i) {
        const int q = i * 4 + (lane >> 4), c = MODE == 1 ? lo + 8 * wave + (q & 7) : lo + 16 * wave + q;     // row of the tile, its column
        const int r = MODE == 1 && layout == 1 ? 64 * ((c >> 5) - (lo >> 5)) + (c & 31) : c - lo;
        ow[i] = c < hi ? (uint32_t)r * rowb + (uint32_t)((lane & 15) ^ q) * 16u : RG_NONE;
    }
    const uint64_t xa = (uint64_t)x;
    const rg_u32x4 rx = {(uint32_t)xa, (uint32_t)(xa >> 32) & 0xffffu, (uint32_t)M * rowb, 0x00020000u};
    uint32_t ox[PX];
#pragma unroll
    for (int i = 0; i < PX; ++i) {
        const int r = (wave * PX + i) * 4 + (lane >> 4);
        ox[i] = r < M ? (uint32_t)r * rowb + (uint32_t)((lane & 15) ^ (r & 15)) * 16u : RG_NONE;
    }
    // bias and residual values of this lane's results, requested ahead of everything (from places that are there, and looked at behind the last product: no wait here)
    uint32_t pb[4], pr[MODE == 0 ? MT : 1][4];
    const uint32_t n0 = (uint32_t)lo + 16 * wave + 4 * kb;       // (may be behind 2^31)
    if (MODE == 0 && bias) {
#pragma unroll
        for (int r = 0; r < 4; ++r) pb[r] = bias[n0 + r < N ? n0 + r : N - 1];
    }
    if (MODE == 0 && res) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const uint16_t* from = res + (int64_t)(16 * t + r16 < M ? 16 * t + r16 : M - 1) * N;
#pragma unroll
            for (int r = 0; r < 4; ++r) pr[t][r] = from[n0 + r < N ? n0 + r : N - 1];
        }
    }
    constexpr int RW = RS ? (XR + T - 1) / T : 1;                // rows whose sums a wave adds: wave, wave + T, ..
    gv_f32x4 sq[RW];
    __shared__ float rs_s[RS ? RW * T : 1];
    if constexpr (RS) {
#pragma unroll
        for (int j = 0; j < RW; ++j) sq[j] = *(const gv_f32x4*)(ss + (int64_t)(wave + T * j < M ? wave + T * j : M - 1) * strips + (4 * lane < strips ? 4 * lane : 0));
    }
    const int all = K / 128, c0 = MODE == 2 ? (int)((int64_t)all * blockIdx.y / gridDim.y) : 0;
    const int chunks = (MODE == 2 ? (int)((int64_t)all * (blockIdx.y + 1) / gridDim.y) : all) - c0;
    // (block b runs on XCD b % 8; where halves start alike they meet in the L2 channels if they lie a power of two apart: 8,192 x 4,096 at 8 rows 16.2 us, 12.1 without)
    const bool halves = N >= 16384 && (N & 4095) != 0;
    int at = (int)(halves ? (MODE == 1 ? blockIdx.x >> 1 : blockIdx.x) >> 3 & 15 : blockIdx.x >> 3) % chunks;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)rg_lds;
    auto fetch = [&](uint32_t buf) {
        const uint32_t so = (uint32_t)(c0 + at) * RG_ROWB;
#pragma unroll
        for (int j = 0; j < PX; ++j)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(buf + XOFF + (wave * PX + j) * 1024), "v"(ox[j]), "s"(rx), "s"(so) : "memory", "m0");
#pragma unroll
        for (int j = 0; j < PW; ++j)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds" ::"s"(buf + (wave * PW + j) * 1024), "v"(ow[j]), "s"(rw[j >> 1]), "s"(so) : "memory", "m0");
        at = at + 1 == chunks ? 0 : at + 1;
    };
    gv_f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = gv_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NB - 1; ++i)
        if (i < chunks) fetch(lds0 + i * BUF);
    uint32_t buf = lds0, nxt = lds0 + (NB - 1) * BUF, g[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) g[u] = (uint32_t)r16 * RG_ROWB + (uint32_t)((4 * u + kb) ^ r16) * 16u;
    for (int i = 0; i < chunks; ++i) {
        if (i + NB - 1 <= chunks) RG_WAIT((NB - 2) * P); else RG_WAIT(0);      // this wave's part of chunk i has landed,
        asm volatile("s_barrier" ::: "memory");                                // every wave's; and every wave has read chunk i - 1, whose place is free
        if (i + NB - 1 < chunks) fetch(nxt);
        nxt = nxt + BUF == lds0 + NB * BUF ? lds0 : nxt + BUF;
#pragma unroll
        for (int h = 0; h < 4; h += 2) {
            rg_u32x4 wf[2], xf[2][MT];
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                asm volatile("ds_read_b128 %0, %1" : "=v"(wf[u]) : "v"(buf + wave * (16 * RG_ROWB) + g[h + u]));
#pragma unroll
                for (int t = 0; t < MT; ++t) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(xf[u][t]) : "v"(buf + XOFF + g[h + u]), "n"(t * 16 * RG_ROWB));
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                asm volatile("" : "+v"(wf[u]));
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    asm volatile("" : "+v"(xf[u][t]));
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, wf[u]), __builtin_bit_cast(bf16x8_t, xf[u][t]), acc[t], 0, 0, 0);
                }
            }
        }
        buf = buf + BUF == lds0 + NB * BUF ? lds0 : buf + BUF;
    }
    if constexpr (RS) {
#pragma unroll
        for (int j = 0; j < RW; ++j) {
            const float sum = wave_sum(4 * lane < strips ? (sq[j][0] + sq[j][1]) + (sq[j][2] + sq[j][3]) : 0.f);
            if (lane == 0) rs_s[wave + T * j] = 1.0f / (sqrtf(sum) * inv_sqrt_d + eps);
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const float f = rs_s[16 * t + r16];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][r] *= f;
        }
    }
    // D[n][m]: lane holds rows 4 kb + r of its wave's tile, m = 16 t + r16
    if constexpr (MODE == 1) {
        const int c = lo + 8 * wave + 4 * (kb & 1);              // kb 0, 1: columns c .. c + 3 of W1; kb 2, 3: the same of W2
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            float z[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) z[r] = __shfl_xor(acc[t][r], 32, 64);
            const int m = 16 * t + r16;
            if (kb < 2 && m < M) {
                const f32x2_t ua = {round_bf(acc[t][0]), round_bf(acc[t][1])}, ub = {round_bf(acc[t][2]), round_bf(acc[t][3])};
                const f32x2_t oa = act_gate2(ua, f32x2_t{round_bf(z[0]), round_bf(z[1])}, act), ob = act_gate2(ub, f32x2_t{round_bf(z[2]), round_bf(z[3])}, act);
                uint16_t* to = y + (int64_t)m * cols + c;
                const float o[4] = {oa[0], oa[1], ob[0], ob[1]};
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (c + r < hi) to[r] = f_to_bf(o[r]);
            }
        }
    } else if constexpr (MODE == 2) {                            // (N / gridDim.x a multiple of 4: the host checks)
#pragma unroll
        for (int t = 0; t < MT; ++t)
            if (16 * t + r16 < M && n0 < hi) *(gv_f32x4*)(ws + ((int64_t)blockIdx.y * M + 16 * t + r16) * N + n0) = acc[t];
    } else {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            float o[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                o[r] = acc[t][r];
                if (bias) o[r] += bf_to_f((uint16_t)pb[r]);
                if (res) o[r] += bf_to_f((uint16_t)pr[t][r]);
                o[r] = out_act(o[r], act);
            }
            if (16 * t + r16 < M) {
                uint16_t* to = y + (int64_t)(16 * t + r16) * N + n0;
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n0 + r < hi) to[r] = f_to_bf(o[r]);
            }
        }
    }
}

// y [M, N] = sum over slices of ws [slices][M][N] (in slice order: deterministic) + bias + residual, one rounding; a thread owns four columns
__global__ __launch_bounds__(256) void skinny_reduce_kernel(const float* __restrict__ ws, const uint16_t* __restrict__ bias, const uint16_t* res,
                                                            uint16_t* y, int M, int N, int slices, int act) {   // res may alias y
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x, total = (int64_t)M * N / 4;
    if (q >= total) return;
    const int64_t e = q * 4;
    const int n = (int)(e % N);
    gv_f32x4 a = *(const gv_f32x4*)(ws + e);
    for (int sl = 1; sl < slices; ++sl) a += *(const gv_f32x4*)(ws + (int64_t)sl * M * N + e);
    float o[4] = {a[0], a[1], a[2], a[3]};
    if (bias) { const uint2 b = *(const uint2*)(bias + n); o[0] += bf_lo(b.x); o[1] += bf_hi(b.x); o[2] += bf_lo(b.y); o[3] += bf_hi(b.y); }
    if (res) { const uint2 r = *(const uint2*)(res + e); o[0] += bf_lo(r.x); o[1] += bf_hi(r.x); o[2] += bf_lo(r.y); o[3] += bf_hi(r.y); }
    uint2 out;
    out.x = pack_bf2(out_act(o[0], act), out_act(o[1], act));
    out.y = pack_bf2(out_act(o[2], act), out_act(o[3], act));
    *(uint2*)(y + e) = out;
}

// Ring launches.  Rows per workgroup: up to 24,576 columns what 256 CUs get each, at least 32; more columns are rounds of up to 64 rows; T: waves for them.  Stages: four
// (42 KB each at T = 6 and 64 batch rows: three); of several rounds three, two at 64 batch rows, so that a CU starts its next workgroup while one ends.  us at 5 / 16 / 32 / 64
// rows, rounds of up to 96 rows and four stages -> this: 28,672 x 1,024 11.6 / 12.3 / 15.4 / 20.0 -> 11.4 / 12.2 / 13.7 / 16.7, 50,304 x 1,024 22.4 / 24.1 / 27.1 / 33.0 ->
// 18.4 / 19.7 / 23.4 / 31.4, 65,536 x 4,096 78 / 80 / 86 / 102 -> 79 / 78 / 80 / 95, 151,936 x 512 34 / 40 / 47 / 59 -> 28 / 32 / 38 / 55 (x 4,096 179 / 192 / 214 / 251 ->
// 182 / 191 / 216 / 263).
struct RingNorm { const float* ss; int strips; float eps, inv_sqrt_d; };     // RS
template <int XR, int T, int MODE, int NB, bool RS = false>
static int ring_go(dim3 grid, const void* x, const void* w, const void* bias, const void* res, void* y, int64_t M, int64_t N, int64_t K, int act, int layout, float* ws,
                   hipStream_t s, RingNorm n = {}) {
    constexpr size_t lds = (size_t)NB * T * (16 * RG_ROWB + (XR / 4 + T - 1) / T * 1024);
    static_assert(lds <= 160 * 1024, "the CU's LDS");
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)skinny_ring_kernel<XR, T, NB, MODE, RS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((skinny_ring_kernel<XR, T, NB, MODE, RS>), grid, dim3(64 * T), lds, s, (const unsigned char*)x, (const unsigned char*)w, (const uint16_t*)bias,
                       (const uint16_t*)res, (uint16_t*)y, (int)M, (int)N, (int)K, act, layout, ws, n.ss, n.strips, n.eps, n.inv_sqrt_d);
    return evo_launch_status();
}
// 4,097 to 7,680 columns from K = 4,096 on (to 7,168: from 2,048): a workgroup per CU here too, of 17 to 30 columns in two waves.  A CU takes in 45 to 55 GB/s while lines come
// from memory, however many are under way, and 132 to 240 workgroups left the others idle (and, to 16 rows, six stages of their 12 KB: 36 KB under way are too few).  Four
// stages and 32 columns -> this, us at 5 / 16 / 24 / 32 rows, weights cold: 4,224 x 4,096 13.3 / 13.7 / 12.7 / 13.3 -> 11.9 / 11.1 / 12.8 / 12.9, 6,144 x 4,096 14.1 / 14.4 / 15.2 /
// 14.2 -> 11.9 / 12.3 / 14.6 / 13.6, 6,720 x 4,096 14.5 / 14.7 / 15.2 / 16.0 -> 12.5 / 13.0 / 14.8 / 14.0, x 11,008 30.2 / 30.9 / 33.4 / 34.9 -> 27.3 / 28.3 / 32.6 / 33.8.  Over 861
// layers, plain and gated, K = 2,048 to 16,384: to 16 rows 0.98 to 1.28, 17 to 32 rows 0.97 to 1.15, 33 to 64 rows 0.96 to 1.10; behind at 17 and 24 rows of K = 2,048 and 4,096 and at 40
// rows, gated, by up to 0.3 and 1.8 us.  Beyond, 31 and 32 columns a workgroup are as good (8,000 x 4,096 14.2 : 14.6), and at small K nothing is gained (6,144 x 1,024 4.9 :
// 5.0, 7,680 x 2,048 7.5 : 7.7).
static bool ring_spread(int64_t N, int64_t K) { return N > 4096 && (N <= 7168 ? K >= 2048 : N <= 7680 && K >= 4096); }
static int64_t ring_groups(int64_t N, int64_t K) {
    const int64_t share = (N + 31) / 32;
    return ring_spread(N, K) ? 256 : share < 256 ? share : N <= 256 * 96 ? 256 : 256 * ((N + 256 * 64 - 1) / (256 * 64));
}
static int ring_waves(int64_t N, int64_t K) {
    const int64_t groups = ring_groups(N, K), rows = (N + groups - 1) / groups;
    return rows <= 32 ? 2 : rows <= 48 ? 3 : rows <= 64 ? 4 : 6;
}
// What workgroup `block` of N weight rows (gated: N / 2 result columns) takes: out = workgroups, its first column, the next one's, columns that it has room for
extern "C" int evo_linear_ring_share(int64_t N, int64_t K, int64_t gated, int64_t block, int64_t* out) {
    if (!out || N <= 0 || N > 0x7fffffff - 16 || K <= 0 || K % 128 || (gated && N % 2)) return -1;
    const int64_t groups = ring_groups(N, K), cols = gated ? N / 2 : N;
    if (block < 0 || block >= groups) return -1;
    out[0] = groups;
    out[1] = ring_edge((uint32_t)cols, (uint32_t)groups, (uint32_t)block);
    out[2] = ring_edge((uint32_t)cols, (uint32_t)groups, (uint32_t)block + 1);
    out[3] = (gated ? 8 : 16) * ring_waves(N, K);
    return 0;
}
// parts > 0: MODE 2, 64 rows a workgroup (N a multiple of 64)
template <int MODE>
static int ring_launch(const void* x, const void* w, const void* bias, const void* res, void* y, int64_t M, int64_t N, int64_t K, int act, int layout, float* ws, int parts,
                       hipStream_t s) {
    const int waves = ring_waves(N, K);
    const dim3 grid((unsigned)(parts ? N / 64 : ring_groups(N, K)), (unsigned)(parts ? parts : 1));
#define EVO_RG(XR, T, NB) ring_go<XR, T, MODE, NB>(grid, x, w, bias, res, y, M, N, K, act, layout, ws, s)
#define EVO_RG1(T) (M <= 16 ? EVO_RG(16, T, 4) : M <= 32 ? EVO_RG(32, T, 4) : EVO_RG(64, T, (T == 6 ? 3 : 4)))
#define EVO_RGN(T) (M <= 16 ? EVO_RG(16, T, 3) : M <= 32 ? EVO_RG(32, T, 3) : EVO_RG(64, T, 2))
    if constexpr (MODE == 2) return EVO_RG1(4);
    else {
        if (grid.x > 256) return waves == 3 ? EVO_RGN(3) : EVO_RGN(4);         // (33 to 64 rows)
        if (M <= 16 && ring_spread(N, K)) return EVO_RG(16, 2, 6);
        return waves == 2 ? EVO_RG1(2) : waves == 3 ? EVO_RG1(3) : waves == 4 ? EVO_RG1(4) : EVO_RG1(6);
    }
#undef EVO_RGN
#undef EVO_RG1
#undef EVO_RG
}

// RS, 5 to 32 rows and up to 24,576 weight rows: as many waves and stages as ring_launch takes
template <int MODE>
static int ring_factors(const void* x, const void* w, const void* bias, void* y, int64_t M, int64_t N, int64_t K, int layout, RingNorm n, hipStream_t s) {
    const int waves = ring_waves(N, K);
    const dim3 grid((unsigned)ring_groups(N, K));
    if (grid.x > 256) return -1;
#define EVO_RF(XR, T, NB) ring_go<XR, T, MODE, NB, true>(grid, x, w, bias, nullptr, y, M, N, K, 0, layout, nullptr, s, n)
#define EVO_RF1(T) (M <= 16 ? EVO_RF(16, T, 4) : EVO_RF(32, T, 4))
    if (M <= 16 && ring_spread(N, K)) return EVO_RF(16, 2, 6);
    return waves == 2 ? EVO_RF1(2) : waves == 3 ? EVO_RF1(3) : waves == 4 ? EVO_RF1(4) : EVO_RF1(6);
#undef EVO_RF1
#undef EVO_RF
}

template <int M>
static void gemv_launch(const void* x, const void* w, const void* bias, const void* res, void* y, int64_t N, int64_t K,
                        int act, hipStream_t s) {
    // rows per wave.  Measured (tools/bench_gemv.py, MI355X): R=4 wins for every M (R=8 starves the chip of
    // waves at N=4096; R=2 doubles the L2 re-reads of x): 4.9-5.4 TB/s at M=1-2, 3.0-3.6 TB/s at M=8.
#ifndef GEMV_R_A
#define GEMV_R_A 4
#endif
#ifndef GEMV_R_B
#define GEMV_R_B 4
#endif
#ifndef GEMV_R_C
#define GEMV_R_C 4
#endif
    constexpr int R = M <= 2 ? GEMV_R_A : (M <= 4 ? GEMV_R_B : GEMV_R_C);
    const int64_t waves = (N + R - 1) / R;
    if (N <= 4096 && K >= 2048)
        hipLaunchKernelGGL((gemv_kernel<M, R, true>), dim3((unsigned)waves), dim3(256), 0, s, (const uint4*)x,
                           (const uint4*)w, (const uint16_t*)bias, (const uint16_t*)res, (uint16_t*)y, (int)N, (int)(K / 8), act);
    else
        hipLaunchKernelGGL((gemv_kernel<M, R, false>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, (const uint4*)x,
                           (const uint4*)w, (const uint16_t*)bias, (const uint16_t*)res, (uint16_t*)y, (int)N, (int)(K / 8), act);
}

extern "C" int evo_norm_linear_small_m_bf16(const void* x, const void* scale, const void* w, const void* bias, void* y,
                                            int64_t M, int64_t N, int64_t K, float eps, void* stream) {
    if (M < 1 || M > 8 || N <= 0 || K <= 0 || K % 8 != 0 || N > 0x7fffffff - 16) return -1;
    if (M > 4 && K != 4096) return -1;                       // batches of 5-8 rows exist in the LDS-staged form only
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)(((N + 3) / 4 + 3) / 4)), block(256);
    const float isd = 1.0f / sqrtf((float)K);
    const size_t lds = (size_t)M * K * 2;                   // normalised rows staged in LDS (when they fit)
    const bool stage = K == 4096;                            // the staged kernels are written out for four 1024-element trips
#define EVO_NL(MM)                                                                                            \
    if (stage)                                                                                                \
        hipLaunchKernelGGL((gemv_norm_kernel<MM, 4, true>), grid, block, lds, s, (const uint4*)x, (const uint4*)scale, \
                           (const uint4*)w, (const uint16_t*)bias, (uint16_t*)y, (int)N, (int)(K / 8), eps, isd); \
    else                                                                                                      \
        hipLaunchKernelGGL((gemv_norm_kernel<MM, 4, false>), grid, block, 0, s, (const uint4*)x, (const uint4*)scale, \
                           (const uint4*)w, (const uint16_t*)bias, (uint16_t*)y, (int)N, (int)(K / 8), eps, isd)
#define EVO_NLS(MM)                                                                                           \
    hipLaunchKernelGGL((gemv_norm_kernel<MM, 4, true>), grid, block, lds, s, (const uint4*)x, (const uint4*)scale, \
                       (const uint4*)w, (const uint16_t*)bias, (uint16_t*)y, (int)N, (int)(K / 8), eps, isd)
    switch (M) {
        case 1: EVO_NL(1); break;
        case 2: EVO_NL(2); break;
        case 3: EVO_NL(3); break;
        case 4: EVO_NL(4); break;
        case 5: EVO_NLS(5); break;
        case 6: EVO_NLS(6); break;
        case 7: EVO_NLS(7); break;
        default: EVO_NLS(8); break;
    }
#undef EVO_NLS
#undef EVO_NL
    return evo_launch_status();
}

extern "C" int evo_hyena_decode_fused_small_m(const void* x, const void* norm_scale, const void* proj_w, const void* proj_b,
                                              void* fir_state, float* iir_state, const void* fir_w, const void* fir_b,
                                              const float* poles, const float* residues, const void* dskip, void* y,
                                              int64_t M, int64_t D, int64_t n_heads, float eps, void* stream) {
    if (M < 1 || M > 8 || D <= 0 || D != n_heads * 128 || D % 8 != 0) return -1;
    if (M > 4 && D != 4096) return -1;                       // batches of 5-8 rows exist in the LDS-staged form only
    hipStream_t s = (hipStream_t)stream;
    // channels per wave, measured under a hipGraph on MI355X (tools/experiments/hyena_decode_cpw_bench.py): one channel per wave
    // (twice the waves, half the bytes in flight each) is 5 % faster at M = 1 and 6 % at M = 4, two channels win at M = 2
    // (22.8 / 26.1 / 42.6 us with two, 21.6 / 29.9 / 40.0 us with one, M = 1 / 2 / 4).  Same arithmetic either way.
#ifndef GEMV_HYENA_CPW_STAGED
#define GEMV_HYENA_CPW_STAGED 1
#endif
#ifndef GEMV_HYENA_CPW_STAGED1
#define GEMV_HYENA_CPW_STAGED1 1
#endif
    const float isd = 1.0f / sqrtf((float)D);
    const size_t lds = (size_t)M * D * 2;
#define EVO_HD(MM, CPW, ST)                                                                                   \
    hipLaunchKernelGGL((gemv_norm_hyena_kernel<MM, CPW, ST>), dim3((unsigned)((D / CPW + 3) / 4)), dim3(256), ST ? lds : 0, s, \
                       (const uint4*)x, (const uint4*)norm_scale,                                             \
                       (const uint4*)proj_w, (const uint16_t*)proj_b, (uint16_t*)fir_state, iir_state,          \
                       (const uint16_t*)fir_w, (const uint16_t*)fir_b, poles, residues, (const uint16_t*)dskip, \
                       (uint16_t*)y, (int)D, (int)(D / 8), eps, isd)
    const bool stage = D == 4096;
    switch (M) {
        case 1: if (stage) EVO_HD(1, GEMV_HYENA_CPW_STAGED1, true); else EVO_HD(1, 1, false); break;
        case 2: if (stage) EVO_HD(2, GEMV_HYENA_CPW_STAGED, true); else EVO_HD(2, 2, false); break;
        case 3: if (stage) EVO_HD(3, GEMV_HYENA_CPW_STAGED, true); else EVO_HD(3, 2, false); break;
        case 4: if (stage) EVO_HD(4, GEMV_HYENA_CPW_STAGED, true); else EVO_HD(4, 1, false); break;
        case 5: EVO_HD(5, 1, true); break;
        case 6: EVO_HD(6, 1, true); break;
        case 7: EVO_HD(7, 1, true); break;
        default: EVO_HD(8, 1, true); break;
    }
#undef EVO_HD
    return evo_launch_status();
}

static int mlp_gate_launch(const void* x, const void* scale, const void* w12, void* a, int64_t M, int64_t I, int64_t K,
                           float eps, int64_t grouped, int act, hipStream_t s) {
    if (M < 1 || M > 8 || I <= 0 || I % 2 != 0 || K <= 0 || K % 8 != 0 || I > 0x3fffffff) return -1;
    if (grouped && I % 32 != 0) return -1;
    const int grp = grouped ? 1 : 0;
    if (M > 4 && !(scale && K == 4096)) return -1;           // batches of 5-8 rows exist in the LDS-staged form only
    const dim3 grid((unsigned)((I / 2 + 3) / 4)), block(256);
    const float isd = 1.0f / sqrtf((float)K);
    const size_t lds = (size_t)M * K * 2;
    const bool stage = scale && K == 4096;
#define EVO_MG(MM)                                                                                            \
    if (scale && stage)                                                                                       \
        hipLaunchKernelGGL((gemv_gate_kernel<MM, true, true>), grid, block, lds, s, (const uint4*)x, (const uint4*)scale, \
                           (const uint4*)w12, (uint16_t*)a, (int)I, (int)(K / 8), eps, isd, grp, act);             \
    else if (scale)                                                                                           \
        hipLaunchKernelGGL((gemv_gate_kernel<MM, true, false>), grid, block, 0, s, (const uint4*)x, (const uint4*)scale, \
                           (const uint4*)w12, (uint16_t*)a, (int)I, (int)(K / 8), eps, isd, grp, act);             \
    else                                                                                                      \
        hipLaunchKernelGGL((gemv_gate_kernel<MM, false, false>), grid, block, 0, s, (const uint4*)x, (const uint4*)nullptr, \
                           (const uint4*)w12, (uint16_t*)a, (int)I, (int)(K / 8), 0.f, 0.f, grp, act)
#define EVO_MGS(MM)                                                                                           \
    hipLaunchKernelGGL((gemv_gate_kernel<MM, true, true>), grid, block, lds, s, (const uint4*)x, (const uint4*)scale, \
                       (const uint4*)w12, (uint16_t*)a, (int)I, (int)(K / 8), eps, isd, grp, act)
    switch (M) {
        case 1: EVO_MG(1); break;
        case 2: EVO_MG(2); break;
        case 3: EVO_MG(3); break;
        case 4: EVO_MG(4); break;
        case 5: EVO_MGS(5); break;
        case 6: EVO_MGS(6); break;
        case 7: EVO_MGS(7); break;
        default: EVO_MGS(8); break;
    }
#undef EVO_MGS
#undef EVO_MG
    return evo_launch_status();
}

extern "C" int evo_mlp_gate_small_m_bf16(const void* x, const void* w12, void* a, int64_t M, int64_t I, int64_t K,
                                         int64_t grouped, int64_t act, void* stream) {
    if (act != 0 && act != 1) return -1;
    // (three and four rows: 34.4 -> 28.6 us at I = 11,008, K = 4,096; small layers, or where the asynchronous loads can't go, keep the dot2 form)
    const bool ring = I > 0 && I % 32 == 0 && K > 0 && K % 128 == 0 && I <= 0x1fffffff && K <= 0x9fffff && (((uintptr_t)x | (uintptr_t)w12) & 15) == 0;
    if (M >= 5 ? M <= 64 : (M >= 3 && ring && I * K >= 1 << 24)) {
        // the MFMA weight-streaming form with the gate in its epilogue, both weight layouts
        if (!ring) return -1;
        return ring_launch<1>(x, w12, nullptr, nullptr, a, M, 2 * I, K, (int)act, grouped ? 1 : 2, nullptr, 0, (hipStream_t)stream);
    }
    return mlp_gate_launch(x, nullptr, w12, a, M, I, K, 0.f, grouped, (int)act, (hipStream_t)stream);
}

extern "C" int evo_norm_mlp_gate_small_m_bf16(const void* x, const void* scale, const void* w12, void* a, int64_t M,
                                              int64_t I, int64_t K, float eps, int64_t grouped, void* stream) {
    if (!scale) return -1;
    return mlp_gate_launch(x, scale, w12, a, M, I, K, eps, grouped, 0, (hipStream_t)stream);
}

// Parts of K where the batch rows would be read more often than the weights, 64 weight rows a workgroup and no more workgroups than CUs (each takes a CU's LDS: a second
// round of a few costs as much as the first).  0: one sum.  us at 33 / 64 rows, one sum (up to 8,192 columns) or one part more (3,072) -> this: 3,072 x 4,096 14.6 / 17.0 ->
// 10.9 / 12.7, 4,160 x 8,192 28.7 / 29.9 -> 17.7 / 20.9, 5,120 x 11,008 37.1 / 39.9 -> 24.7 / 27.7, 6,912 x 4,096 16.6 / 17.6 -> 14.8 / 17.7, x 8,192 29.2 / 31.1 -> 23.3 / 28.0,
// 8,192 x 8,192 29.6 / 31.5 -> 25.6 / 29.3, but x 4,096 16.4 / 17.7 -> 15.9 / 18.4, x 2,048 10.3 / 11.4 -> 11.2 / 13.4.  At 17 / 32 rows two parts are not ahead: 5,120 x 11,008 27.6 / 29.6 -> 23.6 / 24.4 in
// three, 6,912 x 11,008 29.2 / 31.6 -> 32.3 / 33.4 in two.
static int small_m_parts(int64_t M, int64_t N, int64_t K) {
    if (M < 17 || M > 64 || N > 8192 || N < 1024 || N % 64 != 0 || K < 1024 || K % 128 != 0 || K > 0x9fffff || (K < 8192 && M <= 32) || (N > 4096 && K < (N <= 7168 ? 4096 : 8192))) return 0;
    int64_t parts = 256 / (N / 64);
    if (N > 4096 && M <= 32 && parts < 3) return 0;
    if (parts > K / 256) parts = K / 256;
    if (parts > 8) parts = 8;
    return parts >= 2 ? (int)parts : 0;
}
extern "C" int evo_linear_parts(int64_t M, int64_t N, int64_t K) { return small_m_parts(M, N, K); }
extern "C" int evo_linear_parts_bf16(const void* x, const void* w, float* ws, int64_t M, int64_t N, int64_t K, int64_t parts, void* stream) {
    if (!x || !w || !ws || parts < 2 || parts != small_m_parts(M, N, K) || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)ws) & 15)) return -1;
    return ring_launch<2>(x, w, nullptr, nullptr, nullptr, M, N, K, 0, 0, ws, (int)parts, (hipStream_t)stream);
}

extern "C" int evo_linear_small_m_bf16(const void* x, const void* w, const void* bias, const void* residual, void* y,
                                       int64_t M, int64_t N, int64_t K, void* ws, int64_t ws_bytes, int64_t act, void* stream) {
    if (M < 1 || M > 64 || N <= 0 || K <= 0 || K % 8 != 0 || N > 0x7fffffff - 16) return -1;
    if ((M > 8 && K % 32 != 0) || (act != 0 && act != 3)) return -1;
    hipStream_t s = (hipStream_t)stream;
    // Three and four rows take the matrix cores' forms too where those are ahead of the dot2 form below (us at 4 rows: 4,096 x 4,096 9.5 -> 7.9, K = 11,008 19.7 -> 16.1,
    // 16,384 x 4,096 26.2 -> 22.1; at 2 rows 8.0, 17.2 and 24.3 against the same).  Layers of 4,097 to 16,383 columns stay: the fused Hyena step of up to four rows sums its
    // 12,288 columns in the dot2 form's order, and agrees with the unfused one bit for bit.
    if ((M >= 5 || (M >= 3 && K % 128 == 0 && (N <= 4096 ? N >= 2048 && K >= 2048 : N >= 16384))) && K % 32 == 0) {
        // (asynchronous loads of 16 bytes; an offset of 96 rows, 64 batch rows or 16 weight rows in 32 bits)
        if (K % 128 == 0 && (((uintptr_t)x | (uintptr_t)w) & 15) == 0 && K <= 0x9fffff) {
            const int64_t parts = ws && ((uintptr_t)ws & 15) == 0 ? small_m_parts(M, N, K) : 0;
            if (parts && ws_bytes >= parts * M * N * 4) {
                const int rc = ring_launch<2>(x, w, nullptr, nullptr, nullptr, M, N, K, 0, 0, (float*)ws, (int)parts, s);
                if (rc) return rc;
                hipLaunchKernelGGL(skinny_reduce_kernel, dim3((unsigned)((M * N / 4 + 255) / 256)), dim3(256), 0, s, (const float*)ws, (const uint16_t*)bias,
                                   (const uint16_t*)residual, (uint16_t*)y, (int)M, (int)N, (int)parts, (int)act);
                return evo_launch_status();
            }
            // wide layers
            if (N > 4096) return ring_launch<0>(x, w, bias, residual, y, M, N, K, (int)act, 0, nullptr, 0, s);
            // (few workgroups, the unembedding's 512 columns: more waves in each -- us at 8 / 16 / 32 rows, K = 4,096: 6.0 / 6.8 / 8.4, with four 6.1 / 6.9 / 8.8)
            if (N < 2048) {
                if (M <= 8) return kw_launch<8, 8, 128, 2>(x, w, bias, residual, y, M, N, K, (int)act, s);
                if (M <= 16) return kw_launch<16, 8, 128, 2>(x, w, bias, residual, y, M, N, K, (int)act, s);
                if (M <= 32) return kw_launch<32, 4, 128, 2>(x, w, bias, residual, y, M, N, K, (int)act, s);
            }
            if (M <= 8) return kw_launch<8, 4, 128, 3>(x, w, bias, residual, y, M, N, K, (int)act, s);
            if (M <= 16) return kw_launch<16, 4, 128, 2>(x, w, bias, residual, y, M, N, K, (int)act, s);
            if (M <= 32 && K <= 1024) return kw_launch<32, 4, 128, 2>(x, w, bias, residual, y, M, N, K, (int)act, s);     // (a chunk or two a wave: 3.6 -> 3.3 us at 512)
            if (M <= 32) return kw_launch<32, 3, 128, 2>(x, w, bias, residual, y, M, N, K, (int)act, s);
        }
        // what is left (K not in whole chunks): two n tiles per workgroup (every x fragment feeds two weight fragments) where that still leaves a workgroup or more per CU
        const dim3 block(512);
#define EVO_SK(MT, NT)                                                                                                     \
        hipLaunchKernelGGL((skinny_mfma_kernel<MT, NT>), dim3((unsigned)((N + 16 * NT - 1) / (16 * NT))), block, 0, s, (const uint4*)x, (const uint4*)w, \
                           (const uint16_t*)bias, (const uint16_t*)residual, (uint16_t*)y, (int)M, (int)N, (int)(K / 8), (int)act)
        if (N >= 8192 && M > 16) { if (M <= 32) EVO_SK(2, 2); else if (M <= 48) EVO_SK(3, 2); else EVO_SK(4, 2); }
        else { if (M <= 16) EVO_SK(1, 1); else if (M <= 32) EVO_SK(2, 1); else if (M <= 48) EVO_SK(3, 1); else EVO_SK(4, 1); }
#undef EVO_SK
        return evo_launch_status();
    }
    switch (M) {
        case 1: gemv_launch<1>(x, w, bias, residual, y, N, K, (int)act, s); break;
        case 2: gemv_launch<2>(x, w, bias, residual, y, N, K, (int)act, s); break;
        case 3: gemv_launch<3>(x, w, bias, residual, y, N, K, (int)act, s); break;
        case 4: gemv_launch<4>(x, w, bias, residual, y, N, K, (int)act, s); break;
        case 5: gemv_launch<5>(x, w, bias, residual, y, N, K, (int)act, s); break;
        case 6: gemv_launch<6>(x, w, bias, residual, y, N, K, (int)act, s); break;
        case 7: gemv_launch<7>(x, w, bias, residual, y, N, K, (int)act, s); break;
        default: gemv_launch<8>(x, w, bias, residual, y, N, K, (int)act, s); break;
    }
    return evo_launch_status();
}

// ---- a norm between two layers without a launch, 5 to 32 rows (skinny_kw_kernel EP 3, skinny_ring_kernel RS)
extern "C" int evo_linear_residual_scaled_bf16(const void* x, const void* w, const void* bias, void* y, const void* scale, void* xg, float* ss, int64_t M, int64_t N, int64_t K,
                                               void* stream) {
    if (!x || !w || !y || !scale || !xg || !ss || M < 5 || M > 32 || N < 2048 || N > 4096 || N % 64 != 0 || K < 1152 || K % 128 != 0 || K > 0x9fffff || small_m_parts(M, N, K)) return -1;
    if ((((uintptr_t)x | (uintptr_t)w | (uintptr_t)ss) & 15) || (((uintptr_t)bias | (uintptr_t)y | (uintptr_t)scale | (uintptr_t)xg) & 7)) return -1;
    hipStream_t s = (hipStream_t)stream;
    if (M <= 8) return kw_go<8, 4, 128, 3, 3>(x, w, bias, y, y, M, N, K, 0, s, scale, xg, ss);
    if (M <= 16) return kw_go<16, 4, 128, 2, 3>(x, w, bias, y, y, M, N, K, 0, s, scale, xg, ss);
    return kw_go<32, 3, 128, 2, 3>(x, w, bias, y, y, M, N, K, 0, s, scale, xg, ss);
}

static bool factors_ok(const void* xg, const float* ss, const void* w, int64_t M, int64_t N, int64_t K) {
    return xg && ss && w && M >= 5 && M <= 32 && N > 4096 && N <= 24576 && K >= 2048 && K <= 4096 && K % 128 == 0 && (((uintptr_t)xg | (uintptr_t)ss | (uintptr_t)w) & 15) == 0;
}

extern "C" int evo_linear_factors_bf16(const void* xg, const float* ss, float eps, const void* w, const void* bias, void* y, int64_t M, int64_t N, int64_t K, void* stream) {
    if (!factors_ok(xg, ss, w, M, N, K) || !y) return -1;
    return ring_factors<0>(xg, w, bias, y, M, N, K, 0, {ss, (int)(K / 16), eps, 1.0f / sqrtf((float)K)}, (hipStream_t)stream);
}

extern "C" int evo_mlp_gate_factors_bf16(const void* xg, const float* ss, float eps, const void* w12, void* a, int64_t M, int64_t I, int64_t K, int64_t grouped, void* stream) {
    if (I <= 0 || I > 0x3fffffff || I % 32 != 0 || !factors_ok(xg, ss, w12, M, 2 * I, K) || !a) return -1;
    return ring_factors<1>(xg, w12, nullptr, a, M, 2 * I, K, grouped ? 1 : 2, {ss, (int)(K / 16), eps, 1.0f / sqrtf((float)K)}, (hipStream_t)stream);
}
