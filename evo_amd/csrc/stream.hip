// Token-local kernels of models whose residual stream is kept in fp32: scaled embedding, the norm of a sublayer's output added to the
// stream, the norm of their sum, the final norm, the gated norm behind a linear-attention mixer, the gate of a gated MLP.  One workgroup per row, fp32 math,
// one rounding on the way out; storage type T is bf16 or fp32.  Entry points: include/evo_mi355x.h.
#include "mixers_common.h"
#include "../../include/evo_mi355x.h"

#define STREAM_DISPATCH(KERNEL, VECOK, GRID, ...)                                                                          \
    do {                                                                                                                   \
        const dim3 g_(GRID), b_(256);                                                                                      \
        hipStream_t s_ = (hipStream_t)stream;                                                                              \
        if (f32) {                                                                                                         \
            if (VECOK) hipLaunchKernelGGL((KERNEL<float, 8>), g_, b_, 0, s_, __VA_ARGS__);                                 \
            else hipLaunchKernelGGL((KERNEL<float, 1>), g_, b_, 0, s_, __VA_ARGS__);                                       \
        } else {                                                                                                           \
            if (VECOK) hipLaunchKernelGGL((KERNEL<uint16_t, 8>), g_, b_, 0, s_, __VA_ARGS__);                              \
            else hipLaunchKernelGGL((KERNEL<uint16_t, 1>), g_, b_, 0, s_, __VA_ARGS__);                                    \
        }                                                                                                                  \
        return evo_launch_status();                                                                                        \
    } while (0)

// The same for kernels of one workgroup a row: rows of whole runs of eight a thread (2,048, 4,096 and 8,192 elements) have forms without a condition, for sizes where these are
// ahead (AHEAD)
#define ROW_DISPATCH(KERNEL, VECOK, AHEAD, D_, GRID, ...)                                                                   \
    do {                                                                                                                   \
        const dim3 g_(GRID), b_(256);                                                                                      \
        hipStream_t s_ = (hipStream_t)stream;                                                                              \
        const int runs_ = !(VECOK) ? -1 : !(AHEAD) ? 0 : (D_) == 2048 ? 1 : (D_) == 4096 ? 2 : (D_) == 8192 ? 4 : 0;       \
        if (f32) { ROW_LAUNCH(KERNEL, float, __VA_ARGS__); } else { ROW_LAUNCH(KERNEL, uint16_t, __VA_ARGS__); }           \
        return evo_launch_status();                                                                                        \
    } while (0)
#define ROW_LAUNCH(KERNEL, T, ...)                                                                                         \
    switch (runs_) {                                                                                                       \
        case 1: hipLaunchKernelGGL((KERNEL<T, 8, 1>), g_, b_, 0, s_, __VA_ARGS__); break;                                  \
        case 2: hipLaunchKernelGGL((KERNEL<T, 8, 2>), g_, b_, 0, s_, __VA_ARGS__); break;                                  \
        case 4: hipLaunchKernelGGL((KERNEL<T, 8, 4>), g_, b_, 0, s_, __VA_ARGS__); break;                                  \
        case 0: hipLaunchKernelGGL((KERNEL<T, 8, 0>), g_, b_, 0, s_, __VA_ARGS__); break;                                  \
        default: hipLaunchKernelGGL((KERNEL<T, 1, 0>), g_, b_, 0, s_, __VA_ARGS__);                                        \
    }

// ---------------------------------------------------------------------------------------------- embedding
// x = scale * w[id]; an id outside the table gives a zero row and raises *bad_flag
template <typename T, int V>
__global__ __launch_bounds__(256) void embed_stream_kernel(const int64_t* __restrict__ ids, const void* __restrict__ w_, float* __restrict__ x,
                                                           uint16_t* __restrict__ xb, int D, int64_t vocab, float scale, int* __restrict__ bad_flag) {
    const T* w = (const T*)w_;
    const int64_t row = blockIdx.x;
    const int64_t id = ids[row];
    const bool ok = id >= 0 && id < vocab;
    if (!ok && bad_flag && threadIdx.x == 0) *bad_flag = 1;
    for (int c = threadIdx.x * V; c < D; c += 256 * V) {
        float f[V];
        if (ok) vec_io<T, V>::load(w + id * D + c, f);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = ok ? f[e] * scale : 0.f;
        vec_io<float, V>::store(x + row * D + c, f);
        if (xb) vec_io<uint16_t, V>::store(xb + row * D + c, f);
    }
}

extern "C" int evo_embed_stream(const int64_t* ids, const void* w, float* x, void* xb, int64_t n_tok, int64_t D, int64_t vocab, float scale,
                                int* bad_flag, int64_t f32, void* stream) {
    if (n_tok < 0 || n_tok > 0x7fffffff || D <= 0 || D > 0x7fffffff || vocab <= 0) return -1;
    if (n_tok == 0) return 0;
    STREAM_DISPATCH(embed_stream_kernel, D % 8 == 0, (unsigned)n_tok, ids, w, x, (uint16_t*)xb, (int)D, vocab, scale, bad_flag);
}

// ---------------------------------------------------------------------------------------------- x += norm(y) * (off + w)
// SUM: x = norm(alpha x + y) * (off + w); `y` below is then the sum.
// y stays in registers between the two passes (rows up to 4,096 elements); x is written in fp32 and, for the next sublayer's matrix
// product, once more in bf16.
// PARTS: y is the sum of `parts` fp32 planes [gridDim.x, D] one behind the other, added in their order and rounded to bf16 (what evo_linear_small_m_bf16 stores).
//
// RUNS > 0: the row is exactly RUNS runs of V elements a thread.  Everything a row needs -- y or its parts four at a time, x, the norm's weight -- is then requested
// together, without a condition among the requests.  A decode step's launch is a chain of latencies: with the weight (cold: a whole step's weights went by since) and x
// asked for behind the reduction there were two of them: rows of 4,096 in a step of four layers 3.5 -> 2.8 us at 8 rows, on the parts of 24 rows 5.2 -> 3.8, the gated norm
// 3.9 -> 2.4 (an empty launch is 1.6).
template <typename T, int V, bool PARTS>
__device__ __forceinline__ void closing_load(const void* __restrict__ row, int c, int D, int parts, float* f) {
    if constexpr (PARTS) {
        const float* p = (const float*)row + c;
        const int64_t plane = (int64_t)gridDim.x * D;
        vec_io<float, V>::load(p, f);
        for (int s = 1; s < parts; s += 3) {                     // (three requests at once; a plane behind the last is the last again, and not added)
            float q[3][V];
#pragma unroll
            for (int k = 0; k < 3; ++k) vec_io<float, V>::load(p + (s + k < parts ? s + k : parts - 1) * plane, q[k]);
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int e = 0; e < V; ++e) f[e] = s + k < parts ? f[e] + q[k][e] : f[e];
        }
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = bf_to_f(f_to_bf(f[e]));
    } else vec_io<T, V>::load((const T*)row + c, f);
}

template <typename T, int V, bool SUM, bool PARTS, int RUNS>
__device__ __forceinline__ void closing_row(const void* __restrict__ y_, const void* __restrict__ w_, const float* __restrict__ x, int D, float alpha, float eps, float off,
                                            int parts, float* red, float (&r)[RUNS][V]) {   // -> the row's new x in r
    const T* w = (const T*)w_;
    const int64_t row = blockIdx.x;
    float f[RUNS][V], g[RUNS][V];
#pragma unroll
    for (int i = 0; i < RUNS; ++i) {
        const int c = (threadIdx.x + 256 * i) * V;
        vec_io<float, V>::load(x + row * D + c, r[i]);
        vec_io<T, V>::load(w + c, g[i]);
    }
#pragma unroll
    for (int i = 0; i < RUNS; ++i) closing_load<T, V, PARTS>(PARTS ? (const void*)((const float*)y_ + row * D) : (const void*)((const T*)y_ + row * D), (threadIdx.x + 256 * i) * V, D, parts, f[i]);
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
#pragma unroll
        for (int e = 0; e < V; ++e) {
            if (SUM) f[i][e] = fmaf(alpha, r[i][e], f[i][e]);
            ss = fmaf(f[i][e], f[i][e], ss);
        }
    const float inv = 1.0f / sqrtf(block_sum_256(ss, red) / (float)D + eps);
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
#pragma unroll
        for (int e = 0; e < V; ++e) r[i][e] = SUM ? f[i][e] * inv * (off + g[i][e]) : fmaf(f[i][e] * inv, off + g[i][e], r[i][e]);
}

template <typename T, int V, bool SUM, bool PARTS = false, int RUNS = 0>
__device__ __forceinline__ void closing_norm(const void* __restrict__ y_, const void* __restrict__ w_, float* __restrict__ x,
                                             uint16_t* __restrict__ xb, int D, float alpha, float eps, float off, int parts = 0) {
    __shared__ float red[4];
    const int64_t row = blockIdx.x;
    if constexpr (RUNS > 0) {
        float r[RUNS][V];
        closing_row<T, V, SUM, PARTS, RUNS>(y_, w_, x, D, alpha, eps, off, parts, red, r);
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
            const int c = (threadIdx.x + 256 * i) * V;
            vec_io<float, V>::store(x + row * D + c, r[i]);
            if (xb) vec_io<uint16_t, V>::store(xb + row * D + c, r[i]);
        }
        return;
    }
    constexpr int KEEP = V == 8 ? 2 : 4;                         // runs of V elements a thread keeps in registers (D <= 256 V KEEP)
    const T* w = (const T*)w_;
    const void* y = PARTS ? (const void*)((const float*)y_ + row * D) : (const void*)((const T*)y_ + row * D);
    float keep[KEEP][V];
    float ss = 0.f;
    auto load = [&](int c, float* f) {
        closing_load<T, V, PARTS>(y, c, D, parts, f);
        if constexpr (SUM) {
            float r[V];
            vec_io<float, V>::load(x + row * D + c, r);
#pragma unroll
            for (int e = 0; e < V; ++e) f[e] = fmaf(alpha, r[e], f[e]);
        }
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int c = (threadIdx.x + 256 * i) * V;
        if (c < D) {
            load(c, keep[i]);
#pragma unroll
            for (int e = 0; e < V; ++e) ss = fmaf(keep[i][e], keep[i][e], ss);
        }
    }
    for (int c = (threadIdx.x + 256 * KEEP) * V; c < D; c += 256 * V) {
        float f[V];
        load(c, f);
#pragma unroll
        for (int e = 0; e < V; ++e) ss = fmaf(f[e], f[e], ss);
    }
    const float inv = 1.0f / sqrtf(block_sum_256(ss, red) / (float)D + eps);
    auto finish = [&](int c, const float* f) {
        float g[V], r[V];
        vec_io<T, V>::load(w + c, g);
        if constexpr (!SUM) vec_io<float, V>::load(x + row * D + c, r);
#pragma unroll
        for (int e = 0; e < V; ++e) r[e] = SUM ? f[e] * inv * (off + g[e]) : fmaf(f[e] * inv, off + g[e], r[e]);
        vec_io<float, V>::store(x + row * D + c, r);
        if (xb) vec_io<uint16_t, V>::store(xb + row * D + c, r);
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int c = (threadIdx.x + 256 * i) * V;
        if (c < D) finish(c, keep[i]);
    }
    for (int c = (threadIdx.x + 256 * KEEP) * V; c < D; c += 256 * V) {
        float f[V];
        load(c, f);
        finish(c, f);
    }
}

template <typename T, int V, int RUNS>
__global__ __launch_bounds__(256) void postnorm_residual_kernel(const void* __restrict__ y, const void* __restrict__ w, float* __restrict__ x,
                                                                uint16_t* __restrict__ xb, int D, float eps, float off) {
    closing_norm<T, V, false, false, RUNS>(y, w, x, xb, D, 1.f, eps, off);
}
template <typename T, int V, int RUNS>
__global__ __launch_bounds__(256) void sum_norm_kernel(const void* __restrict__ y, const void* __restrict__ w, float* __restrict__ x,
                                                       uint16_t* __restrict__ xb, int D, float alpha, float eps, float off) {
    closing_norm<T, V, true, false, RUNS>(y, w, x, xb, D, alpha, eps, off);
}

extern "C" int evo_postnorm_residual(const void* y, const void* w, float* x, void* xb, int64_t M, int64_t D, float eps, float w_offset,
                                     int64_t f32, void* stream) {
    if (M < 0 || M > 0x7fffffff || D <= 0 || D > 0x3fffffff) return -1;
    if (M == 0) return 0;
    // (8,192 columns, the loop : the row at once, us, rows that the last-level cache holds: bf16 200 rows 1.0 x, 300 7.8 : 8.2, 400 8.7 : 9.3, 513 10.7 : 11.6, 700 13.1 : 13.8, 1,000 18.1 : 18.8;
    // fp32 300 7.6 : 8.3, 513 10.2 : 11.5, 1,000 18.9 : 19.6, 1,500 and more 1.0 x; cold rows at once are ahead at 300 and 400, 11.6 : 9.7)
    ROW_DISPATCH(postnorm_residual_kernel, D % 8 == 0, D != 8192 || M <= 256 || M > 1024, D, (unsigned)M, y, w, x, (uint16_t*)xb, (int)D, eps, w_offset);
}

extern "C" int evo_sum_norm(const void* y, const void* w, float* x, void* xb, int64_t M, int64_t D, float alpha, float eps, float w_offset,
                            int64_t f32, void* stream) {
    if (!y || !w || !x || M < 0 || M > 0x7fffffff || D <= 0 || D > 0x3fffffff) return -1;
    if (M == 0) return 0;
    // (8,192 columns, the loop : the row at once, us: 256 rows 9.1 : 8.0, 400 10.9 : 10.6, 512 12.1 : 12.4, 600 14.2 : 15.6, 768 16.9 : 17.3, 1,000 22.1 : 21.9, 2,048 49 : 41)
    ROW_DISPATCH(sum_norm_kernel, D % 8 == 0, D != 8192 || M <= 400 || M > 900, D, (unsigned)M, y, w, x, (uint16_t*)xb, (int)D, alpha, eps, w_offset);
}

// Both on the parts of a dense layer's sum (evo_linear_parts_bf16, evo_dense_parts_bf16): the launch that added and rounded them was 4.7 us of its own, a decode layer of 17 to 64
// rows.  Rows at once of 4,096 elements alone: of the other widths that layers come in parts with (Stream.product: up to 4,096 columns) only 2,048 is whole runs, and there it is ahead
// of the loop up to 300 rows (four parts, us: 24 rows 3.3 : 2.8, 256 5.4 : 5.0, 512 7.4 : 7.4, 660 9.1 : 9.4, 1,000 12.3 : 12.1): 0.4 us that steps of such
// models could still gain.
template <bool SUM, int RUNS>
__global__ __launch_bounds__(256) void closing_parts_kernel(const float* __restrict__ y, const void* __restrict__ w, float* __restrict__ x, uint16_t* __restrict__ xb, int D,
                                                            float alpha, float eps, float off, int parts) {
    closing_norm<uint16_t, 8, SUM, true, RUNS>(y, w, x, xb, D, alpha, eps, off, parts);
}

extern "C" int evo_closing_parts(const float* y, int64_t parts, const void* w, float* x, void* xb, int64_t M, int64_t D, int64_t sum, float alpha, float eps, float w_offset,
                                 void* stream) {
    if (!y || !w || !x || !xb || parts < 1 || parts > 64 || M < 0 || M > 0x7fffffff || D <= 0 || D > 0x3fffffff || D % 8 != 0) return -1;
    if (((uintptr_t)y | (uintptr_t)w | (uintptr_t)x | (uintptr_t)xb) & 15) return -1;
    if (M == 0) return 0;
#define CP(SUM, RUNS) hipLaunchKernelGGL((closing_parts_kernel<SUM, RUNS>), dim3((unsigned)M), dim3(256), 0, (hipStream_t)stream, y, w, x, (uint16_t*)xb, (int)D,   \
                                         sum ? alpha : 1.f, eps, w_offset, (int)parts)
    if (D == 4096) { if (sum) CP(true, 2); else CP(false, 2); }
    else if (sum) CP(true, 0); else CP(false, 0);
#undef CP
    return evo_launch_status();
}

// ---------------------------------------------------------------------------------------------- out = norm(x) * (off + w), x the stream
// RUNS: as in closing_norm
template <typename T, int V, int RUNS>
__global__ __launch_bounds__(256) void rmsnorm_stream_kernel(const float* __restrict__ x_, const void* __restrict__ w_, void* __restrict__ out_, int D,
                                                             float eps, float off) {
    __shared__ float red[4];
    const T* w = (const T*)w_;
    const int64_t row = blockIdx.x;
    const float* x = x_ + row * D;
    T* out = (T*)out_ + row * D;
    float ss = 0.f;
    if constexpr (RUNS > 0) {
        float f[RUNS][V], g[RUNS][V];
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
            const int c = (threadIdx.x + 256 * i) * V;
            vec_io<float, V>::load(x + c, f[i]);
            vec_io<T, V>::load(w + c, g[i]);
        }
#pragma unroll
        for (int i = 0; i < RUNS; ++i)
#pragma unroll
            for (int e = 0; e < V; ++e) ss = fmaf(f[i][e], f[i][e], ss);
        const float inv = 1.0f / sqrtf(block_sum_256(ss, red) / (float)D + eps);
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
#pragma unroll
            for (int e = 0; e < V; ++e) f[i][e] = f[i][e] * inv * (off + g[i][e]);
            vec_io<T, V>::store(out + (threadIdx.x + 256 * i) * V, f[i]);
        }
        return;
    }
    for (int c = threadIdx.x * V; c < D; c += 256 * V) {
        float f[V];
        vec_io<float, V>::load(x + c, f);
#pragma unroll
        for (int e = 0; e < V; ++e) ss = fmaf(f[e], f[e], ss);
    }
    const float inv = 1.0f / sqrtf(block_sum_256(ss, red) / (float)D + eps);
    for (int c = threadIdx.x * V; c < D; c += 256 * V) {
        float f[V], g[V];
        vec_io<float, V>::load(x + c, f);
        vec_io<T, V>::load(w + c, g);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = f[e] * inv * (off + g[e]);
        vec_io<T, V>::store(out + c, f);
    }
}

extern "C" int evo_rmsnorm_stream(const float* x, const void* w, void* out, int64_t M, int64_t D, float eps, float w_offset, int64_t f32,
                                  void* stream) {
    if (M < 0 || M > 0x7fffffff || D <= 0 || D > 0x3fffffff) return -1;
    if (M == 0) return 0;
    ROW_DISPATCH(rmsnorm_stream_kernel, D % 8 == 0, true, D, (unsigned)M, x, w, out, (int)D, eps, w_offset);
}

// ---------------------------------------------------------------------------------------------- the last closing norm and the final one
// out = norm(x') * (off + wf) of the x' that a closing norm makes, which nothing reads any more: neither it nor its copy is stored.  The same bits as the two launches.  Parts:
// rows of 4,096 elements, the ones that closing_parts_kernel takes at once.
template <typename T, bool SUM, bool PARTS, int RUNS>
__global__ __launch_bounds__(256) void closing_final_kernel(const void* __restrict__ y, const void* __restrict__ w, const float* __restrict__ x, const void* __restrict__ wf_,
                                                            void* __restrict__ out_, int D, float alpha, float eps, float off, int parts) {
    constexpr int V = 8;
    __shared__ float red[4], red2[4];
    const T* wf = (const T*)wf_;
    T* out = (T*)out_ + (int64_t)blockIdx.x * D;
    float g[RUNS][V], r[RUNS][V], ss = 0.f;
#pragma unroll
    for (int i = 0; i < RUNS; ++i) vec_io<T, V>::load(wf + (threadIdx.x + 256 * i) * V, g[i]);
    closing_row<T, V, SUM, PARTS, RUNS>(y, w, x, D, alpha, eps, off, parts, red, r);
#pragma unroll
    for (int i = 0; i < RUNS; ++i)
#pragma unroll
        for (int e = 0; e < V; ++e) ss = fmaf(r[i][e], r[i][e], ss);
    const float inv = 1.0f / sqrtf(block_sum_256(ss, red2) / (float)D + eps);
#pragma unroll
    for (int i = 0; i < RUNS; ++i) {
#pragma unroll
        for (int e = 0; e < V; ++e) r[i][e] = r[i][e] * inv * (off + g[i][e]);
        vec_io<T, V>::store(out + (threadIdx.x + 256 * i) * V, r[i]);
    }
}

extern "C" int evo_closing_final(const void* y, int64_t parts, const void* w, const float* x, const void* wf, void* out, int64_t M, int64_t D, int64_t sum, float alpha, float eps,
                                 float w_offset, int64_t f32, void* stream) {
    if (!y || !w || !x || !wf || !out || parts < 0 || parts > 64 || M < 0 || M > 0x7fffffff || (D != 2048 && D != 4096 && D != 8192)) return -1;
    if (parts && (f32 || D != 4096)) return -1;
    if (((uintptr_t)y | (uintptr_t)w | (uintptr_t)x | (uintptr_t)wf | (uintptr_t)out) & 15) return -1;
    if (M == 0) return 0;
#define CF(T, SUM, PARTS, RUNS) hipLaunchKernelGGL((closing_final_kernel<T, SUM, PARTS, RUNS>), dim3((unsigned)M), dim3(256), 0, (hipStream_t)stream, y, w, x, wf, out, (int)D, \
                                                   alpha, eps, w_offset, (int)parts)
#define CF_RUNS(T, SUM) do { if (D == 2048) CF(T, SUM, false, 1); else if (D == 4096) CF(T, SUM, false, 2); else CF(T, SUM, false, 4); } while (0)
    if (parts) { if (sum) CF(uint16_t, true, true, 2); else CF(uint16_t, false, true, 2); }
    else if (f32) { if (sum) CF_RUNS(float, true); else CF_RUNS(float, false); }
    else if (sum) CF_RUNS(uint16_t, true); else CF_RUNS(uint16_t, false);
#undef CF_RUNS
#undef CF
    return evo_launch_status();
}

// ---------------------------------------------------------------------------------------------- out = norm(o) * w * sigmoid(g)
// RUNS: as in closing_norm
template <typename T, int V, int RUNS>
__global__ __launch_bounds__(256) void gated_norm_kernel(const void* __restrict__ o_, const void* __restrict__ g_, int64_t ldg,
                                                         const void* __restrict__ w_, void* __restrict__ out_, int D, float eps) {
    constexpr int KEEP = V == 8 ? 2 : 4;
    __shared__ float red[4];
    const T* w = (const T*)w_;
    const int64_t row = blockIdx.x;
    const T* o = (const T*)o_ + row * D;
    const T* g = (const T*)g_ + row * ldg;
    T* out = (T*)out_ + row * D;
    if constexpr (RUNS > 0) {
        float f[RUNS][V], gg[RUNS][V], ww[RUNS][V], ss = 0.f;
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
            const int c = (threadIdx.x + 256 * i) * V;
            vec_io<T, V>::load(o + c, f[i]);
            vec_io<T, V>::load(g + c, gg[i]);
            vec_io<T, V>::load(w + c, ww[i]);
        }
#pragma unroll
        for (int i = 0; i < RUNS; ++i)
#pragma unroll
            for (int e = 0; e < V; ++e) ss = fmaf(f[i][e], f[i][e], ss);
        const float inv = 1.0f / sqrtf(block_sum_256(ss, red) / (float)D + eps);
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
#pragma unroll
            for (int e = 0; e < V; ++e) f[i][e] = f[i][e] * inv * ww[i][e] * sigmoid_t<T>(gg[i][e]);
            vec_io<T, V>::store(out + (threadIdx.x + 256 * i) * V, f[i]);
        }
        return;
    }
    float keep[KEEP][V];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int c = (threadIdx.x + 256 * i) * V;
        if (c < D) {
            vec_io<T, V>::load(o + c, keep[i]);
#pragma unroll
            for (int e = 0; e < V; ++e) ss = fmaf(keep[i][e], keep[i][e], ss);
        }
    }
    for (int c = (threadIdx.x + 256 * KEEP) * V; c < D; c += 256 * V) {
        float f[V];
        vec_io<T, V>::load(o + c, f);
#pragma unroll
        for (int e = 0; e < V; ++e) ss = fmaf(f[e], f[e], ss);
    }
    const float inv = 1.0f / sqrtf(block_sum_256(ss, red) / (float)D + eps);
    auto finish = [&](int c, const float* f) {
        float gg[V], ww[V], r[V];
        vec_io<T, V>::load(g + c, gg);
        vec_io<T, V>::load(w + c, ww);
#pragma unroll
        for (int e = 0; e < V; ++e) r[e] = f[e] * inv * ww[e] * sigmoid_t<T>(gg[e]);
        vec_io<T, V>::store(out + c, r);
    };
#pragma unroll
    for (int i = 0; i < KEEP; ++i) {
        const int c = (threadIdx.x + 256 * i) * V;
        if (c < D) finish(c, keep[i]);
    }
    for (int c = (threadIdx.x + 256 * KEEP) * V; c < D; c += 256 * V) {
        float f[V];
        vec_io<T, V>::load(o + c, f);
        finish(c, f);
    }
}

extern "C" int evo_gated_norm(const void* o, const void* g, int64_t ldg, const void* w, void* out, int64_t M, int64_t D, float eps, int64_t f32,
                              void* stream) {
    if (M < 0 || M > 0x7fffffff || D <= 0 || D > 0x3fffffff || ldg < D) return -1;
    if (M == 0) return 0;
    const bool vec = D % 8 == 0 && ldg % 8 == 0 && ((uintptr_t)g & 15) == 0;
    // (bf16, the loop : the row at once, us.  2,048 columns: 512 rows 3.3 : 3.3, 600 3.4 : 3.6, 1,536 5.0 : 5.5, 4,096 11.2 : 11.6, 8,190 19.5 : 19.1; 4,096 columns: 400 rows
    // 4.1 : 3.8, 1,000 6.0 : 6.1, 2,048 10.0 : 11.0, 4,096 19.1 : 19.0, 8,190 36.2 : 33.0; 8,192 and fp32 0.95 to 1.3)
    ROW_DISPATCH(gated_norm_kernel, vec, f32 || D == 8192 || M <= 512 || M > 4096, D, (unsigned)M, o, g, ldg, w, out, (int)D, eps);
}

// ---------------------------------------------------------------------------------------------- a = silu(z[:, :I]) * z[:, I:]
template <typename T, int V>
__global__ __launch_bounds__(256) void silu_gate_kernel(const void* __restrict__ z_, void* __restrict__ a_, int64_t M, int64_t I) {
    const T* z = (const T*)z_;
    T* a = (T*)a_;
    const int64_t per = I / V, total = M * per;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / per, c = (i - row * per) * V;
        float u[V], v[V];
        vec_io<T, V>::load(z + row * 2 * I + c, u);
        vec_io<T, V>::load(z + row * 2 * I + I + c, v);
#pragma unroll
        for (int e = 0; e < V; ++e) u[e] = silu_t<T>(u[e]) * v[e];
        vec_io<T, V>::store(a + row * I + c, u);
    }
}

extern "C" int evo_silu_gate(const void* z, void* a, int64_t M, int64_t I, int64_t f32, void* stream) {
    if (M < 0 || I <= 0) return -1;
    if (M == 0) return 0;
    const int64_t total = M * (I % 8 == 0 ? I / 8 : I);
    const unsigned grid = (unsigned)((total + 255) / 256 < 16384 ? (total + 255) / 256 : 16384);
    STREAM_DISPATCH(silu_gate_kernel, I % 8 == 0, grid, z, a, M, I);
}

// ---------------------------------------------------------------------------------------------- z[:, :n] = act(z[:, :n]) in place
template <typename T, int V>
__global__ __launch_bounds__(256) void act_cols_kernel(void* __restrict__ z_, int64_t ld, int64_t M, int64_t n, int act) {
    T* z = (T*)z_;
    const int64_t per = n / V, total = M * per;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / per;
        T* p = z + row * ld + (i - row * per) * V;
        float f[V];
        vec_io<T, V>::load(p, f);
#pragma unroll
        for (int e = 0; e < V; ++e) f[e] = act_t<T>(f[e], act);
        vec_io<T, V>::store(p, f);
    }
}

extern "C" int evo_act_cols(void* z, int64_t ld, int64_t M, int64_t n, int64_t act, int64_t f32, void* stream) {
    if (M < 0 || n <= 0 || ld < n || act < 1 || act > 3) return -1;
    if (M == 0) return 0;
    const bool vec = n % 8 == 0 && ld % 8 == 0 && ((uintptr_t)z & 15) == 0;
    const int64_t total = M * (vec ? n / 8 : n);
    const unsigned grid = (unsigned)((total + 255) / 256 < 16384 ? (total + 255) / 256 : 16384);
    STREAM_DISPATCH(act_cols_kernel, vec, grid, z, ld, M, n, (int)act);
}
