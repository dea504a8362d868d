// fp32 values as three bf16 ones each, and outputs that have to be taken again: what gemm_f32.hip and gemm_f32_ahead.hip share.
#pragma once
#include "common.h"
#define F3_BK 32

// what a layer is estimated to take on gemm_f32.hip's tiles, us
double f3_tiles_us(int64_t M, int64_t N, int64_t K);

__device__ __forceinline__ void f3_split(const float4 a, const float4 b, uint4& h, uint4& m, uint4& l) {
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t o[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        o[0][e] = pack_bf2(v[2 * e], v[2 * e + 1]);
        float r0 = v[2 * e] - bf_lo(o[0][e]), r1 = v[2 * e + 1] - bf_hi(o[0][e]);
        o[1][e] = pack_bf2(r0, r1);
        r0 -= bf_lo(o[1][e]);
        r1 -= bf_hi(o[1][e]);
        o[2][e] = pack_bf2(r0, r1);
    }
    h = make_uint4(o[0][0], o[0][1], o[0][2], o[0][3]);
    m = make_uint4(o[1][0], o[1][1], o[1][2], o[1][3]);
    l = make_uint4(o[2][0], o[2][1], o[2][2], o[2][3]);
}

// Outputs taken again with the fp32 matrix instructions, by the wave that holds them.  An infinite operand has no parts (inf - inf), one near the largest value
// rounds to an infinite h, and the bf16 instructions take parts and sums under 2^-126 as zero: an operand loses at most 2^-124, an output of K products at
// most K 2^-124 (|x| + |w| + 2), |x| and |w| the largest of its rows.  What is not finite or under 2^26 of that is taken again; a row without a value other
// than zero is right as it is.  A wave takes a few one after the other, many as a product of its whole part.  (300 x 4,096 x 4,096, 88 us: with a NaN in one
// row 118, in all rows 224 -- 2,400 and 16,450 output by output --; the maxima and the look at the outputs cost 1 %.)
__device__ __forceinline__ void f3_row_max(float& m, const float4 a, const float4 b) {
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a.x), "v"(a.y));
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(a.z), "v"(a.w));
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(b.x), "v"(b.y));
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(m) : "v"(b.z), "v"(b.w));
}
// the least and the largest magnitude so far (the largest is NaN once a value was)
__device__ __forceinline__ void f3_range(float& lo, float& hi, float a, float b) {
    asm("v_min3_f32 %0, %0, |%1|, |%2|" : "+v"(lo) : "v"(a), "v"(b));
    asm("v_maximum3_f32 %0, %0, |%1|, |%2|" : "+v"(hi) : "v"(a), "v"(b));
}

// The end of a wave's part, TM x TN products of 32 x 32 whose sums `acc` are stored: rows from m0 (of M) and columns from n0 (of N), k-steps k0 .. k1 of 32.
// x_max, w_max: the largest magnitude of each of these rows of x and of w (-inf: zeros only), in LDS; `look`: an output of this lane may have to be taken again.
template <int TM, int TN, class At>
__device__ __forceinline__ void f3_again(f32x16_t (&acc)[TM][TN], bool look, const float* x_, const float* w_, const float* bias, int64_t m0, int64_t M, int n0, int N, int K, int k0, int k1,
                                         const float* x_max, const float* w_max, At at) {
    const int lane = threadIdx.x & 63, half = lane >> 5, l31 = lane & 31;
    const float least = (float)(k1 - k0) * (F3_BK * 0x1p-98f);
    if (__builtin_amdgcn_ballot_w64(look) == 0) return;
    uint32_t odd[(TM * TN + 1) / 2] = {};                      // which ones: 16 outputs of each of two products
    int n_odd = 0;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int r = i * 32 + l31;
        if (m0 + r >= M) continue;
        const float bound = fmaf(least, x_max[r], least);
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int c = j * 32 + q * 8 + half * 4;
                if (n0 + c >= N) continue;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float u = fabsf(acc[i][j][4 * q + e]);
                    odd[(i * TN + j) >> 1] |= (u >= fmaf(least, w_max[c + e], bound) && u <= 3.402823466e38f ? 0u : 1u) << (((i * TN + j) & 1) * 16 + 4 * q + e);
                }
            }
    }
#pragma unroll
    for (uint32_t w : odd) n_odd += __popc(w);
#pragma unroll
    for (int d = 1; d < 64; d *= 2) n_odd += __shfl_xor(n_odd, d, 64);
    if (n_odd == 0) return;
    if (n_odd <= 8 * TM * TN) {                                // a few (sums that cancel to zero): one after the other, the wave along k
#pragma unroll
        for (int s = 0; s < (TM * TN + 1) / 2; ++s)
            for (uint64_t lanes = __builtin_amdgcn_ballot_w64(odd[s] != 0); lanes; lanes &= lanes - 1) {
                const int owner = __builtin_ctzll(lanes);
                for (uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)odd[s], owner); bits; bits &= bits - 1) {
                    const int t = __builtin_ctz(bits), ij = 2 * s + (t >> 4), i = ij / TN, j = ij - i * TN;
                    const int64_t m = m0 + i * 32 + (owner & 31);
                    const int n = n0 + j * 32 + ((t >> 2) & 3) * 8 + (owner >> 5) * 4 + (t & 3);
                    const float *x = x_ + m * K, *w = w_ + (int64_t)n * K;
                    float sum = 0.f;
#pragma unroll 4
                    for (int k = k0 * F3_BK + 4 * lane; k < k1 * F3_BK; k += 256) {
                        const f32x4_t u = *(const f32x4_t*)(x + k), v = *(const f32x4_t*)(w + k);
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum = fmaf(u[e], v[e], sum);
                    }
                    sum = wave_sum(sum);
                    if (lane == owner) *at(m, n) = bias ? sum + bias[n] : sum;
                }
            }
        return;
    }
    // lane (l31, half): four neighbouring k of its rows per request, a product of two k per component, as both operands take them
    const float *xr[TM], *wr[TN];
#pragma unroll
    for (int i = 0; i < TM; ++i) {
        const int64_t m = m0 + i * 32 + l31;
        xr[i] = x_ + (m < M ? m : M - 1) * K + (int64_t)k0 * F3_BK + half * 4;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int n = n0 + j * 32 + l31;
        wr[j] = w_ + (int64_t)(n < N ? n : N - 1) * K + (int64_t)k0 * F3_BK + half * 4;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll 1
    for (int k = k0; k < k1; ++k) {
        f32x4_t xf[TM][4], wf[TN][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
            for (int i = 0; i < TM; ++i) xf[i][t] = *(const f32x4_t*)(xr[i] + 8 * t);
#pragma unroll
            for (int j = 0; j < TN; ++j) wf[j][t] = *(const f32x4_t*)(wr[j] + 8 * t);
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < TM; ++i)
#pragma unroll
                    for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[j][t][e], xf[i][t][e], acc[i][j], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < TM; ++i) xr[i] += F3_BK;
#pragma unroll
        for (int j = 0; j < TN; ++j) wr[j] += F3_BK;
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int t = 0; t < 16; ++t)
                if (odd[(i * TN + j) >> 1] >> (((i * TN + j) & 1) * 16 + t) & 1) {     // (set only for outputs that are there)
                    const int n = n0 + j * 32 + (t >> 2) * 8 + half * 4 + (t & 3);
                    *at(m0 + i * 32 + l31, n) = bias ? acc[i][j][t] + bias[n] : acc[i][j][t];
                }
}
