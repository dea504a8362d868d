// Linear attention with one constant decay per head:  S_t = a_h S_{t-1} + k_t v_t^T,  o_t = S_t^T q_t,  S [dk, dv] fp32 per sequence and head.
// q, k, v are the columns of one projection row z = [q (H dk) | k (H dk) | v (H dv) | ...] after their SiLU (the recurrent form can apply it);
// sequences are packed (cu = first row of each, B + 1 entries).
//
// Prompt form (bf16): chunks of 64 tokens on the matrix cores.  With A = a_h, inside a chunk starting from S
//     o_i = A^{i+1} S^T q_i + sum_{j <= i} A^{i-j} (q_i . k_j) v_j          S' = A^n S + sum_j A^{n-1-j} k_j v_j^T
// q, k, v are exact bf16 operands; the fp32 factors (S, the decayed scores, the decayed v) enter the products as bf16 hi + lo pairs,
// 2^-17 relative, so state and scores keep their fp32 meaning.  A workgroup owns one (sequence, head, segment, DV value columns); a wave owns
// 16 of the columns, so the state lives in the accumulators: S is accumulated as [k rows, v columns], which IS the layout of the S^T operand
// of the next product under the split k order of frag_split -- it never passes through LDS.  The decayed scores are shared: every wave
// computes a block or two of them, their hi and lo halves go through the LDS rows of k (done with by then).
// Long sequences are cut into segments that run in parallel: (1) every segment's end state from zero, (2) a scan over segments, (3) outputs.  Sequences of one segment
// in the same launch take (3) alone, straight on their state, and no workspace.
#include "mixers_common.h"
#include "../../include/evo_mi355x.h"

#define LC 64                                                    // tokens per chunk

struct LightArgs {
    const void* z; void* o; float* state; const float* log2_decay; const int* cu; const int* resume;
    float* seg;                                                  // [slot][H][dk][dv] or null: states per segment, at segment_slot
    int64_t ld;
    int H, dk, dv, n_seg, seg_len, act;                          // act: z still needs its SiLU (recurrent form)
};

// ------------------------------------------------------------------------------------------------ chunked form
template <int DK, int DV, bool OUT, bool VEC>
__global__ __launch_bounds__(4 * DV, 2) void lightning_chunk_kernel(LightArgs a) {
    constexpr int NW = DV / 16, NT = 64 * NW;                    // waves (16 value columns each), threads
    constexpr int NKB = DK / 16, NKK = DK / 32, PR = DK + 8, PT = LC + 4, KR = PR > 2 * PT ? PR : 2 * PT;   // 16-row blocks of S; LDS pitches of rows and columns
    constexpr int KG = (DK + 63) / 64, VG = DV / 64, GS = NT / 256;   // groups of 64 key / value columns; groups staged at a time
    constexpr int KI = (KG + GS - 1) / GS, VI = (VG + GS - 1) / GS;   // groups per thread
    __shared__ __attribute__((aligned(16))) uint16_t q_rows[OUT ? LC * PR : 8], k_rows[OUT ? LC * KR : 8], k_cols[DK * PT], v_cols[DV * PT];
    uint16_t* const p_hi = k_rows;                               // [64 queries][PT] each: the decayed scores, over k's rows (KR: room for either)
    uint16_t* const p_lo = k_rows + LC * PT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    // (heads first: workgroup i runs on XCD i % 8, and a short sequence's later segments are empty -- segments first, five sequences of 3,000 and 300 tokens in
    //  segments of 384 had all of their short ones on one XCD: 204 -> 102 us)
    const int h = blockIdx.x % a.H, seg = blockIdx.x / a.H % a.n_seg, vt = blockIdx.x / a.H / a.n_seg, b = blockIdx.z;
    const int dk = a.dk, dv = a.dv, v0 = vt * DV;
    const int row0 = a.cu[b] + seg * a.seg_len;
    int len = a.cu[b + 1] - row0;
    len = len < a.seg_len ? len : a.seg_len;
    if (len <= 0 && (seg > 0 || len < 0)) return;
    const bool cut = a.seg && a.cu[b + 1] - a.cu[b] > a.seg_len;
    if (!OUT && !cut) return;
    const float l2 = a.log2_decay[h];
    const uint16_t* zq = (const uint16_t*)a.z + row0 * a.ld + (int64_t)h * dk;
    const uint16_t* zk = zq + (int64_t)a.H * dk;
    const uint16_t* zv = (const uint16_t*)a.z + row0 * a.ld + (int64_t)2 * a.H * dk + (int64_t)h * dv + v0;
    const int dvt = dv - v0 < DV ? dv - v0 : DV;                 // value columns of this workgroup
    // powers of the decay by exponents a lane needs in every chunk: queries i = 16 ib + c16, keys j = 16 jb + 4 g + r
    float p_diag[4], p_off[4], p_end[4];                         // a^(c16 - 4 g - r) (0 above the diagonal), a^(16 - 4 g - r), a^(15 - 4 g - r)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int j = 4 * g + r;
        p_diag[r] = c16 < j ? 0.f : pow_log2(l2, c16 - j);
        p_off[r] = pow_log2(l2, 16 - j);
        p_end[r] = pow_log2(l2, 15 - j);
    }
    const float p_q = pow_log2(l2, c16), p_1 = pow_log2(l2, 1), p_16 = pow_log2(l2, 16), p_32 = pow_log2(l2, 32), p_64 = pow_log2(l2, LC);
    const int col = 16 * wave + c16;                             // this lane's value column as an operand row / accumulator column

    f32x4_t S[NKB];
    const int64_t st_off = ((int64_t)b * a.H + h) * dk * dv;
    {
        const float* src = nullptr;
        if (OUT && cut && (seg > 0 || a.resume)) src = a.seg + (segment_slot(a.cu, b, seg, a.seg_len) * a.H + h) * dk * dv;
        else if (OUT && a.resume && a.resume[b]) src = a.state + st_off;
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = 16 * kb + 4 * g + r;
                S[kb][r] = src && k < dk && col < dvt ? src[(int64_t)k * dv + v0 + col] : 0.f;
            }
    }

    // eight threads share a row: thread (tokens 2 p2 and 2 p2 + 1, columns ct + 64 i of its groups i)
    const int p2 = (tid >> 3) & 31, ct = (tid & 7) * 8, g0 = tid >> 8;
    mx_u32x4 rq[KI][2], rk[KI][2], rv[VI][2];
    auto fetch = [&](const uint16_t* p, int c, int width) -> mx_u32x4 {
        if (VEC) return *(const mx_u32x4*)(p + c);
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = c + e < width ? p[c + e] : 0u;
        return mx_u32x4{w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16, w[6] | w[7] << 16};
    };
    // (tokens past the end repeat the last one and columns past the head's repeat its last eight: such keys carry no weight -- a decay factor
    //  of zero, scores of queries that are not stored --, such columns meet zeros in q; so the aligned form has no branch among its requests)
    uint32_t q_keep[KI];
#pragma unroll
    for (int i = 0; i < KI; ++i) q_keep[i] = ct + 64 * (g0 + GS * i) < dk ? 0xffffffffu : 0u;
    auto load = [&](int t0, int n) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int64_t off = (int64_t)(t0 + (2 * p2 + u < n ? 2 * p2 + u : n - 1)) * a.ld;
#pragma unroll
            for (int i = 0; i < KI; ++i) {
                const int c = ct + 64 * (g0 + GS * i), cc = !VEC || c < dk ? c : dk - 8;
                rk[i][u] = fetch(zk + off, cc, dk);
                if (OUT) rq[i][u] = fetch(zq + off, cc, dk);
            }
#pragma unroll
            for (int i = 0; i < VI; ++i) {
                const int c = ct + 64 * (g0 + GS * i);
                rv[i][u] = fetch(zv + off, !VEC || c < dvt ? c : dvt - 8, dvt);
            }
        }
    };
    auto put_cols = [&](uint16_t* dst, int c, mx_u32x4 x, mx_u32x4 y) __attribute__((always_inline)) {   // this token pair's columns c .. c + 7
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            *(uint32_t*)(dst + (c + 2 * e) * PT + 2 * p2) = (x[e] & 0xffffu) | y[e] << 16;
            *(uint32_t*)(dst + (c + 2 * e + 1) * PT + 2 * p2) = x[e] >> 16 | (y[e] & 0xffff0000u);
        }
    };
    auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < KI; ++i) {
            const int c = ct + 64 * (g0 + GS * i);
            if (c < DK) {
                put_cols(k_cols, c, rk[i][0], rk[i][1]);
                if (OUT) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        *(mx_u32x4*)(k_rows + (2 * p2 + u) * PR + c) = rk[i][u];
                        *(mx_u32x4*)(q_rows + (2 * p2 + u) * PR + c) = rq[i][u] & q_keep[i];
                    }
                }
            }
        }
#pragma unroll
        for (int i = 0; i < VI; ++i)
            if (g0 + GS * i < VG) put_cols(v_cols, ct + 64 * (g0 + GS * i), rv[i][0], rv[i][1]);
    };

    const int n_chunk = (len + LC - 1) / LC;
    if (n_chunk > 0) load(0, len);
    for (int ch = 0; ch < n_chunk; ++ch) {
        const int t0 = ch * LC, n = len - t0 < LC ? len - t0 : LC;
        stage();
        __syncthreads();
        if (ch + 1 < n_chunk) load(t0 + LC, len - t0 - LC);
        const uint16_t* vbase = v_cols + col * PT + 4 * g;
        if (OUT) {
            // ---- decayed scores: twelve 16 x 16 blocks (ib, jb), jb <= ib, and the two zero blocks the 32-wide sum below reads, shared out
            constexpr int NB = (12 + NW - 1) / NW;
            uint32_t hi[NB][2], lo[NB][2];
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const int x = wave + NW * t;                     // block x: rows 0 and 1 have two blocks each, rows 2 and 3 four
                const int ib = x < 4 ? x >> 1 : (x - 4 < 4 ? 2 : 3), jb = x < 4 ? x & 1 : (x - 4) & 3, back = ib - jb;
                f32x4_t p = {0.f, 0.f, 0.f, 0.f};
                if (x < 12 && back >= 0) {
#pragma unroll
                    for (int kk = 0; kk < NKK; ++kk)
                        p = mfma16(frag_split(k_rows + (16 * jb + c16) * PR + 32 * kk + 4 * g), frag_split(q_rows + (16 * ib + c16) * PR + 32 * kk + 4 * g), p);
                    // a^(i - j): on the diagonal from the table, else a^c16 a^(16 - 4 g - r) a^(16 (back - 1))
                    const float f = p_q * (back <= 1 ? 1.f : back == 2 ? p_16 : p_32);
#pragma unroll
                    for (int r = 0; r < 4; ++r) p[r] *= back == 0 ? p_diag[r] : f * p_off[r];
                }
                split_hi_lo(p[0], p[1], hi[t][0], lo[t][0]);
                split_hi_lo(p[2], p[3], hi[t][1], lo[t][1]);
                __builtin_amdgcn_sched_barrier(0);
            }
            mx_frag s_hi[NKK], s_lo[NKK];                        // S^T as an operand: row = value column, k order of frag_split
#pragma unroll
            for (int kk = 0; kk < NKK; ++kk) {
                uint32_t x[4], y[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) split_hi_lo(S[2 * kk + (q >> 1)][2 * (q & 1)], S[2 * kk + (q >> 1)][2 * (q & 1) + 1], x[q], y[q]);
                s_hi[kk] = frag_of(x[0], x[1], x[2], x[3]);
                s_lo[kk] = frag_of(y[0], y[1], y[2], y[3]);
            }
            __syncthreads();                                     // (every wave is done with k's rows)
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const int x = wave + NW * t;
                const int ib = x < 4 ? x >> 1 : (x - 4 < 4 ? 2 : 3), jb = x < 4 ? x & 1 : (x - 4) & 3;
                if (x < 12) {
                    *(uint2*)(p_hi + (16 * ib + c16) * PT + 16 * jb + 4 * g) = make_uint2(hi[t][0], hi[t][1]);
                    *(uint2*)(p_lo + (16 * ib + c16) * PT + 16 * jb + 4 * g) = make_uint2(lo[t][0], lo[t][1]);
                }
            }
            __syncthreads();
#pragma unroll
            for (int ip = 0; ip < 2; ++ip) {                     // queries 32 ip .. 32 ip + 31: two 16-blocks side by side
                if (32 * ip >= n) break;
                f32x4_t o[2], o2[2];
#pragma unroll
                for (int u = 0; u < 2; ++u) o[u] = o2[u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int kk = 0; kk < NKK; ++kk) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const mx_frag qf = frag_split(q_rows + (32 * ip + 16 * u + c16) * PR + 32 * kk + 4 * g);
                        o[u] = mfma16(s_hi[kk], qf, o[u]);
                        o2[u] = mfma16(s_lo[kk], qf, o2[u]);
                    }
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const float ai = p_q * p_1 * (ip ? (u ? p_16 * p_32 : p_32) : (u ? p_16 : 1.f));   // a^(i + 1)
#pragma unroll
                    for (int r = 0; r < 4; ++r) { o[u][r] = (o[u][r] + o2[u][r]) * ai; o2[u][r] = 0.f; }
                }
#pragma unroll
                for (int jj = 0; jj <= ip; ++jj) {
                    const mx_frag vf = frag_split(vbase + 32 * jj);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int at = (32 * ip + 16 * u + c16) * PT + 32 * jj + 4 * g;
                        o[u] = mfma16(vf, frag_split(p_hi + at), o[u]);
                        o2[u] = mfma16(vf, frag_split(p_lo + at), o2[u]);
                    }
                }
                const int d = 16 * wave + 4 * g;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int i = 32 * ip + 16 * u + c16;
                    if (i < n) {
                        uint16_t* op = (uint16_t*)a.o + (int64_t)(row0 + t0 + i) * a.H * dv + (int64_t)h * dv + v0 + d;
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[u][r] += o2[u][r];
                        if (d + 3 < dvt && (dv & 3) == 0) *(uint2*)op = make_uint2(pack_bf2(o[u][0], o[u][1]), pack_bf2(o[u][2], o[u][3]));
                        else {
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (d + r < dvt) op[r] = f_to_bf(o[u][r]);
                        }
                    }
                }
            }
        }
        // ---- S <- a^n S + K^T (decayed V)
        const float an = n == LC ? p_64 : pow_log2(l2, n);
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[kb][r] *= an;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            if (32 * jj >= n) break;
            float fac[8];                                        // a^(n - 1 - j)
            if (n == LC) {
                const float f = jj ? 1.f : p_32;
#pragma unroll
                for (int e = 0; e < 8; ++e) fac[e] = p_end[e & 3] * (e < 4 ? f * p_16 : f);
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int m = n - 1 - (32 * jj + 16 * (e >> 2) + 4 * g + (e & 3));
                    fac[e] = m < 0 ? 0.f : pow_log2(l2, m);
                }
            }
            const uint2 x = *(const uint2*)(vbase + 32 * jj), y = *(const uint2*)(vbase + 32 * jj + 16);
            const uint32_t w[4] = {x.x, x.y, y.x, y.y};
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) split_hi_lo(bf_lo(w[q]) * fac[2 * q], bf_hi(w[q]) * fac[2 * q + 1], hi[q], lo[q]);
            const mx_frag v_hi = frag_of(hi[0], hi[1], hi[2], hi[3]), v_lo = frag_of(lo[0], lo[1], lo[2], lo[3]);
#pragma unroll
            for (int kb = 0; kb < NKB; ++kb) {
                const mx_frag kf = frag_split(k_cols + (16 * kb + c16) * PT + 32 * jj + 4 * g);
                S[kb] = mfma16(kf, v_hi, S[kb]);
                S[kb] = mfma16(kf, v_lo, S[kb]);
                if (kb & 1) __builtin_amdgcn_sched_barrier(0);   // (bounds the fragments read ahead: 128 registers a lane)
            }
        }
        __syncthreads();
    }
    float* dst = nullptr;                                        // end state: of the segment (state-only walk), or of the sequence
    if (!OUT) dst = a.seg + (segment_slot(a.cu, b, seg, a.seg_len) * a.H + h) * dk * dv;
    else if (a.state && !cut) dst = a.state + st_off;
    if (dst) {
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int k = 16 * kb + 4 * g + r;
                if (k < dk && col < dvt) dst[(int64_t)k * dv + v0 + col] = S[kb][r];
            }
    }
}

// a sequence's slots: segment s <- the state BEFORE it (it held the segment's own end state from zero); state[b] <- the state after the last token
__global__ __launch_bounds__(256) void lightning_scan_kernel(LightArgs a) {
    const int h = blockIdx.y, b = blockIdx.z;
    const int64_t per = (int64_t)a.dk * a.dv, e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= per) return;
    const float l2 = a.log2_decay[h];
    const int len = a.cu[b + 1] - a.cu[b];
    if (len <= a.seg_len) return;
    const int64_t so = ((int64_t)b * a.H + h) * per + e;
    float s = a.resume && a.resume[b] ? a.state[so] : 0.f;
    for (int i = 0; i < a.n_seg; ++i) {
        int n = len - i * a.seg_len;
        if (n <= 0) break;
        n = n < a.seg_len ? n : a.seg_len;
        float* p = a.seg + (segment_slot(a.cu, b, i, a.seg_len) * a.H + h) * per + e;
        const float own = *p;
        *p = s;
        s = s * pow_log2(l2, n) + own;
    }
    if (a.state) a.state[so] = s;
}

template <int DK, int DV, bool VEC>
static void chunk_launch(LightArgs a, int64_t B, hipStream_t s) {
    const dim3 grid((unsigned)(a.H * a.n_seg * ((a.dv + DV - 1) / DV)), 1, (unsigned)B), block(4 * DV);
    if (a.n_seg > 1) {
        hipLaunchKernelGGL((lightning_chunk_kernel<DK, DV, false, VEC>), grid, block, 0, s, a);
        hipLaunchKernelGGL(lightning_scan_kernel, dim3((unsigned)((a.dk * a.dv + 255) / 256), (unsigned)a.H, (unsigned)B), dim3(256), 0, s, a);
    }
    hipLaunchKernelGGL((lightning_chunk_kernel<DK, DV, true, VEC>), grid, block, 0, s, a);
}

extern "C" int evo_lightning_chunk_bf16(const void* z, int64_t ld, void* o, float* state, float* seg, const float* log2_decay, const int* cu,
                                        const int* resume, int64_t B, int64_t H, int64_t dk, int64_t dv, int64_t max_len, int64_t seg_len,
                                        void* stream) {
    if (!z || !o || !log2_decay || !cu || B <= 0 || B > 65535 || H <= 0 || H > 65535 || dk <= 0 || dk > 128 || dv <= 0 || dv > 65536) return -1;
    if (max_len <= 0 || max_len > 0x7fffffff || seg_len <= 0 || seg_len % LC != 0 || ld < H * (2 * dk + dv) || (resume && !state)) return -1;
    LightArgs a = {z, o, state, log2_decay, cu, resume, seg, ld, (int)H, (int)dk, (int)dv, (int)((max_len + seg_len - 1) / seg_len), (int)seg_len, 0};
    if (a.n_seg > 1 && !seg) return -1;
    if (H * a.n_seg * ((dv + 63) / 64) > 0x7fffffff) return -1;
    if (a.n_seg == 1) a.seg = nullptr;
    hipStream_t s = (hipStream_t)stream;
    const bool vec = dk % 8 == 0 && dv % 8 == 0 && ld % 8 == 0 && ((uintptr_t)z & 15) == 0;
    if (!vec) { if (dk <= 32 && dv <= 64) chunk_launch<32, 64, false>(a, B, s); else chunk_launch<128, 128, false>(a, B, s); }
    else if (dk <= 32) { if (dv <= 64) chunk_launch<32, 64, true>(a, B, s); else chunk_launch<32, 128, true>(a, B, s); }
    else if (dk <= 64) { if (dv <= 64) chunk_launch<64, 64, true>(a, B, s); else chunk_launch<64, 128, true>(a, B, s); }
    else { if (dv <= 64) chunk_launch<128, 64, true>(a, B, s); else chunk_launch<128, 128, true>(a, B, s); }
    return evo_launch_status();
}

// ------------------------------------------------------------------------------------------------ recurrent form
// Token by token, any sizes, both storage types: one workgroup per (sequence, head, 8 CW value columns).  Thread (column lane cl, slice):
// columns cl CW .. + CW - 1, rows slice, slice + 32, ... of the state.  The decode step: one token per sequence straight on the state in memory
// (read and written once, 16 bytes per request).
template <typename T, int CW>
__global__ __launch_bounds__(256) void lightning_recur_kernel(LightArgs a, const float* __restrict__ decay) {
    extern __shared__ float sm[];
    const int dk = a.dk, dv = a.dv, h = blockIdx.y, b = blockIdx.z;
    float* qs = sm;                                              // [dk], [dk], [32], [32 slices][8 CW + 1]
    float* ks = qs + dk;
    float* vs = ks + dk;
    float* part = vs + 32;
    const int tid = threadIdx.x, cl = tid & 7, sl = tid >> 3;
    const int c0 = blockIdx.x * 8 * CW, cols = dv - c0 < 8 * CW ? dv - c0 : 8 * CW;
    const float A = decay[h];
    float* st = a.state + ((int64_t)b * a.H + h) * dk * dv + c0;
    const T* z = (const T*)a.z + (int64_t)b * a.ld;
    for (int k = tid; k < 2 * dk; k += 256) {
        const float x = ld1(z + (k < dk ? 0 : (int64_t)(a.H - 1) * dk) + (int64_t)h * dk + k);
        qs[k] = a.act ? silu_t<T>(x) : x;
    }
    if (tid < 8 * CW) {
        const float x = tid < cols ? ld1(z + (int64_t)2 * a.H * dk + (int64_t)h * dv + c0 + tid) : 0.f;
        vs[tid] = a.act ? silu_t<T>(x) : x;
    }
    __syncthreads();
    float v[CW], o[CW];
#pragma unroll
    for (int e = 0; e < CW; ++e) { v[e] = vs[cl * CW + e]; o[e] = 0.f; }
    if (cl * CW < cols) {
#pragma unroll 4
        for (int k = sl; k < dk; k += 32) {
            float s[CW];
            float* p = st + (int64_t)k * dv + cl * CW;
            if constexpr (CW == 4) { const float4 x = *(const float4*)p; s[0] = x.x; s[1] = x.y; s[2] = x.z; s[3] = x.w; }
            else s[0] = *p;
#pragma unroll
            for (int e = 0; e < CW; ++e) {
                s[e] = fmaf(A, s[e], ks[k] * v[e]);
                o[e] = fmaf(qs[k], s[e], o[e]);
            }
            if constexpr (CW == 4) *(float4*)p = make_float4(s[0], s[1], s[2], s[3]);
            else *p = s[0];
        }
    }
#pragma unroll
    for (int e = 0; e < CW; ++e) part[sl * 33 + cl * CW + e] = o[e];
    __syncthreads();
    if (tid < cols) {
        float s = 0.f;
#pragma unroll 8
        for (int i = 0; i < 32; ++i) s += part[i * 33 + tid];
        st1((T*)a.o + (int64_t)b * a.H * dv + (int64_t)h * dv + c0 + tid, s);
    }
}

// Prompts the same way, LT tokens between barriers: their q, k, v rows are staged together (the next LT's are in flight meanwhile), the slices' shares of
// LT rows of o meet in LDS at the end of the block, summed in the order of the slices.  (fp32 heads of 64 or 128 rows: lightning_f32_kernel.)  R: the state rows of a thread, in registers (dk <= 32 R); 0: in LDS.
// Bound by issue and latency: 70 instructions a token and wave in sequence.  (3 prompts of up to 500 tokens, 32 heads of 128 x 128, fp32, MI355X: 288 us;
// one token between barriers, its rows requested when they were needed and the state in LDS, 685 us.)
// The state in LDS is read and written in 16-byte requests (200 tokens, 4 heads of 512 x 64, fp32: 367 us; element by element 573, the form before 471).
template <typename T, int CW, int R, int LT>
__global__ __launch_bounds__(256) void lightning_tokens_kernel(LightArgs a, const float* __restrict__ decay) {
    extern __shared__ float sm[];
    const int dk = a.dk, dv = a.dv, h = blockIdx.y, b = blockIdx.z;
    float2* kq = (float2*)sm;                                    // [LT][dk] (k, q), [LT][32], [LT][32 slices][33], with R == 0 the state [dk][8 CW]
    float* vs = sm + (CW == 4 ? (2 * LT * dk + 3) & ~3 : 2 * LT * dk);         // (rows of the state below are 16-byte requests then)
    float* part = vs + LT * 32;
    float* tile = part + LT * 32 * 33;
    const int tid = threadIdx.x, cl = tid & 7, sl = tid >> 3;
    const int c0 = blockIdx.x * 8 * CW, cols = dv - c0 < 8 * CW ? dv - c0 : 8 * CW;
    const bool mine = cl * CW < cols;
    const float A = decay[h];
    const int row0 = a.cu[b], n = a.cu[b + 1] - row0;
    float* st = a.state ? a.state + ((int64_t)b * a.H + h) * dk * dv + c0 : nullptr;
    const bool keep = st && a.resume && a.resume[b];
    float S[R ? R : 1][CW];
    if constexpr (R > 0) {
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int e = 0; e < CW; ++e) S[r][e] = keep && mine && sl + 32 * r < dk ? st[(int64_t)(sl + 32 * r) * dv + cl * CW + e] : 0.f;
    } else {
        for (int k = sl; k < dk; k += 32)
#pragma unroll
            for (int e = 0; e < CW; ++e) tile[k * 8 * CW + cl * CW + e] = keep && mine ? st[(int64_t)k * dv + cl * CW + e] : 0.f;
    }
    const T* zr = (const T*)a.z + (int64_t)row0 * a.ld;
    const int64_t hk = (int64_t)h * dk, hv = (int64_t)2 * a.H * dk + (int64_t)h * dv + c0;
    constexpr int RK = R ? R : 1;                                // staged values of k and of q per thread (R == 0: staged without a request ahead)
    float zk[RK], zq[RK], zv;
    // thread (token tid / SW, elements tid % SW + SW j) of a block's k and q; of its v
    constexpr int SW = 256 / LT;
    const int tt = tid / SW, te = tid % SW;
    auto request = [&](int t0) {
        const T* z = zr + (int64_t)(t0 + tt < n ? t0 + tt : n - 1) * a.ld;
        if constexpr (R > 0) {
#pragma unroll
            for (int j = 0; j < RK; ++j) {
                const int k = te + SW * j < dk ? te + SW * j : dk - 1;
                zk[j] = ld1(z + (int64_t)a.H * dk + hk + k);
                zq[j] = ld1(z + hk + k);
            }
        }
        zv = te < cols ? ld1(z + hv + te) : 0.f;
    };
    auto act = [&](float x) { return a.act ? silu_t<T>(x) : x; };
    if (n > 0) request(0);
    for (int t0 = 0; t0 < n; t0 += LT) {
        const int nb = n - t0 < LT ? n - t0 : LT;
        if constexpr (R > 0) {
#pragma unroll
            for (int j = 0; j < RK; ++j)
                if (te + SW * j < dk) kq[tt * dk + te + SW * j] = make_float2(act(zk[j]), act(zq[j]));
        } else if (tt < nb) {
            const T* z = zr + (int64_t)(t0 + tt) * a.ld;
            for (int k = te; k < dk; k += SW) kq[tt * dk + k] = make_float2(act(ld1(z + (int64_t)a.H * dk + hk + k)), act(ld1(z + hk + k)));
        }
        if (te < 32) vs[tt * 32 + te] = act(zv);
        __syncthreads();
        if (t0 + LT < n) request(t0 + LT);
        auto token = [&](int t) __attribute__((always_inline)) {
            float v[CW], o[CW];
            if constexpr (CW == 4 && R > 0) { const float4 x = *(const float4*)(vs + t * 32 + cl * 4); v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w; }
            else {
#pragma unroll
                for (int e = 0; e < CW; ++e) v[e] = vs[t * 32 + cl * CW + e];
            }
#pragma unroll
            for (int e = 0; e < CW; ++e) o[e] = 0.f;
            if constexpr (R > 0) {
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (sl + 32 * r < dk) {
                        const float2 x = kq[t * dk + sl + 32 * r];
#pragma unroll
                        for (int e = 0; e < CW; ++e) {
                            S[r][e] = fmaf(A, S[r][e], x.x * v[e]);
                            o[e] = fmaf(x.y, S[r][e], o[e]);
                        }
                    }
            } else if (mine) {
#pragma unroll 4
                for (int k = sl; k < dk; k += 32) {
                    float* p = tile + k * 8 * CW + cl * CW;
                    const float2 x = kq[t * dk + k];
                    float s[CW];
                    if constexpr (CW == 4) { const float4 y = *(const float4*)p; s[0] = y.x; s[1] = y.y; s[2] = y.z; s[3] = y.w; }
                    else s[0] = *p;
#pragma unroll
                    for (int e = 0; e < CW; ++e) {
                        s[e] = fmaf(A, s[e], x.x * v[e]);
                        o[e] = fmaf(x.y, s[e], o[e]);
                    }
                    if constexpr (CW == 4) *(float4*)p = make_float4(s[0], s[1], s[2], s[3]);
                    else *p = s[0];
                }
            }
#pragma unroll
            for (int e = 0; e < CW; ++e) part[(t * 32 + sl) * 33 + cl * CW + e] = o[e];
        };
        if (nb == LT) {
#pragma unroll
            for (int t = 0; t < LT; ++t) token(t);
        } else {
            for (int t = 0; t < nb; ++t) token(t);
        }
        __syncthreads();
        if (tt < nb && te < cols) {
            float s = 0.f;
#pragma unroll 8
            for (int i = 0; i < 32; ++i) s += part[(tt * 32 + i) * 33 + te];
            st1((T*)a.o + (int64_t)(row0 + t0 + tt) * a.H * dv + (int64_t)h * dv + c0 + te, s);
        }
        // (the next block's staging touches kq / vs only, which every thread has finished reading at the barrier above; its `part`
        //  stores come behind the next barrier, and so behind the sums of this block)
    }
    if (st && mine) {
        if constexpr (R > 0) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (sl + 32 * r < dk)
#pragma unroll
                    for (int e = 0; e < CW; ++e) st[(int64_t)(sl + 32 * r) * dv + cl * CW + e] = S[r][e];
        } else {
            for (int k = sl; k < dk; k += 32)
#pragma unroll
                for (int e = 0; e < CW; ++e) st[(int64_t)k * dv + cl * CW + e] = tile[k * 8 * CW + cl * CW + e];
        }
    }
}

// fp32 prompts of heads of 64 or 128 rows, 32 tokens at a time on v_mfma_f32_16x16x4_f32: with A the decay, inside a chunk that starts from S
//     o_i = A^{i+1} S^T q_i + sum_{j <= i} A^{i-j} (q_i . k_j) v_j          S' = A^n S + sum_j A^{n-1-j} k_j v_j^T
// in fp32 throughout; the powers are rounded once, from fp64.  A workgroup owns 32 value columns of one head and sequence; S stays in the accumulators (wave w: rows
// 16 RT w on) and goes through LDS transposed, so that every operand but k's in the state's sum is read as four consecutive values.  Latency bounds it: three barriers
// a chunk, 104 matrix instructions a wave between them.  The next chunk's rows are requested behind the first barrier.
// 32 heads of 128 x 128, eight tokens between barriers on the vector units (lightning_tokens_kernel) -> this: prompts of 500, 325 and 325 tokens 237 -> 86 us, one of
// 150 77 -> 24, of 2,000 950 -> 250, of 4 9 -> 9; against 64 bits 3.0e-7 -> 1.5e-7 (outputs) and 3.6e-7 -> 1.4e-7 (states) of the first.
// A product with a masked score is 0 v_j: where v is not finite that would reach the tokens before j, and the chunk's sum is taken term by term.
typedef float lf_f32x4 __attribute__((ext_vector_type(4)));
template <int RT>
__global__ __launch_bounds__(256) void lightning_f32_kernel(LightArgs a, const float* __restrict__ decay) {
    constexpr int C = 32, DK = 64 * RT, PQ = DK + 4, PT = C + 4, QN = DK / 32;        // pitches; float4 of q and of k a thread stages
    __shared__ __attribute__((aligned(16))) float q[C * PQ], k[C * PQ], s[32 * PQ], vt[32 * PT], p[C * PT];     // s, vt: [column][..]
    __shared__ float pw[C + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, g = lane >> 4;
    const int h = blockIdx.x, b = blockIdx.z, dv = a.dv, c0 = blockIdx.y * 32, cols = dv - c0 < 32 ? dv - c0 : 32;
    const int row0 = a.cu[b], n = a.cu[b + 1] - row0;
    if (tid <= C) pw[tid] = tid ? (float)pow((double)decay[h], (double)tid) : 1.f;
    float* st = a.state ? a.state + ((int64_t)b * a.H + h) * DK * dv + c0 : nullptr;
    const bool keep = st && a.resume && a.resume[b];
    const int srow = 16 * RT * wave + 4 * g;                      // this lane's state rows: srow + 16 rt + r, columns 16 ct + c
    lf_f32x4 S[RT][2];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[rt][ct][r] = keep && 16 * ct + c < cols ? st[(int64_t)(srow + 16 * rt + r) * dv + 16 * ct + c] : 0.f;
    const float* zr = (const float*)a.z + (int64_t)row0 * a.ld;
    const int64_t hq = (int64_t)h * DK, hk = (int64_t)(a.H + h) * DK, hv = (int64_t)2 * a.H * DK + (int64_t)h * dv + c0;
    const int vtok = tid >> 3, vcol = 4 * (tid & 7);
    lf_f32x4 zq[QN], zk[QN], zv;
    auto request = [&](int t0) {
#pragma unroll
        for (int j = 0; j < QN; ++j) {
            const int i = tid + 256 * j, t = t0 + i / (DK / 4);
            const float* z = zr + (int64_t)(t < n ? t : n - 1) * a.ld + 4 * (i % (DK / 4));
            zq[j] = *(const lf_f32x4*)(z + hq);
            zk[j] = *(const lf_f32x4*)(z + hk);
        }
        zv = *(const lf_f32x4*)(zr + (int64_t)(t0 + vtok < n ? t0 + vtok : n - 1) * a.ld + hv + (vcol < cols ? vcol : 0));
    };
    auto act = [&](float x) { return a.act ? silu_t<float>(x) : x; };
    if (n > 0) request(0);
    __syncthreads();
    const int ti = wave >> 1, tj = wave & 1;                      // this wave's tile of the scores, and of o (tokens 16 ti, columns 16 tj)
    float wm[4], wr[4];                                          // A^(i - j), A^(i + 1) of its values i = 16 ti + 4 g + r, j = 16 tj + c
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int i = 16 * ti + 4 * g + r, d = i - 16 * tj - c;
        wm[r] = d >= 0 ? pw[d] : 0.f;
        wr[r] = pw[i + 1];
    }
    for (int t0 = 0; t0 < n; t0 += C) {
        const int nb = n - t0 < C ? n - t0 : C;
        bool odd = false;
#pragma unroll
        for (int j = 0; j < QN; ++j) {
            const int i = tid + 256 * j, t = i / (DK / 4), at = t * PQ + 4 * (i % (DK / 4));
            lf_f32x4 u = {0.f, 0.f, 0.f, 0.f}, w = u;
            if (t < nb) {
#pragma unroll
                for (int e = 0; e < 4; ++e) { u[e] = act(zq[j][e]); w[e] = act(zk[j][e]); }
            }
            *(lf_f32x4*)(q + at) = u;
            *(lf_f32x4*)(k + at) = w;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = vtok < nb && vcol < cols ? act(zv[e]) : 0.f;
            odd |= !(fabsf(x) <= 3.402823466e38f);
            vt[(vcol + e) * PT + vtok] = x;
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) *(lf_f32x4*)(s + (16 * ct + c) * PQ + srow + 16 * rt) = S[rt][ct];
        const bool apart = __syncthreads_or(odd);
        if (t0 + C < n) request(t0 + C);
        const lf_f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        lf_f32x4 sc8[8], o8[8], o = zero;                        // (sums of their own: an eighth of the roundings in a row)
#pragma unroll
        for (int e = 0; e < 8; ++e) sc8[e] = o8[e] = zero;
#pragma unroll
        for (int u = 0; u < DK / 16; ++u) {
            const lf_f32x4 x = *(const lf_f32x4*)(q + (16 * ti + c) * PQ + 16 * u + 4 * g), y = *(const lf_f32x4*)(k + (16 * tj + c) * PQ + 16 * u + 4 * g),
                           z = *(const lf_f32x4*)(s + (16 * tj + c) * PQ + 16 * u + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sc8[e + 4 * (u & 1)] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], sc8[e + 4 * (u & 1)], 0, 0, 0);
                o8[e + 4 * (u & 1)] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], z[e], o8[e + 4 * (u & 1)], 0, 0, 0);
            }
        }
        const lf_f32x4 sc = ((sc8[0] + sc8[1]) + (sc8[2] + sc8[3])) + ((sc8[4] + sc8[5]) + (sc8[6] + sc8[7])),
                       past = ((o8[0] + o8[1]) + (o8[2] + o8[3])) + ((o8[4] + o8[5]) + (o8[6] + o8[7]));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * ti + 4 * g + r;
            p[i * PT + 16 * tj + c] = i >= 16 * tj + c ? sc[r] * wm[r] : 0.f;
        }
        __syncthreads();
        if (!apart) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const lf_f32x4 x = *(const lf_f32x4*)(p + (16 * ti + c) * PT + 16 * u + 4 * g), y = *(const lf_f32x4*)(vt + (16 * tj + c) * PT + 16 * u + 4 * g);
#pragma unroll
                for (int e = 0; e < 4; ++e) o = __builtin_amdgcn_mfma_f32_16x16x4f32(x[e], y[e], o, 0, 0, 0);
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                for (int j = 0; j <= 16 * ti + 4 * g + r; ++j) o[r] = fmaf(p[(16 * ti + 4 * g + r) * PT + j], vt[(16 * tj + c) * PT + j], o[r]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = 16 * ti + 4 * g + r;
            if (i < nb && 16 * tj + c < cols) ((float*)a.o)[(int64_t)(row0 + t0 + i) * a.H * dv + (int64_t)h * dv + c0 + 16 * tj + c] = fmaf(wr[r], past[r], o[r]);
        }
        const float all = pw[nb];
        lf_f32x4 add[2][RT][2];                                  // (the chunk's own sum, in halves, added to the state in one rounding)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) add[0][rt][0] = add[0][rt][1] = add[1][rt][0] = add[1][rt][1] = zero;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            lf_f32x4 y[2];
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) y[ct] = *(const lf_f32x4*)(vt + (16 * ct + c) * PT + 16 * u + 4 * g);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int j = 16 * u + 4 * g + e;
                const float w = pw[j < nb ? nb - 1 - j : 0];      // (behind the last token k and v are zeros)
#pragma unroll
                for (int rt = 0; rt < RT; ++rt) {
                    const float x = k[j * PQ + 16 * RT * wave + 16 * rt + c];
#pragma unroll
                    for (int ct = 0; ct < 2; ++ct) add[u][rt][ct] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, y[ct][e] * w, add[u][rt][ct], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int r = 0; r < 4; ++r) S[rt][ct][r] = fmaf(all, S[rt][ct][r], add[0][rt][ct][r] + add[1][rt][ct][r]);
        __syncthreads();
    }
    if (st) {
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
            for (int ct = 0; ct < 2; ++ct)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (16 * ct + c < cols) st[(int64_t)(srow + 16 * rt + r) * dv + 16 * ct + c] = S[rt][ct][r];
    }
}

template <typename T, int CW>
static int recur_launch(LightArgs a, const float* decay, int64_t B, hipStream_t s) {
    const size_t lds = (size_t)(2 * a.dk + 32 + 32 * 33) * 4;
    hipLaunchKernelGGL((lightning_recur_kernel<T, CW>), dim3((unsigned)((a.dv + 8 * CW - 1) / (8 * CW)), (unsigned)a.H, (unsigned)B), dim3(256),
                       lds, s, a, decay);
    return evo_launch_status();
}

template <typename T, int CW, int R, int LT>
static int tokens_launch(LightArgs a, const float* decay, int64_t B, hipStream_t s) {
    const size_t lds = ((size_t)LT * (2 * a.dk + 32 + 32 * 33) + (CW == 4 ? (4 - 2 * LT * a.dk % 4) % 4 : 0) + (R ? 0 : a.dk * 8 * CW)) * 4;
    if (lds > 160 * 1024) return -1;
    if (lds > 64 * 1024) (void)hipFuncSetAttribute((const void*)lightning_tokens_kernel<T, CW, R, LT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    hipLaunchKernelGGL((lightning_tokens_kernel<T, CW, R, LT>), dim3((unsigned)((a.dv + 8 * CW - 1) / (8 * CW)), (unsigned)a.H, (unsigned)B), dim3(256),
                       lds, s, a, decay);
    return evo_launch_status();
}

extern "C" int evo_lightning_recurrent(const void* z, int64_t ld, void* o, float* state, const float* decay, const int* cu, const int* resume,
                                       int64_t B, int64_t H, int64_t dk, int64_t dv, int64_t act, int64_t f32, void* stream) {
    if (!z || !o || !decay || B <= 0 || B > 65535 || H <= 0 || H > 65535 || dk <= 0 || dk > 4096 || dv <= 0 || dv > 65536) return -1;
    if (ld < H * (2 * dk + dv) || (!cu && !state) || (resume && !state)) return -1;
    LightArgs a = {z, o, state, nullptr, cu, resume, nullptr, ld, (int)H, (int)dk, (int)dv, 1, 0, act != 0};
    hipStream_t s = (hipStream_t)stream;
    const bool quad = dv % 4 == 0;
    if (f32 && cu && (dk == 64 || dk == 128) && dv % 4 == 0 && ld % 4 == 0 && ((uintptr_t)z & 15) == 0) {      // (16-byte requests)
        const dim3 grid((unsigned)H, (unsigned)((dv + 31) / 32), (unsigned)B);
        if (dk == 64) hipLaunchKernelGGL(lightning_f32_kernel<1>, grid, dim3(256), 0, s, a, decay);
        else hipLaunchKernelGGL(lightning_f32_kernel<2>, grid, dim3(256), 0, s, a, decay);
        return evo_launch_status();
    }
    // (up to 128 rows the state is in registers and eight tokens share a barrier; wider heads have room for one token's rows beside the state)
#define LP(T) (dk <= 128 ? (quad ? tokens_launch<T, 4, 4, 8>(a, decay, B, s) : tokens_launch<T, 1, 4, 8>(a, decay, B, s))                                   \
                         : (quad && dk <= 1024 ? tokens_launch<T, 4, 0, 1>(a, decay, B, s) : tokens_launch<T, 1, 0, 1>(a, decay, B, s)))
#define LR(T) (cu ? LP(T) : (quad ? recur_launch<T, 4>(a, decay, B, s) : recur_launch<T, 1>(a, decay, B, s)))
    return f32 ? LR(float) : LR(uint16_t);
#undef LR
#undef LP
}
