// Softmax attention of packed prompts: causal, optionally over a sliding window whose first tokens stay visible, optionally with one sink per
// head in the denominator; query heads share key / value heads in groups; two attention maps over the same values may be combined on the way
// out (differential attention).  Entry point: include/evo_mi355x.h.
#include "mixers_common.h"
#include "../../include/evo_mi355x.h"

#define LOG2E 1.4426950408889634f

struct WinArgs {
    const void* q; const void* kn; const void* v; const void* kr; void* o;
    const int* cu_q; const int* cu_k; const float* sink;         // sink, kr: may be null
    int64_t ldq, ldkv;                                           // q row pitch; pitch of the kn / v rows
    int H, grp, dn, dr, dv, window, keep, n_qb;                  // grp query heads share a key / value head; kr rows are dr elements, o rows H dv
    float scale, lam, gain, eps;                                 // two maps: o = gain * unit_rms(o1 - lam o2)
};
#define FLOOR -1.0e30f                                           // running maximum before any key: finite, so that no difference of infinities arises

// Visible keys of query i (indexes into the sequence's keys, whose last ones are the queries'): j <= i and (i - j < window or j < keep).  A
// caller that leaves out keys between the kept ones and the window may do so: only order matters to both conditions.
//
// Matrix-core form (bf16).  A workgroup: 64 QC query rows of one (sequence, head); wave w owns 16 QC of them as MFMA COLUMNS: scores come
// as S^T = K Q^T (a lane holds one query's scores of four keys per 16-key block), so the softmax needs two cross-lane steps, the
// probabilities are the next product's operand as they stand (split key order), and O^T = V^T P^T is rescaled by one factor per lane.
// VEC: every row piece of eight elements is 16-byte aligned.
// Work item of this workgroup, (sequence, head, query block) in one number.  The query blocks of a (sequence, head) share most of their keys, as do the heads of a
// key head: they stay on one XCD (block b runs on XCD b % 8).  Where the key heads are a multiple of eight, every XCD gets as many of every sequence; a contiguous run
// of items per XCD, as for other numbers, gives one XCD the longest sequence.  us, runs -> key heads over the XCDs, latent attention of 32 heads / 8 key heads of four
// queries in a window of 1,024 / 16 heads of two maps: 6 sequences of 1,459 to 2,500 tokens 355 / 317 / 509 -> 304 / 268 / 369; 24 of 180 to 600 202 / 185 / 196
// -> 122 / 107 / 126; 3,000 and three times 300 265 / 265 / 442 -> 96 / 94 / 139; one of 8,190 214 / 196 / 705 -> 205 / 191 / 704.
__device__ __forceinline__ int work_item(const WinArgs& a) {
    const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3, G = a.H / a.grp;
    if (G & 7) return xcd * (int)(gridDim.x >> 3) + j;
    const int each = a.grp * a.n_qb;                             // items of a key head: they stay together
    return (j / each * 8 + xcd) * each + j % each;
}

// MAPS == 2: the two column blocks of a wave are the two maps of the same 16 queries -- rows of q and k hold [map 1 | map 2] per head --, the
// values are shared, and the maps meet in the epilogue.  KEEP: a.keep is not zero.  NW: waves
// (8: wide heads, whose sums leave a SIMD room for two waves of one workgroup only).  NH: a tile's keys are gone through in NH parts (2: half
// the registers for scores).
template <int KS, int DVB, int QC, bool VEC, bool KEEP, int MAPS, int MINW, int NW = 4, int NH = 1>
__global__ __launch_bounds__(64 * NW, MINW) void window_attn_kernel(WinArgs a, int B) {
    static_assert(MAPS == 1 || QC == 2, "two maps are two column blocks");
    constexpr int DQ = 32 * KS, PR = MAPS * DQ + 8, PT = 64 + 4, DVP = 16 * DVB, QW = 16 * QC / MAPS, QB = NW * QW;   // QW: queries of a wave
    constexpr int KG = DQ / 64, VG = DVP / 64;                   // groups of 64 key / value dimensions
    constexpr int KU = 8 / NW, VI = VG * 4 / NW;                 // keys per thread; groups of value dimensions per thread
    static_assert(NW == 4 || VG % 2 == 0, "eight waves share the value groups by halves");
    __shared__ __attribute__((aligned(16))) uint16_t k_rows[64 * PR], v_cols[DVP * PT];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    const int item = work_item(a), qb = item % a.n_qb, h = item / a.n_qb % a.H, b = item / a.n_qb / a.H;
    if (b >= B) return;                                          // (the grid is rounded up to a multiple of 8)
    const int q0 = a.cu_q[b], nq = a.cu_q[b + 1] - q0, k0 = a.cu_k[b], nk = a.cu_k[b + 1] - k0;
    if (qb * QB >= nq) return;
    const int off = nk - nq;                                     // key index of query 0
    const int dh = a.dn + a.dr, dn = a.dn, dv = a.dv, hk = h / a.grp;
    const uint16_t* kr = (const uint16_t*)a.kr + (int64_t)k0 * a.dr;
    const uint16_t* kn = (const uint16_t*)a.kn + (int64_t)k0 * a.ldkv + (int64_t)hk * dn * MAPS;
    const uint16_t* vg = (const uint16_t*)a.v + (int64_t)k0 * a.ldkv + (int64_t)hk * dv;
    mx_frag qf[QC][KS];
    int qi[QC];                                                  // this lane's query of each column block, as a key index
#pragma unroll
    for (int c = 0; c < QC; ++c) {
        const int i = qb * QB + wave * QW + (MAPS == 2 ? 0 : 16 * c) + c16;
        qi[c] = i + off;
        const uint16_t* p = (const uint16_t*)a.q + (int64_t)(q0 + (i < nq ? i : nq - 1)) * a.ldq + (int64_t)(h * MAPS + (MAPS == 2 ? c : 0)) * dh;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int d = 32 * ks + 8 * g;
            uint4 v = make_uint4(0u, 0u, 0u, 0u);
            if constexpr (VEC) { if (d < dh) v = *(const uint4*)(p + d); }
            else {
                uint32_t w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) w[e] = d + e < dh ? p[d + e] : 0u;
                v = make_uint4(w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16, w[6] | w[7] << 16);
            }
            qf[c][ks] = __builtin_bit_cast(mx_frag, v);
        }
    }
    const float sc2 = a.scale * LOG2E;
    f32x4_t o[QC][DVB];
    float mx[QC], den[QC];                                       // den: this lane's share (its keys); the sink sits in lane group 0's
#pragma unroll
    for (int c = 0; c < QC; ++c) {
        mx[c] = a.sink ? a.sink[h] * LOG2E : FLOOR;
        den[c] = a.sink && g == 0 ? 1.0f : 0.0f;
#pragma unroll
        for (int db = 0; db < DVB; ++db) o[c][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // eight threads share a row: thread (row rt = tid / 8, dims ct + 64 i) of keys rt and (four waves) rt + 32, values of keys 2 vt and 2 vt + 1
    // (eight waves: half of the value dims each).  A tile's base is uniform, offsets within it are 32 bits; eight waves make them anew for every
    // tile: held across tiles they spill.
    mx_u32x4 rk[MAPS * KG][KU], rv[VI][2];
    auto any8 = [](const uint16_t* x, int nx, const uint16_t* y, int ny, int d) {       // eight dims of [x (nx) | y (ny) | zeros], any alignment
        uint32_t w[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) w[e] = d + e < nx ? x[d + e] : (d + e < nx + ny ? y[d + e - nx] : 0u);
        return mx_u32x4{w[0] | w[1] << 16, w[2] | w[3] << 16, w[4] | w[5] << 16, w[6] | w[7] << 16};
    };
    // (keys past the end and dimensions past the head's repeat valid ones -- their scores are masked, the queries are zero there, their
    //  outputs are not stored --, so that the aligned form has no branch among its requests)
    const uint32_t row_bytes = (uint32_t)a.ldkv * 2;
    auto here = [](int v) __attribute__((always_inline)) {
        if constexpr (NW == 8) asm volatile("" : "+v"(v));
        return v;
    };
    auto load_k = [&](int j0) __attribute__((always_inline)) {
        const char* tile = (const char*)(kn + j0 * a.ldkv);
        const int t = here(tid), rt = t >> 3, ct = (t & 7) * 8;
#pragma unroll
        for (int u = 0; u < KU; ++u) {
            const int r = rt + 32 * u < nk - j0 ? rt + 32 * u : nk - 1 - j0;
            const uint16_t *pn = kn + (j0 + r) * a.ldkv, *pr_ = kr + (int64_t)(j0 + r) * a.dr;
#pragma unroll
            for (int i = 0; i < MAPS * KG; ++i) {
                const int d = ct + 64 * (i % KG), dc = d < dh ? d : dh - 8;
                if constexpr (!VEC) rk[i][u] = any8(pn + (i / KG) * dn, dn, pr_, a.dr, d);
                else if constexpr (MAPS == 2)                    // (a shared key part goes with one map only)
                    rk[i][u] = *(const mx_u32x4*)(tile + ((uint32_t)r * row_bytes + 2u * (uint32_t)((i / KG) * dn + dc)));
                else rk[i][u] = *(const mx_u32x4*)(dc < dn ? pn + dc : pr_ + (dc - dn));
            }
        }
    };
    auto load_v = [&](int j0) __attribute__((always_inline)) {
        const char* tile = (const char*)(vg + j0 * a.ldkv);
        const int t = here(tid), vt = (t >> 3) & 31, vi0 = (t >> 8) * VI, ct = (t & 7) * 8;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int r = 2 * vt + u < nk - j0 ? 2 * vt + u : nk - 1 - j0;
#pragma unroll
            for (int i = 0; i < VI; ++i) {
                const int d = ct + 64 * (vi0 + i);
                if constexpr (!VEC) rv[i][u] = any8(vg + (j0 + r) * a.ldkv, dv, vg, 0, d);
                else rv[i][u] = *(const mx_u32x4*)(tile + ((uint32_t)r * row_bytes + 2u * (uint32_t)(d < dv ? d : dv - 8)));
            }
        }
    };
    auto stage = [&]() __attribute__((always_inline)) {
        const int t = here(tid), rt = t >> 3, vt = rt & 31, vi0 = (t >> 8) * VI, ct = (t & 7) * 8;
#pragma unroll
        for (int i = 0; i < MAPS * KG; ++i)
#pragma unroll
            for (int u = 0; u < KU; ++u) *(mx_u32x4*)(k_rows + (rt + 32 * u) * PR + ct + 64 * i) = rk[i][u];
#pragma unroll
        for (int i = 0; i < VI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t x = rv[i][0][e], y = rv[i][1][e];
                uint16_t* c = v_cols + (ct + 64 * (vi0 + i) + 2 * e) * PT + 2 * vt;
                *(uint32_t*)c = (x & 0xffffu) | y << 16;
                *(uint32_t*)(c + PT) = x >> 16 | (y & 0xffff0000u);
            }
    };

    const int last_q = (qb + 1) * QB < nq ? (qb + 1) * QB - 1 : nq - 1;
    int j_lo = qb * QB + off - a.window + 1;
    j_lo = j_lo < 0 ? 0 : j_lo & ~63;
    const int j_hi = last_q + off;                               // last key any row of this block sees
    const int w_first = qb * QB + wave * QW + off, w_last = w_first + QW - 1;   // this wave's queries as key indexes
    const int keep = !KEEP ? 0 : (a.keep < j_lo ? a.keep : j_lo);   // kept keys ahead of the window's tiles: tiles [0, keep) come first
    auto after = [&](int j) { return KEEP && j < j_lo && j + 64 >= keep ? j_lo : j + 64; };
    int j0 = keep > 0 ? 0 : j_lo;
    load_k(j0);
    load_v(j0);
    for (int next = j0; j0 <= j_hi; j0 = next) {
        stage();
        __syncthreads();
        next = after(j0);
        const bool more = next <= j_hi;
        const bool mine = j0 <= w_last && (j0 + 63 > w_first - a.window || (KEEP && j0 < a.keep));   // some query of this wave sees some key of the tile
        constexpr int NJ = 4 / NH;                               // 16-key blocks of a part
#pragma unroll
        for (int hh = 0; hh < NH; ++hh) {
        f32x4_t s[QC][NJ];
        if (mine) {
#pragma unroll
            for (int jb = 0; jb < NJ; ++jb) {
#pragma unroll
                for (int c = 0; c < QC; ++c) s[c][jb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    const uint16_t* kp = k_rows + (16 * (hh * NJ + jb) + c16) * PR + 32 * ks + 8 * g;
                    const mx_frag kf = __builtin_bit_cast(mx_frag, *(const uint4*)kp);
#pragma unroll
                    for (int c = 0; c < QC; ++c)
                        s[c][jb] = mfma16(MAPS == 2 && c == 1 ? __builtin_bit_cast(mx_frag, *(const uint4*)(kp + DQ)) : kf, qf[c][ks], s[c][jb]);
                }
                if (jb & 1) __builtin_amdgcn_sched_barrier(0);   // (bounds the fragments read ahead)
            }
        }
        // the next tile's requests go out in two parts, between the phases: with all of them ahead of the scores the register file spills
        __builtin_amdgcn_sched_barrier(0);
        if (hh == NH - 1 && more) load_k(next);
        __builtin_amdgcn_sched_barrier(0);
        mx_frag pf[QC][NJ / 2];
        if (mine) {
            if (j0 + 63 > w_first || (j0 <= w_last - a.window && (!KEEP || j0 + 63 >= a.keep))) {   // the tile holds an edge of some query's window
#pragma unroll
                for (int c = 0; c < QC; ++c)
#pragma unroll
                    for (int jb = 0; jb < NJ; ++jb)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const int j = j0 + 16 * (hh * NJ + jb) + 4 * g + r, age = qi[c] - j;
                            s[c][jb][r] = age >= 0 && (age < a.window || (KEEP && j < a.keep)) ? s[c][jb][r] * sc2 : -INFINITY;
                        }
            } else {
#pragma unroll
                for (int c = 0; c < QC; ++c)
#pragma unroll
                    for (int jb = 0; jb < NJ; ++jb)
#pragma unroll
                        for (int r = 0; r < 4; ++r) s[c][jb][r] *= sc2;
            }
#pragma unroll
            for (int c = 0; c < QC; ++c) {
                float top = mx[c];
#pragma unroll
                for (int jb = 0; jb < NJ; ++jb) top = fmaxf(top, fmaxf(fmaxf(s[c][jb][0], s[c][jb][1]), fmaxf(s[c][jb][2], s[c][jb][3])));
                top = fmaxf(top, __shfl_xor(top, 16, 64));
                top = fmaxf(top, __shfl_xor(top, 32, 64));
                if (__builtin_amdgcn_ballot_w64(top > mx[c])) {          // the running maximum moved in some column: rescale
                    const float f = __builtin_amdgcn_exp2f(mx[c] - top);
                    mx[c] = top;
                    den[c] *= f;
#pragma unroll
                    for (int db = 0; db < DVB; ++db)
#pragma unroll
                        for (int r = 0; r < 4; ++r) o[c][db][r] *= f;
                }
                uint32_t w[2 * NJ];
#pragma unroll
                for (int jb = 0; jb < NJ; ++jb) {
                    float e[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        e[r] = __builtin_amdgcn_exp2f(s[c][jb][r] - mx[c]);
                        den[c] += e[r];
                    }
                    w[2 * jb] = pack_bf2(e[0], e[1]);
                    w[2 * jb + 1] = pack_bf2(e[2], e[3]);
                }
#pragma unroll
                for (int jj = 0; jj < NJ / 2; ++jj) pf[c][jj] = frag_of(w[4 * jj], w[4 * jj + 1], w[4 * jj + 2], w[4 * jj + 3]);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (hh == NH - 1 && more) load_v(next);
        __builtin_amdgcn_sched_barrier(0);
        if (mine) {
#pragma unroll
            for (int jj = 0; jj < NJ / 2; ++jj)
#pragma unroll
                for (int db = 0; db < DVB; ++db) {
                    const mx_frag vf = frag_split(v_cols + (16 * db + c16) * PT + 32 * (hh * (NJ / 2) + jj) + 4 * g);
#pragma unroll
                    for (int c = 0; c < QC; ++c) o[c][db] = mfma16(vf, pf[c][jj], o[c][db]);
                    if ((db & 3) == 3) __builtin_amdgcn_sched_barrier(0);
                }
        }
        }
        __syncthreads();
    }
    float inv[QC];
#pragma unroll
    for (int c = 0; c < QC; ++c) {
        float l = den[c];
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        inv[c] = 1.0f / l;
    }
    if constexpr (MAPS == 2) {                                   // the difference of the maps, its unit norm over the head's values
        const float i1 = inv[0], i2 = inv[1] * a.lam;
        float ss = 0.f;
#pragma unroll
        for (int db = 0; db < DVB; ++db)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float x = o[0][db][r] * i1 - o[1][db][r] * i2;
                o[0][db][r] = x;
                if (16 * db + 4 * g + r < dv) ss = fmaf(x, x, ss);
            }
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        inv[0] = a.gain / sqrtf(ss / (float)dv + a.eps);
    }
#pragma unroll
    for (int c = 0; c < QC / MAPS; ++c) {
        const int i = qi[c] - off;
        if (i < nq) {
            uint16_t* op = (uint16_t*)a.o + (int64_t)(q0 + i) * a.H * dv + (int64_t)h * dv;
#pragma unroll
            for (int db = 0; db < DVB; ++db) {
                const int d = 16 * db + 4 * g;
                if (d + 3 < dv && (dv & 3) == 0)
                    *(uint2*)(op + d) = make_uint2(pack_bf2(o[c][db][0] * inv[c], o[c][db][1] * inv[c]), pack_bf2(o[c][db][2] * inv[c], o[c][db][3] * inv[c]));
                else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (d + r < dv) op[d + r] = f_to_bf(o[c][db][r] * inv[c]);
                }
            }
        }
    }
}

// The same for the head sizes below at length (bf16), with nothing but products and the softmax in the loop: rows of K and V go to LDS by DMA as they lie
// (granules of 16 bytes XORed by their row on the source side), NS tiles of 64 keys deep, one barrier per tile, and the value fragments are read transposed.
// A workgroup is eight waves of 32 queries (two column blocks); with two maps, four query groups by two maps -- a wave reads its map's keys only --, which
// meet in LDS at the end.  A running maximum moves only when a score passes it by 2^WT_STEP (every rounding is relative; sums keep 2^-127 of room).
// Causal blocks start with the longest.
// Bound by the chain of a tile -- fragments, scores, maximum, exponentials, values -- of the two waves on a SIMD: about 3.5 us of which the matrix cores take 1.1 to 1.5.
// MI355X, before (register staging, V transposed by 4-byte stores, one wave for both maps) -> here: two maps, 16 heads of 128 and 256, 8,190 tokens causal
// 1,872 -> 943 us (874 TF); 32 heads of 192 and 128, window 1,024, six prompts of 700 to 2,500 tokens 526 -> 403; 32 heads of 128, window 1,024 and kept
// tokens, 8,190 tokens 292 -> 217.  (Waves of a SIMD half a tile apart by two barriers per tile were slower: 465 for the second.)
#define WT_STEP 8.0f
typedef short wt_s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) wt_s16x4* wt_tr_ptr;
// the maximum over the four lanes of a column (lanes 16 apart), one swap each instead of a trip through LDS
__device__ __forceinline__ float wt_row_max(float v) {
    const uint32_t u = __float_as_uint(v);
    const auto p = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = fmaxf(__uint_as_float((uint32_t)p[0]), __uint_as_float((uint32_t)p[1]));
    const uint32_t x = __float_as_uint(v);
    const auto q = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return fmaxf(__uint_as_float((uint32_t)q[0]), __uint_as_float((uint32_t)q[1]));
}
template <int DN, int DR, int DV, int MAPS, bool KEEP>
__global__ __launch_bounds__(512, 2) void window_tile_kernel(WinArgs a, int B) {
    static_assert(DN == 128 && (DR == 0 || DR == 64) && (DV == 128 || DV == 256) && (MAPS == 1 || DR == 0), "row widths of the swizzles");
    constexpr int KN = 64 * DN * 2, KR = 64 * DR * 2, VB = 64 * DV * 2, STAGE = MAPS * KN + KR + VB, NS = STAGE > 48 * 1024 ? 2 : STAGE > 36 * 1024 ? 3 : 4;
    constexpr int KS = DN / 32, RS = DR / 32, DVB = DV / 16, PK = KN / 8192, PR = KR / 8192, PV = VB / 8192, P = MAPS * PK + PR + PV;   // DMA pieces (1 KiB) per wave
    constexpr int VRP = 1024 / (2 * DV), VG = DV / 8;            // value rows per piece, granules of a value row
    constexpr int QB = 256 / MAPS;
    static_assert(NS * STAGE <= 160 * 1024, "the CU's LDS");
    __shared__ __attribute__((aligned(16))) unsigned char smem[NS * STAGE];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    const int map = MAPS == 2 ? wave >> 2 : 0, grp = MAPS == 2 ? wave & 3 : wave;      // (waves w and w + 4 share a SIMD)
    const int item = work_item(a), qb = a.n_qb - 1 - item % a.n_qb, h = item / a.n_qb % a.H, b = item / a.n_qb / a.H;
    if (b >= B) return;                                          // (the grid is rounded up to a multiple of 8)
    const int q0 = a.cu_q[b], nq = a.cu_q[b + 1] - q0, k0 = a.cu_k[b], nk = a.cu_k[b + 1] - k0;
    const int off = nk - nq;                                     // key index of query 0
    // two maps: blocks of 32 queries start at multiples of 32 keys, so that every tile a wave takes holds a key that all of its queries see (a value that
    // is not finite goes no further than with blocks of 16); block 0 is the short one
    const int qs = qb * QB - (MAPS == 2 ? off & 31 : 0);         // this workgroup's first query (may be negative)
    if (qs >= nq) return;
    const int hk = h / a.grp;
    constexpr int dh = DN + DR;
    const uint64_t kr = (uint64_t)((const uint16_t*)a.kr + (int64_t)k0 * DR);
    const uint64_t kn = (uint64_t)((const uint16_t*)a.kn + (int64_t)k0 * a.ldkv + (int64_t)hk * DN * MAPS);
    const uint64_t vg = (uint64_t)((const uint16_t*)a.v + (int64_t)k0 * a.ldkv + (int64_t)hk * DV);
    const uint32_t rowb = (uint32_t)a.ldkv * 2;

    mx_frag qf[2][KS + RS];
    int qi[2];                                                   // this lane's query of each column block, as a key index
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int i = qs + grp * 32 + 16 * c + c16;
        qi[c] = i + off;
        const uint16_t* p = (const uint16_t*)a.q + (int64_t)(q0 + (i < 0 ? 0 : i < nq ? i : nq - 1)) * a.ldq + (int64_t)(h * MAPS + map) * dh;
#pragma unroll
        for (int ks = 0; ks < KS + RS; ++ks) qf[c][ks] = __builtin_bit_cast(mx_frag, *(const uint4*)(p + 32 * ks + 8 * g));
    }
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
        for (int ks = 0; ks < KS + RS; ++ks) asm volatile("" : "+v"(qf[c][ks]));       // (waited for here: a wait in the loop would be one for the DMA)

    // DMA: piece i of this wave is piece wave + 8 i of a slab: key rows 4 to a piece (granule r ^ (row & 15)), shared key rows 8 (r ^ (row / 2 & 7)), value
    // rows 2 or 4 (r ^ 2 (row & 7)).  Row offsets are in the lanes' part: the descriptor's bound returns zeros behind the last key.
    typedef uint32_t wt_u32x4 __attribute__((ext_vector_type(4)));
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    const int kr_ = 4 * wave + (lane >> 4), rr_ = 8 * wave + (lane >> 3), vr_ = VRP * wave + lane / VG;
    const uint32_t k_off = (uint32_t)kr_ * rowb + (uint32_t)(((lane & 15) ^ (kr_ & 15)) * 16);
    const uint32_t r_off = (uint32_t)rr_ * (2 * DR) + (uint32_t)(((lane & 7) ^ ((rr_ >> 1) & 7)) * 16);
    const uint32_t v_off = (uint32_t)vr_ * rowb + (uint32_t)(((lane % VG) ^ (2 * (vr_ & 7))) * 16);
    auto dma = [&](uint32_t dst, uint32_t voff, wt_u32x4 rsrc) __attribute__((always_inline)) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(dst), "v"(voff), "s"(rsrc) : "memory", "m0");
    };
    auto fetch = [&](int j0, bool any, int slot) __attribute__((always_inline)) {      // (none: the same requests with an empty bound)
        const int left = any ? (nk - j0 < 64 ? nk - j0 : 64) : 0;
        const uint64_t ka = kn + (any ? (uint64_t)j0 * rowb : 0), va = vg + (any ? (uint64_t)j0 * rowb : 0), ra = kr + (any ? (uint64_t)j0 * (2 * DR) : 0);
        const uint32_t rows = left > 0 ? (uint32_t)(left - 1) * rowb : 0u;
        const wt_u32x4 sk = {(uint32_t)ka, (uint32_t)(ka >> 32) & 0xffffu, left > 0 ? rows + MAPS * DN * 2 : 0u, 0x00020000u};
        const wt_u32x4 sv = {(uint32_t)va, (uint32_t)(va >> 32) & 0xffffu, left > 0 ? rows + DV * 2 : 0u, 0x00020000u};
        const wt_u32x4 sr = {(uint32_t)ra, (uint32_t)(ra >> 32) & 0xffffu, (uint32_t)left * (2 * DR), 0x00020000u};
        const uint32_t base = lds0 + (uint32_t)slot * STAGE + wave * 1024;
#pragma unroll
        for (int m = 0; m < MAPS; ++m)
#pragma unroll
            for (int i = 0; i < PK; ++i) dma(base + m * KN + i * 8192, k_off + (uint32_t)i * 32u * rowb + m * (DN * 2), sk);
        if constexpr (DR > 0) {
#pragma unroll
            for (int i = 0; i < PR; ++i) dma(base + MAPS * KN + i * 8192, r_off + i * (64 * 2 * DR), sr);
        }
#pragma unroll
        for (int i = 0; i < PV; ++i) dma(base + MAPS * KN + KR + i * 8192, v_off + (uint32_t)(i * 8 * VRP) * rowb, sv);
    };

    const float sc2 = a.scale * LOG2E;
    f32x4_t o[2][DVB];
    float mx[2], den[2];                                         // den: this lane's share (its keys); the sink sits in lane group 0's
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        mx[c] = a.sink && !(a.sink[h] * LOG2E <= FLOOR) ? a.sink[h] * LOG2E : FLOOR;     // (a NaN stays one)
        den[c] = a.sink && g == 0 ? 1.0f : 0.0f;
#pragma unroll
        for (int db = 0; db < DVB; ++db) o[c][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    // fragment addresses in a stage: key row c16 (+ 16 jb), granule 4 ks + g; value rows 4 g + c16 / 4 (+ 16 u), columns 16 db + 4 (c16 % 4)
    uint32_t k_rd[KS], r_rd[RS > 0 ? RS : 1], v_rd[8];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) k_rd[ks] = map * KN + c16 * (DN * 2) + ((4 * ks + g) ^ c16) * 16;
#pragma unroll
    for (int ks = 0; ks < RS; ++ks) r_rd[ks] = MAPS * KN + c16 * (DR * 2) + ((4 * ks + g) ^ ((c16 >> 1) & 7)) * 16;
#pragma unroll
    for (int db = 0; db < 8; ++db) {
        const int r = 4 * g + (c16 >> 2);
        v_rd[db] = MAPS * KN + KR + r * (DV * 2) + ((2 * db + ((c16 & 3) >> 1)) ^ (2 * (r & 7))) * 16 + (c16 & 1) * 8;
    }

    const int last_q = qs + QB < nq ? qs + QB - 1 : nq - 1;
    int j_lo = qs + off - a.window + 1;
    j_lo = j_lo < 0 ? 0 : j_lo & ~63;
    const int j_hi = last_q + off;                               // last key any row of this block sees
    const int w_first = qs + grp * 32 + off, w_last = w_first + 31;             // this wave's queries as key indexes
    const int keep = !KEEP ? 0 : (a.keep < j_lo ? a.keep : j_lo);   // kept keys ahead of the window's tiles: tiles [0, keep) come first
    auto after = [&](int j) { return KEEP && j < j_lo && j + 64 >= keep ? j_lo : j + 64; };
    int j0 = keep > 0 ? 0 : j_lo, jf = j0, slot = 0, fslot = NS - 1;
#pragma unroll
    for (int t = 0; t < NS - 1; ++t) {
        fetch(jf, jf <= j_hi, t);
        if (jf <= j_hi) jf = after(jf);
    }
    for (; j0 <= j_hi; j0 = after(j0)) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * P) : "memory");     // own pieces of this tile; barrier: everyone's, and everyone is done with the last
        asm volatile("s_barrier" ::: "memory");
        fetch(jf, jf <= j_hi, fslot);
        if (jf <= j_hi) jf = after(jf);
        const unsigned char* st = smem + slot * STAGE;
        fslot = slot;
        slot = slot + 1 == NS ? 0 : slot + 1;
        if (!(j0 <= w_last && (j0 + 63 > w_first - a.window || (KEEP && j0 < a.keep)))) continue;   // no query of this wave sees a key of the tile
        f32x4_t s[2][4];
        {
            constexpr int KF = KS + RS, NF = 4 * KF, D = 4;      // fragments of the tile; read ahead
            auto frag = [&](int f) __attribute__((always_inline)) {
                const int jb = f / KF, ks = f % KF;
                return *(const uint4*)(ks < KS ? st + k_rd[ks < KS ? ks : 0] + jb * (16 * DN * 2) : st + r_rd[ks < KS ? 0 : ks - KS] + jb * (16 * DR * 2));
            };
            uint4 kf[D];
#pragma unroll
            for (int f = 0; f < D; ++f) kf[f] = frag(f);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const int jb = f / KF, ks = f % KF;
                if (ks == 0) s[0][jb] = s[1][jb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int c = 0; c < 2; ++c) s[c][jb] = mfma16(__builtin_bit_cast(mx_frag, kf[f % D]), qf[c][ks], s[c][jb]);
                if (f + D < NF) kf[f % D] = frag(f + D);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (j0 + 63 > w_first || (j0 <= w_last - a.window && (!KEEP || j0 + 63 >= a.keep))) {   // the tile holds an edge of some query's window
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int jb = 0; jb < 4; ++jb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int j = j0 + 16 * jb + 4 * g + r, age = qi[c] - j;
                        s[c][jb][r] = age >= 0 && (age < a.window || (KEEP && j < a.keep)) ? s[c][jb][r] : -INFINITY;
                    }
        }
        mx_frag pf[2][2];
        // (both column blocks side by side: their chains fill each other's latencies)
        float top[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float t[4];
#pragma unroll
            for (int jb = 0; jb < 4; ++jb) t[jb] = fmaxf(fmaxf(s[c][jb][0], s[c][jb][1]), fmaxf(s[c][jb][2], s[c][jb][3]));
            top[c] = wt_row_max(fmaxf(fmaxf(t[0], t[1]), fmaxf(t[2], t[3]))) * sc2;
        }
        if (__builtin_amdgcn_ballot_w64(top[0] > mx[0] + WT_STEP || top[1] > mx[1] + WT_STEP)) {       // a running maximum moves in some column: rescale
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const float m = fmaxf(mx[c], top[c]), f = __builtin_amdgcn_exp2f(mx[c] - m);
                mx[c] = m;
                den[c] *= f;
#pragma unroll
                for (int db = 0; db < DVB; ++db)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[c][db][r] *= f;
            }
        }
        uint32_t w[2][8];
#pragma unroll
        for (int jb = 0; jb < 4; ++jb)
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float e[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) e[r] = __builtin_amdgcn_exp2f(fmaf(s[c][jb][r], sc2, -mx[c]));
                den[c] += (e[0] + e[1]) + (e[2] + e[3]);
                w[c][2 * jb] = pack_bf2(e[0], e[1]);
                w[c][2 * jb + 1] = pack_bf2(e[2], e[3]);
            }
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int jj = 0; jj < 2; ++jj) pf[c][jj] = frag_of(w[c][4 * jj], w[c][4 * jj + 1], w[c][4 * jj + 2], w[c][4 * jj + 3]);
        {
            constexpr int NF = 2 * DVB, D = 4;
            uint2 va[D], vb[D];
            auto frag = [&](int f, int i) __attribute__((always_inline)) {
                const int jj = f / DVB, db = f % DVB;
                const unsigned char* p = st + v_rd[db & 7] + (db >> 3) * 256 + jj * (32 * DV * 2);
                va[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((wt_tr_ptr)p));
                vb[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((wt_tr_ptr)(p + 16 * DV * 2)));
            };
#pragma unroll
            for (int f = 0; f < D; ++f) frag(f, f);
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                const mx_frag vf = frag_of(va[f % D].x, va[f % D].y, vb[f % D].x, vb[f % D].y);
#pragma unroll
                for (int c = 0; c < 2; ++c) o[c][f % DVB] = mfma16(vf, pf[c][f / DVB], o[c][f % DVB]);
                if (f + D < NF) frag(f + D, f % D);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");             // (the empty requests: nothing may land after the exit, or on what comes below)
    float inv[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        float l = den[c];
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        inv[c] = 1.0f / l;
    }
    if constexpr (MAPS == 2) {                                   // the difference of the maps, its unit norm over the head's values
        f32x4_t* x = (f32x4_t*)smem + grp * (2 * DVB * 64) + lane;      // [4 query groups][2][DVB][64 lanes]: 128 KB
        asm volatile("s_barrier" ::: "memory");                  // (everyone is done with the last tile)
        if (map == 1) {
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int db = 0; db < DVB; ++db) x[(c * DVB + db) * 64] = o[c][db] * (inv[c] * a.lam);
        }
        __syncthreads();
        if (map == 1) return;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            float ss = 0.f;
#pragma unroll
            for (int db = 0; db < DVB; ++db) {
                const f32x4_t y = x[(c * DVB + db) * 64];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    o[c][db][r] = fmaf(o[c][db][r], inv[c], -y[r]);
                    ss = fmaf(o[c][db][r], o[c][db][r], ss);
                }
            }
            ss += __shfl_xor(ss, 16, 64);
            ss += __shfl_xor(ss, 32, 64);
            inv[c] = a.gain / sqrtf(ss / (float)DV + a.eps);
        }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const int i = qi[c] - off;
        if (i >= 0 && i < nq) {
            uint16_t* op = (uint16_t*)a.o + (int64_t)(q0 + i) * a.H * DV + (int64_t)h * DV + 4 * g;
#pragma unroll
            for (int db = 0; db < DVB; ++db)
                *(uint2*)(op + 16 * db) = make_uint2(pack_bf2(o[c][db][0] * inv[c], o[c][db][1] * inv[c]), pack_bf2(o[c][db][2] * inv[c], o[c][db][3] * inv[c]));
        }
    }
}

// fp32 on the matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands and sums).  A workgroup: 64 queries of one (sequence, head), 16 a wave as MFMA columns;
// 32 keys at a time in LDS, the rows of K and V 4 floats apart from a multiple of 64 (both read patterns meet every bank once).  Scores come as
// S^T = K Q^T with the reduced index taken as d = 16 s + 4 g + j (a lane's four d are one 16-byte read), a lane holds keys 4 g + r of its query, which is
// the operand of O^T = V^T P^T when that product's key index is taken in the same order.  MAPS == 2: the two maps are two column blocks.
// Bound by the fp32 matrix rate (256 flop a cycle and CU) at length, by its 2 - 16 key tiles at the sizes of a checked trace.  The wave-per-query form
// below read every key row once per query with one lane a key: 3 prompts of 240 - 500 tokens x 32 heads of 192 x 128 took 5,080 us (139 here),
// 16 heads of two maps 128 x 256 4,292 us (280 here).
template <int KS, int DVB, int MAPS>
__global__ __launch_bounds__(256, 1) void window_attn_f32_kernel(WinArgs a) {
    constexpr int DQ = 16 * KS, PK = MAPS * DQ + 4, DVP = 16 * DVB, PV = DVP + 4, KT = 32;
    __shared__ __attribute__((aligned(16))) float ks[KT * PK], vs[KT * PV];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c16 = lane & 15, g = lane >> 4;
    // (heads first: block i runs on XCD i % 8, and query blocks first would give one XCD the last, longest blocks of 512 queries; those start first.
    //  3 prompts of 267 to 500: latent 199 -> 147 us, grouped heads 141 -> 119, two maps 274 -> 226)
    const int h = blockIdx.x % a.H, b = blockIdx.z;
    const int q0 = a.cu_q[b], nq = a.cu_q[b + 1] - q0, k0 = a.cu_k[b], nk = a.cu_k[b + 1] - k0;
    const int qb = (a.n_qb - 1 - blockIdx.x / a.H) * 64;
    if (qb >= nq) return;
    const int off = nk - nq, dh = a.dn + a.dr, hk = h / a.grp;
    const float* kr = (const float*)a.kr + (int64_t)k0 * a.dr;
    const float* kn = (const float*)a.kn + (int64_t)k0 * a.ldkv + (int64_t)hk * a.dn * MAPS;
    const float* vg = (const float*)a.v + (int64_t)k0 * a.ldkv + (int64_t)hk * a.dv;
    const int i = qb + 16 * wave + c16, ki = i + off;            // this lane's query, as a row and as a key
    f32x4_t qf[MAPS][KS];
#pragma unroll
    for (int map = 0; map < MAPS; ++map) {
        const float* q = (const float*)a.q + (int64_t)(q0 + (i < nq ? i : nq - 1)) * a.ldq + (int64_t)(h * MAPS + map) * dh;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d = 16 * s + 4 * g;
            qf[map][s] = d < dh ? *(const f32x4_t*)(q + d) : f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
    }
    f32x4_t o[MAPS][DVB];
    float m[MAPS], l[MAPS];
#pragma unroll
    for (int map = 0; map < MAPS; ++map) {
        m[map] = a.sink ? a.sink[h] : -INFINITY;
        l[map] = a.sink && g == 0 ? 1.0f : 0.0f;                 // (the lanes of a query hold parts of its sum)
#pragma unroll
        for (int e = 0; e < DVB; ++e) o[map][e] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
    const int last = (qb + 63 < nq - 1 ? qb + 63 : nq - 1) + off;
    const int lo = qb + off - a.window + 1 > 0 ? qb + off - a.window + 1 : 0, kept = a.keep < lo ? a.keep : lo;
    for (int part = kept > 0 ? 0 : 1; part < 2; ++part)          // the kept keys ahead of every window, then the windows
        for (int j0 = part ? lo : 0, end = part ? last + 1 : kept; j0 < end; j0 += KT) {
            __syncthreads();
            for (int e = tid; e < KT * (MAPS * DQ / 4); e += 256) {
                const int r = e / (MAPS * DQ / 4), c = (e - r * (MAPS * DQ / 4)) * 4, map = c / DQ, d = c - map * DQ, j = j0 + r;
                f32x4_t v = {0.f, 0.f, 0.f, 0.f};
                if (j < end) {
                    if (d < a.dn) v = *(const f32x4_t*)(kn + j * a.ldkv + map * a.dn + d);
                    else if (d < dh) v = *(const f32x4_t*)(kr + (int64_t)j * a.dr + (d - a.dn));
                }
                *(f32x4_t*)(ks + r * PK + c) = v;
            }
            int odd = 0;                                         // an infinite value or none: it may only reach the queries that see its key
            for (int e = tid; e < KT * (DVP / 4); e += 256) {
                const int r = e / (DVP / 4), d = (e - r * (DVP / 4)) * 4, j = j0 + r;
                const f32x4_t v = j < end && d < a.dv ? *(const f32x4_t*)(vg + j * a.ldkv + d) : f32x4_t{0.f, 0.f, 0.f, 0.f};
                *(f32x4_t*)(vs + r * PV + d) = v;
#pragma unroll
                for (int u = 0; u < 4; ++u) odd |= !(fabsf(v[u]) <= 3.402823466e38f);
            }
            odd = __syncthreads_or(odd);
#pragma unroll
            for (int map = 0; map < MAPS; ++map) {
                f32x4_t p[2];
                float top = -INFINITY;
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    p[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                    const float* kp = ks + (16 * t + c16) * PK + map * DQ + 4 * g;
#pragma unroll
                    for (int s = 0; s < KS; ++s) {
                        const f32x4_t kv = *(const f32x4_t*)(kp + 16 * s);
#pragma unroll
                        for (int j = 0; j < 4; ++j) p[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[j], qf[map][s][j], p[t], 0, 0, 0);
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int j = j0 + 16 * t + 4 * g + r;
                        const bool seen = j < end && j <= ki && (ki - j < a.window || j < a.keep);
                        p[t][r] = seen ? p[t][r] * a.scale : -INFINITY;
                        top = fmaxf(top, p[t][r]);
                    }
                }
                top = fmaxf(top, __shfl_xor(top, 16, 64));
                top = fmaxf(fmaxf(top, __shfl_xor(top, 32, 64)), m[map]);
                const float base = top == -INFINITY ? 0.f : top, f = expf(m[map] - base);      // (no key seen yet: everything stays zero)
                m[map] = top;
                float sum = 0.f;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) { p[t][r] = expf(p[t][r] - base); sum += p[t][r]; }
                l[map] = l[map] * f + sum;
                if (odd) {
#pragma unroll
                    for (int e = 0; e < DVB; ++e) o[map][e] *= f;
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            for (int u = 0; u < 4; ++u) {
                                const int row = 16 * t + 4 * u + r, j = j0 + row;
                                const float pj = __shfl(p[t][r], 16 * u + c16, 64);
                                if (j < end && j <= ki && (ki - j < a.window || j < a.keep))
#pragma unroll
                                    for (int e = 0; e < DVB; ++e) o[map][e] += pj * *(const f32x4_t*)(vs + row * PV + 16 * e + 4 * g);
                            }
                } else
#pragma unroll
                for (int e = 0; e < DVB; ++e) {
                    o[map][e] *= f;
#pragma unroll
                    for (int t = 0; t < 2; ++t)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            o[map][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(vs[(16 * t + 4 * g + r) * PV + 16 * e + c16], p[t][r], o[map][e], 0, 0, 0);
                }
            }
        }
#pragma unroll
    for (int map = 0; map < MAPS; ++map) {
        l[map] += __shfl_xor(l[map], 16, 64);
        l[map] += __shfl_xor(l[map], 32, 64);
#pragma unroll
        for (int e = 0; e < DVB; ++e) o[map][e] /= l[map];
    }
    float gain = 1.0f;
    if constexpr (MAPS == 2) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < DVB; ++e) {
            o[0][e] -= a.lam * o[1][e];
#pragma unroll
            for (int r = 0; r < 4; ++r) ss = fmaf(o[0][e][r], o[0][e][r], ss);      // (columns behind dv are zero)
        }
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        gain = a.gain / sqrtf(ss / (float)a.dv + a.eps);
    }
    if (i < nq) {
        float* op = (float*)a.o + (int64_t)(q0 + i) * a.H * a.dv + (int64_t)h * a.dv + 4 * g;
#pragma unroll
        for (int e = 0; e < DVB; ++e)
            if (16 * e + 4 * g < a.dv) *(f32x4_t*)(op + 16 * e) = o[0][e] * gain;
    }
}

// Any sizes, both storage types: one wave per (query, head); lanes are keys for the scores, value columns for the sum
template <typename T, int MAPS>
__global__ __launch_bounds__(64) void window_attn_any_kernel(WinArgs a) {
    extern __shared__ float qs[];                                // dn + dr floats
    const int qr = blockIdx.x, h = blockIdx.y, b = blockIdx.z, lane = threadIdx.x;
    const int q0 = a.cu_q[b], nq = a.cu_q[b + 1] - q0, k0 = a.cu_k[b], nk = a.cu_k[b + 1] - k0;
    if (qr >= nq) return;
    const int dh = a.dn + a.dr, ki = qr + nk - nq, hk = h / a.grp;
    const T* vg = (const T*)a.v + (int64_t)k0 * a.ldkv + (int64_t)hk * a.dv;
    const T* kr = (const T*)a.kr + (int64_t)k0 * a.dr;
    const int j_lo = ki - a.window + 1 < 0 ? 0 : ki - a.window + 1, keep = a.keep < j_lo ? a.keep : j_lo;
    float o[MAPS][8];
#pragma unroll
    for (int map = 0; map < MAPS; ++map) {
        const T* q = (const T*)a.q + (int64_t)(q0 + qr) * a.ldq + (int64_t)(h * MAPS + map) * dh;
        __syncthreads();
        for (int d = lane; d < dh; d += 64) qs[d] = ld1(q + d);
        __syncthreads();
        const T* kn = (const T*)a.kn + (int64_t)k0 * a.ldkv + (int64_t)(hk * MAPS + map) * a.dn;
        float m = a.sink ? a.sink[h] : -INFINITY, l = a.sink ? 1.0f : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[map][e] = 0.f;
        for (int part = keep > 0 ? 0 : 1; part < 2; ++part)      // the kept keys ahead of the window, then the window
            for (int j0 = part ? j_lo : 0, end = part ? ki + 1 : keep; j0 < end; j0 += 64) {
                const int j = j0 + lane;
                float s = -INFINITY;
                if (j < end) {
                    s = 0.f;
                    for (int d = 0; d < a.dn; ++d) s = fmaf(qs[d], ld1(kn + j * a.ldkv + d), s);
                    for (int d = 0; d < a.dr; ++d) s = fmaf(qs[a.dn + d], ld1(kr + (int64_t)j * a.dr + d), s);
                    s *= a.scale;
                }
                const float top = fmaxf(m, wave_max(s)), f = expf(m - top), p = expf(s - top);
                m = top;
                l = l * f + wave_sum(p);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[map][e] *= f;
                const int n = end - j0 < 64 ? end - j0 : 64;
                for (int u = 0; u < n; ++u) {
                    const float pu = __shfl(p, u, 64);
                    const T* vr = vg + (j0 + u) * a.ldkv;
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (lane + 64 * e < a.dv) o[map][e] = fmaf(pu, ld1(vr + lane + 64 * e), o[map][e]);
                }
            }
#pragma unroll
        for (int e = 0; e < 8; ++e) o[map][e] /= l;
    }
    float gain = 1.0f;
    if constexpr (MAPS == 2) {
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            o[0][e] -= a.lam * o[1][e];
            if (lane + 64 * e < a.dv) ss = fmaf(o[0][e], o[0][e], ss);
        }
        gain = a.gain / sqrtf(wave_sum(ss) / (float)a.dv + a.eps);
    }
    T* op = (T*)a.o + (int64_t)(q0 + qr) * a.H * a.dv + (int64_t)h * a.dv;
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (lane + 64 * e < a.dv) st1(op + lane + 64 * e, o[0][e] * gain);
}

extern "C" int evo_window_attn(const void* q, int64_t ldq, const void* kn, const void* v, int64_t ldkv, const void* kr, void* o, const int* cu_q,
                               const int* cu_k, const float* sink, int64_t B, int64_t H, int64_t kv_heads, int64_t maps, int64_t dn, int64_t dr,
                               int64_t dv, int64_t window, int64_t keep, int64_t max_q, float scale, float lam, float gain, float eps, int64_t f32,
                               int64_t mfma, void* stream) {
    if (!q || !kn || !v || !o || !cu_q || !cu_k || B <= 0 || B > 65535 || H <= 0 || H > 65535 || kv_heads <= 0 || H % kv_heads != 0) return -1;
    if (dn < 0 || dr < 0 || (dr > 0 && !kr) || dn + dr <= 0 || dn + dr > 8192 || dv <= 0 || dv > 512 || window <= 0 || keep < 0 || max_q <= 0 || max_q > 0x3fffffff) return -1;
    if ((maps != 1 && maps != 2) || (maps == 2 && (dr > 0 || sink)) || ldq < H * maps * (dn + dr) || ldkv < kv_heads * dv || ldkv < kv_heads * maps * dn) return -1;
    const int w = window > 0x3fffffff ? 0x3fffffff : (int)window, kp = keep > 0x3fffffff ? 0x3fffffff : (int)keep;
    WinArgs a = {q, kn, v, kr, o, cu_q, cu_k, sink, ldq, ldkv, (int)H, (int)(H / kv_heads), (int)dn, (int)dr, (int)dv, w, kp, 0, scale, lam, gain, eps};
    hipStream_t s = (hipStream_t)stream;
    const int64_t dq = dn + dr;
    if (!f32 && mfma && dq <= (maps == 2 ? 128 : 256) && dv <= 256) {
        const bool vec = dn % 8 == 0 && dr % 8 == 0 && dv % 8 == 0 && ldq % 8 == 0 && ldkv % 8 == 0 && ldkv <= 0xffffff &&
                         (((uintptr_t)q | (uintptr_t)kn | (uintptr_t)v | (uintptr_t)kr) & 15) == 0;
        // (more than one block of queries of the workgroups below, head sizes of their swizzles, a positive scale: the maximum is taken before it;
        //  two maps without a window: at its lower edge a block of 32 queries reaches 16 keys further than one of 16)
        if (vec && max_q > 128 && scale > 0.f && dn == 128 && ((dr == 64 && dv == 128 && !kp && maps == 1) || (dr == 0 && (maps == 1 ? dv == 128 : dv == 256 && !kp && w >= 1 << 29)))) {
            a.n_qb = (int)(maps == 2 ? (max_q + 31 + 127) / 128 : (max_q + 255) / 256);
            const int64_t items = (int64_t)a.n_qb * H * B;
            if (items <= 0x7ffffff0) {
                const dim3 wg((unsigned)((items + 7) / 8 * 8)), wb(512);
                if (maps == 2) hipLaunchKernelGGL((window_tile_kernel<128, 0, 256, 2, false>), wg, wb, 0, s, a, (int)B);
                else if (dr) hipLaunchKernelGGL((window_tile_kernel<128, 64, 128, 1, false>), wg, wb, 0, s, a, (int)B);
                else if (kp) hipLaunchKernelGGL((window_tile_kernel<128, 0, 128, 1, true>), wg, wb, 0, s, a, (int)B);
                else hipLaunchKernelGGL((window_tile_kernel<128, 0, 128, 1, false>), wg, wb, 0, s, a, (int)B);
                return evo_launch_status();
            }
        }
#define WA1(KS, DVB, QC, VEC, KEEP, MAPS, MINW, NW)                                                                        \
    do {                                                                                                                   \
        a.n_qb = (int)((max_q + 16 * NW * QC / MAPS - 1) / (16 * NW * QC / MAPS));                                         \
        const int64_t items = (int64_t)a.n_qb * H * B;                                                                     \
        if (items > 0x7ffffff0) return -1;                                                                                 \
        hipLaunchKernelGGL((window_attn_kernel<KS, DVB, QC, VEC, KEEP, MAPS, MINW, NW, (MAPS == 2 && NW == 8 ? 2 : 1)>), dim3((unsigned)((items + 7) / 8 * 8)), dim3(64 * NW), 0, s, a, (int)B); \
    } while (0)
#define WAN(KS, DVB, QC, VEC, MAPS, MINW, NW) do { if (kp) WA1(KS, DVB, QC, VEC, true, MAPS, MINW, NW); else WA1(KS, DVB, QC, VEC, false, MAPS, MINW, NW); } while (0)
#define WA(KS, DVB, QC, VEC, MAPS, MINW) WAN(KS, DVB, QC, VEC, MAPS, MINW, 4)
#define WAV(KS, QC) do { if (dv <= 64) WA(KS, 4, QC, true, 1, 2); else if (dv <= 128) WA(KS, 8, QC, true, 1, 2); else WA(KS, 16, 1, true, 1, 2); } while (0)
#define WA2(KS) do { if (dv <= 64) WA(KS, 4, 2, true, 2, 2); else if (dv <= 128) WA(KS, 8, 2, true, 2, 2); \
                     else if (!kp) WA1(KS, 16, 2, true, false, 2, 2, 8); \
                     else WA1(KS, 16, 2, true, true, 2, (KS > 2 ? 1 : 2), (KS > 2 ? 4 : 8)); } while (0)   /* (kept tokens cost registers) */
        if (maps == 2) { if (!vec) WA(4, 16, 2, false, 2, 1); else if (dq <= 64) WA2(2); else WA2(4); }
        else if (!vec) { if (dq <= 64 && dv <= 64) WA(2, 4, 2, false, 1, 2); else WA(8, 16, 1, false, 1, 2); }
        else if (dq <= 64) WAV(2, 2);
        else if (dq <= 128) WAV(4, 2);
        else if (dq <= 192) {                                    // (kept tokens cost registers: one column block)
            if (dv <= 64) WA(6, 4, 2, true, 1, 2);
            else if (dv > 128) WA(6, 16, 1, true, 1, 2);
            else if (kp) WA1(6, 8, 1, true, true, 1, 2, 4);
            else WA1(6, 8, 2, true, false, 1, 2, 4);
        }
        else if (dv <= 64) WA(8, 4, 1, true, 1, 2);
        else if (dv <= 128) WA(8, 8, 1, true, 1, 2);
        else WA(8, 16, 1, true, 1, 1);
#undef WA2
#undef WAV
#undef WA
#undef WAN
#undef WA1
        return evo_launch_status();
    }
    if (f32 && mfma && dq <= (maps == 2 ? 128 : 256) && dv <= 256 && dn % 4 == 0 && dr % 4 == 0 && dv % 4 == 0 && ldq % 4 == 0 && ldkv % 4 == 0 &&
        (((uintptr_t)q | (uintptr_t)kn | (uintptr_t)v | (uintptr_t)kr | (uintptr_t)o) & 15) == 0) {
        a.n_qb = (int)((max_q + 63) / 64);
        if (a.n_qb * H > 0x7fffffff) return -1;
        const dim3 fgrid((unsigned)(a.n_qb * H), 1, (unsigned)B);
#define WF(KS, DVB, MAPS) hipLaunchKernelGGL((window_attn_f32_kernel<KS, DVB, MAPS>), fgrid, dim3(256), 0, s, a)
#define WFV(KS, MAPS) do { if (dv <= 64) WF(KS, 4, MAPS); else if (dv <= 128) WF(KS, 8, MAPS); else WF(KS, 16, MAPS); } while (0)
        if (maps == 2) { if (dq <= 64) WFV(4, 2); else WFV(8, 2); }
        else if (dq <= 64) WFV(4, 1);
        else if (dq <= 128) WFV(8, 1);
        else if (dq <= 192) WFV(12, 1);
        else WFV(16, 1);
#undef WFV
#undef WF
        return evo_launch_status();
    }
    const dim3 grid((unsigned)max_q, (unsigned)H, (unsigned)B);
#define WY(T, MAPS) hipLaunchKernelGGL((window_attn_any_kernel<T, MAPS>), grid, dim3(64), (size_t)dq * 4, s, a)
    if (f32) { if (maps == 2) WY(float, 2); else WY(float, 1); }
    else { if (maps == 2) WY(uint16_t, 2); else WY(uint16_t, 1); }
#undef WY
    return evo_launch_status();
}
