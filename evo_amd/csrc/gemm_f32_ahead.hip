// fp32 dense layers with the rows of x split ahead:  y [M, N] = x [M, K] w [N, K]^T (+ bias), the three bf16 parts and six products of gemm_f32.hip.
//
// What bounds a layer: from about 250 rows on the card's power (1.6 - 1.9 GHz of 2.4), below it also the 2 - 4 us of each launch around the products and a CU's
// intake.  gemm_f32.hip splits every row of x and of w once for each tile that it meets and passes both through registers into LDS: 32 % of the SIMDs' cycles
// beside 61 % of products.  Here one small launch splits x, in the order in which products take it, so that its parts come into LDS by themselves; a wave owns 32
// rows of w outright, brings them into LDS of its own as they are and splits them in registers for its own products, once per tile of up to 128 rows: 16 % of the
// cycles.  Products are 16 x 16 x 32 (half the sums read and written per product of 32 x 32 x 16, which drew 5 - 9 % more power), and the five small ones go to
// sums of their own (2^-8 of the large ones): a large sum is rounded once in 32 k, not 12 times.
// us, gemm_f32.hip -> here (MI355X, sweep of 19 row counts): 22,016 x 4,096 139 -> 116 at 80 rows, 234 -> 203 at 161, 359 -> 256 at 263, 629 -> 487 at 513, 1,131 -> 916 at
// 1,151, 1,784 -> 1,605 at 2,000; 4,096 x 11,008 86 -> 67, 121 -> 105, 188 -> 159, 316 -> 263, 604 -> 528, 880 -> 841; 4,096 x 4,096 82 -> 71 at 263, 227 -> 205 at 1,151.
// Error against 64 bits (random normal operands): K = 256 2.4e-7 -> 0.9e-7, 1,024 2.4e-7 -> 1.9e-7, 4,096 3.5e-7 -> 1.5e-7, 11,008 6.0e-7 -> 3.4e-7.
// Tried: waves side by side over 64 columns, one a SIMD (5 - 10 % slower: nothing hides its splitting); all six products into one sum (error as gemm_f32.hip's);
// sums of 32 k added by the vector units (12 % slower); the weight past the caches (half lines are fetched twice).
#include "gemm_f32.h"
#include "../../include/evo_mi355x.h"

#define FA_BN 256                            // columns of a tile: a wave per 32
#define FA_CHUNKS 16                         // parts of a row that the maxima are kept of

typedef uint32_t fa_u32x4 __attribute__((ext_vector_type(4)));

struct FaArgs {
    const float* x; const unsigned char* xs; const float* xmax; const float* w; const float* bias; float* y; float* parts;
    int64_t M; int N, K, Mp, tiles_m, tiles_n;
    int full, rest, shares;                  // tiles taken whole by a workgroup each; tiles shared out by their stages, and the workgroups that take a share each
};

// the first stage of share b, and the share that stage s belongs to (of all stages of the tiles shared out)
__host__ __device__ __forceinline__ int64_t fa_first(int64_t stages, int shares, int64_t b) { return stages * b / shares; }
__host__ __device__ __forceinline__ int fa_share(int64_t stages, int shares, int64_t s) { return (int)(((s + 1) * shares - 1) / stages); }

// tile -> row tile and column tile: eight row tiles next to each other before the next column tile
__device__ __forceinline__ void fa_tile(int tile, int tiles_m, int tiles_n, int& tm, int& tn) {
    const int per = 8 * tiles_n, g = tile / per, gsz = min(tiles_m - 8 * g, 8);
    tm = 8 * g + (tile - g * per) % gsz;
    tn = (tile - g * per) / gsz;
}

// ---------------------------------------------------------------------------------------------------------------- x ahead
// x -> xs [row block of 16][K / 32][h, m, l][lane][8 bf16], a lane's 16 bytes as a product takes them (lane = 16 quarter + row, k = 8 quarter .. + 7; rows behind
// the last are zeros), and xmax [FA_CHUNKS][Mp], the largest magnitude of a part of a row.
__global__ __launch_bounds__(256) void f32_split_kernel(const float* x, unsigned char* xs, float* xmax, int64_t M, int K, int Mp) {
    __shared__ float top[4][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lq = lane >> 4, l15 = lane & 15, n = K >> 5, c = blockIdx.x;
    const int64_t rb = blockIdx.y, row = rb * 16 + l15;
    const int s0 = (int)((int64_t)n * c / FA_CHUNKS), s1 = (int)((int64_t)n * (c + 1) / FA_CHUNKS);
    const float* src = x + (row < M ? row : 0) * K + lq * 8;
    unsigned char* dst = xs + rb * n * 3072 + lane * 16;
    float most = 0.f;
    for (int s = s0 + wave; s < s1; s += 4) {
        float4 a = *(const float4*)(src + s * 32), b = *(const float4*)(src + s * 32 + 4);
        if (row >= M) a = b = make_float4(0.f, 0.f, 0.f, 0.f);
        uint4 h, m, l;
        f3_split(a, b, h, m, l);
        f3_row_max(most, a, b);
        unsigned char* d = dst + (int64_t)s * 3072;
        *(uint4*)d = h;
        *(uint4*)(d + 1024) = m;
        *(uint4*)(d + 2048) = l;
    }
    most = fmaxf(most, __shfl_xor(most, 16, 64));
    most = fmaxf(most, __shfl_xor(most, 32, 64));
    if (lane < 16) top[wave][lane] = most;
    __syncthreads();
    if (threadIdx.x < 16) xmax[(int64_t)c * Mp + rb * 16 + threadIdx.x] = fmaxf(fmaxf(top[0][threadIdx.x], top[1][threadIdx.x]), fmaxf(top[2][threadIdx.x], top[3][threadIdx.x]));
}

// ---------------------------------------------------------------------------------------------------------------- products
// Outputs of a wave (16 TM rows, 32 columns) taken again with the fp32 matrix instructions, k-steps k0 .. k1 of 32: bit 8 i + 4 c + e of a lane's `odd` is
// column 16 c + 4 (lane / 16) + e of row 16 i + lane % 16.  A row block with a few of them: one after the other, the wave along k; with many: its whole product.
template <int TM>
__device__ __forceinline__ void fa_again(uint64_t odd, const float* x, const float* w, const float* bias, float* out, int64_t pitch, int64_t rows, int K, int k0, int k1) {
    const int lane = threadIdx.x & 63, lq = lane >> 4, l15 = lane & 15;
#pragma unroll 1
    for (int i = 0; i < TM; ++i) {
        const uint32_t mine = (uint32_t)(odd >> (8 * i)) & 255u;
        int n = __popc(mine);
#pragma unroll
        for (int d = 1; d < 64; d *= 2) n += __shfl_xor(n, d, 64);
        if (n == 0) continue;
        if (n <= 16) {
            for (uint64_t lanes = __builtin_amdgcn_ballot_w64(mine != 0); lanes; lanes &= lanes - 1) {
                const int owner = __builtin_ctzll(lanes);
                for (uint32_t bits = (uint32_t)__builtin_amdgcn_readlane((int)mine, owner); bits; bits &= bits - 1) {
                    const int b = __builtin_ctz(bits), r = i * 16 + (owner & 15), c = (b >> 2) * 16 + (owner >> 4) * 4 + (b & 3);
                    const float *xr = x + (int64_t)r * K, *wr = w + (int64_t)c * K;
                    float sum = 0.f;
#pragma unroll 4
                    for (int k = k0 * F3_BK + 4 * lane; k < k1 * F3_BK; k += 256) {
                        const f32x4_t u = *(const f32x4_t*)(xr + k), v = *(const f32x4_t*)(wr + k);
#pragma unroll
                        for (int e = 0; e < 4; ++e) sum = fmaf(u[e], v[e], sum);
                    }
                    sum = wave_sum(sum);
                    if (lane == owner) out[r * pitch + c] = bias ? sum + bias[c] : sum;
                }
            }
            continue;
        }
        const int64_t r = i * 16 + l15;
        const float* xr = x + (r < rows ? r : rows - 1) * K + lq * 4;
        const float* wr = w + (int64_t)l15 * K + lq * 4;
        f32x4_t sum[2] = {};
#pragma unroll 2
        for (int k = k0 * F3_BK; k < k1 * F3_BK; k += 16) {
            const f32x4_t u = *(const f32x4_t*)(xr + k), v0 = *(const f32x4_t*)(wr + k), v1 = *(const f32x4_t*)(wr + (int64_t)16 * K + k);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(v0[e], u[e], sum[0], 0, 0, 0);
                sum[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(v1[e], u[e], sum[1], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (mine >> b & 1) {                                 // (set only for rows that are there)
                const int c = (b >> 2) * 16 + lq * 4 + (b & 3);
                const float v = sum[b >> 2][b & 3];
                out[r * pitch + c] = bias ? v + bias[c] : v;
            }
    }
}

// Workgroup = BM = 16 TM rows x 256 columns of y, eight waves of 32 columns each in 16 x 16 x 32 products, D stages of 32 k ahead.
template <int TM, int D>
__global__ __launch_bounds__(512, 2) void gemm_f32_ahead_kernel(FaArgs a) {
    constexpr int CN = 2, NW = 8, BM = 16 * TM, NX = 3 * TM, PX = (NX + NW - 1) / NW, PW = 2 * CN, P = PX + PW, XS = NX * 1024, WS = 32768, XB = (D + 1) * XS;
    static_assert(TM >= 2 && TM <= 8 && D >= 2 && XB + D * WS <= 163840, "stages in LDS");
    __shared__ __attribute__((aligned(16))) unsigned char smem[XB + D * WS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lq = lane >> 4, l15 = lane & 15;
    // whole tiles first, the shares behind them; block b runs on XCD b % 8: every XCD gets a contiguous run of either
    const bool shared = (int)blockIdx.x >= a.full;
    const int nk = a.K / F3_BK, n_blocks = shared ? a.shares : a.full;
    int block;
    {
        const int bid = shared ? (int)blockIdx.x - a.full : (int)blockIdx.x, q = n_blocks >> 3, r = n_blocks & 7, xcd = bid & 7;
        block = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (bid >> 3);
    }
    const int64_t steps = (int64_t)a.rest * nk, s1 = shared ? fa_first(steps, a.shares, block + 1) : (int64_t)(block + 1) * nk;
    int64_t s0 = shared ? fa_first(steps, a.shares, block) : (int64_t)block * nk;
    const int64_t first = s0;

    const uint32_t kx = (uint32_t)a.K * 96u;                     // bytes of a row block of xs
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    // a piece of w: 8 rows of 128 B, granule g of 16 bytes of row r at slot g ^ (r & 7)
    const uint32_t wv = (uint32_t)(lane >> 3) * (uint32_t)a.K * 4u + (((lane & 7) ^ (lane >> 3)) & 7) * 16u;
    uint32_t xv[PX], xd[PX];
#pragma unroll
    for (int p = 0; p < PX; ++p) {
        const int i = min(wave + NW * p, NX - 1);               // (the last piece more than once: the same bytes)
        xv[p] = (uint32_t)(i / 3) * kx + (uint32_t)(i % 3) * 1024u + lane * 16;
        xd[p] = lds0 + i * 1024;
    }
    const uint32_t wd = lds0 + XB + wave * 4096;
    const uint32_t wr[2] = {(uint32_t)(XB + wave * 4096 + l15 * 128 + (((2 * lq) ^ l15) & 7) * 16), (uint32_t)(XB + wave * 4096 + l15 * 128 + (((2 * lq + 1) ^ l15) & 7) * 16)};

#pragma unroll 1
    while (s0 < s1) {                                            // (a share holds stages of one tile or of two)
        const int t = (int)(s0 / nk), tile = (shared ? a.full : 0) + t;
        const int64_t end = min(s1, (int64_t)(t + 1) * nk);
        const int k0 = (int)(s0 - (int64_t)t * nk), k1 = (int)(end - (int64_t)t * nk);
        const bool whole = k1 - k0 == nk;
        int tm, tn;
        fa_tile(tile, a.tiles_m, a.tiles_n, tm, tn);
        const int64_t m0 = (int64_t)tm * BM;
        const int n0 = tn * FA_BN + wave * 32;
        const uint64_t xa = (uint64_t)a.xs + (uint64_t)tm * TM * kx, wa = (uint64_t)(a.w + (int64_t)n0 * a.K);
        const int64_t blocks = (a.Mp >> 4) - (int64_t)tm * TM;   // (row blocks behind the last: past the descriptor's end, zeros; so are columns behind the last)
        const fa_u32x4 rx = {(uint32_t)xa, (uint32_t)(xa >> 32) & 0xffffu, (uint32_t)min(blocks, (int64_t)TM) * kx, 0x00020000u};
        const fa_u32x4 rw = {(uint32_t)wa, (uint32_t)(wa >> 32) & 0xffffu, n0 < a.N ? 128u * (uint32_t)a.K : 0u, 0x00020000u};
        // stages in turn from one of the tile's own on; behind the last one it again, into a slot nobody reads
        int at_x = k0 + (int)((uint32_t)tn * 2u % (uint32_t)(k1 - k0)), left_x = k1 - k0, at_w = at_x, left_w = left_x;
        auto fetch_w = [&](uint32_t slot) {
#pragma unroll
            for (int j = 0; j < PW; ++j)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(wd + slot + j * 1024), "v"(wv + (uint32_t)j * 32u * (uint32_t)a.K), "s"(rw), "s"((uint32_t)at_w * 128u) : "memory", "m0");
            if (--left_w > 0) at_w = at_w + 1 < k1 ? at_w + 1 : k0;
        };
        auto fetch_x = [&](uint32_t slot) {
#pragma unroll
            for (int p = 0; p < PX; ++p)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(xd[p] + slot), "v"(xv[p]), "s"(rx), "s"((uint32_t)at_x * 3072u) : "memory", "m0");
            if (--left_x > 0) at_x = at_x + 1 < k1 ? at_x + 1 : k0;
        };

        f32x4_t acc[TM][CN], low[TM][CN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int c = 0; c < CN; ++c) acc[i][c] = low[i][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        float top[CN] = {};                                     // the largest of this lane's values of its rows of w
        bf16x8_t wf[2][CN][3], xf[2][3];
        float4 raw[CN][2];
        auto load_raw = [&](uint32_t slot) {
#pragma unroll
            for (int c = 0; c < CN; ++c)
#pragma unroll
                for (int e = 0; e < 2; ++e) raw[c][e] = *(const float4*)(smem + slot + wr[e] + c * 2048);
        };
        auto split = [&](int c, bf16x8_t (&f)[3]) {
            uint4 h, m, l;
            f3_split(raw[c][0], raw[c][1], h, m, l);
            f3_row_max(top[c], raw[c][0], raw[c][1]);
            f[0] = __builtin_bit_cast(bf16x8_t, h);
            f[1] = __builtin_bit_cast(bf16x8_t, m);
            f[2] = __builtin_bit_cast(bf16x8_t, l);
        };
        auto read = [&](uint32_t slot, int i, bf16x8_t (&f)[3]) {
#pragma unroll
            for (int p = 0; p < 3; ++p) f[p] = *(const bf16x8_t*)(smem + slot + (i * 3 + p) * 1024 + lane * 16);
        };
        fetch_w(0);
#pragma unroll
        for (int s = 1; s < D; ++s) { fetch_w(s * WS); fetch_x((s - 1) * XS); }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * P) : "memory");
        load_raw(0);
#pragma unroll
        for (int c = 0; c < CN; ++c) split(c, wf[0][c]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        fetch_w(0);
        fetch_x((D - 1) * XS);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * P) : "memory");
        asm volatile("s_barrier" ::: "memory");
        read(0, 0, xf[0]);
        uint32_t slot = 0, nslot = XS, fslot = D * XS, wslot = WS;      // x of this stage, of the next, to be filled; w of the next stage
        for (int k = k0; k < k1; ++k) {
            load_raw(wslot);
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                if (i == TM - 1) {                               // x of the next stage and w of the one behind it have landed, everyone has read the x before this
                    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 2) * P) : "memory");
                    asm volatile("s_barrier" ::: "memory");
                    fetch_w(wslot);
                    fetch_x(fslot);
                }
                read(i + 1 < TM ? slot : nslot, (i + 1) % TM, xf[(i + 1) & 1]);
#pragma unroll
                for (int c = 0; c < CN; ++c)
                    if (c * (TM - 1) / CN == i) split(c, wf[1][c]);
                if ((CN - 1) * (TM - 1) / CN == i) asm volatile("" ::"v"(raw[CN - 1][1].w));     // (the reads of the slot that is filled next are done)
                constexpr int PX_[5] = {0, 2, 1, 0, 1}, PW_[5] = {2, 0, 1, 1, 0};            // the smallest products first
#pragma unroll
                for (int q = 0; q < 5; ++q)
#pragma unroll
                    for (int c = 0; c < CN; ++c) low[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[0][c][PW_[q]], xf[i & 1][PX_[q]], low[i][c], 0, 0, 0);
#pragma unroll
                for (int c = 0; c < CN; ++c) acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[0][c][0], xf[i & 1][0], acc[i][c], 0, 0, 0);
            }
#pragma unroll
            for (int p = 0; p < 3; ++p) {
#pragma unroll
                for (int c = 0; c < CN; ++c) wf[0][c][p] = wf[1][c][p];
                if (TM & 1) xf[0][p] = xf[1][p];
            }
            fslot = slot;
            slot = nslot;
            nslot = nslot + XS == XB ? 0 : nslot + XS;
            wslot = wslot + WS == D * WS ? 0 : wslot + WS;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int c = 0; c < CN; ++c) acc[i][c] += low[i][c];
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");      // (the stages fetched again land before the LDS is used for other things)
        __syncthreads();
        float *x_max = (float*)smem, *w_max = x_max + BM + wave * 32;        // (a row of zeros: -inf, which no output is under)
#pragma unroll
        for (int c = 0; c < CN; ++c) {
            top[c] = fmaxf(top[c], __shfl_xor(top[c], 16, 64));
            top[c] = fmaxf(top[c], __shfl_xor(top[c], 32, 64));
            if (lq == 0) w_max[c * 16 + l15] = top[c] > 0.f ? top[c] : -INFINITY;
        }
        if (tid < BM) {
            float most = 0.f;
            if (m0 + tid < a.M) {
#pragma unroll
                for (int c = 0; c < FA_CHUNKS; ++c) most = fmaxf(most, a.xmax[(int64_t)c * a.Mp + m0 + tid]);
            }
            x_max[tid] = most > 0.f ? most : -INFINITY;
        }
        __syncthreads();
        if (n0 < a.N) {
            // a part of a tile: its workgroup's first piece in the place of the share, a second one in the place of the tile
            float* out = whole ? a.y + m0 * a.N + n0 : a.parts + (int64_t)(s0 == first ? block : a.shares + t) * (BM * FA_BN) + wave * 32;
            const int64_t pitch = whole ? a.N : FA_BN;
            const float* bias = whole && a.bias ? a.bias + n0 : nullptr;
            const float least = (float)(k1 - k0) * (F3_BK * 0x1p-98f);
            float wide[CN][4];
#pragma unroll
            for (int c = 0; c < CN; ++c)
#pragma unroll
                for (int e = 0; e < 4; ++e) wide[c][e] = w_max[c * 16 + lq * 4 + e];
            uint64_t odd = 0;                                    // outputs to be taken again: 4 CN bits of each row block
#pragma unroll
            for (int i = 0; i < TM; ++i) {
                const int r = i * 16 + l15;
                if (m0 + r >= a.M) continue;
                const float bound = fmaf(least, x_max[r], least);
#pragma unroll
                for (int c = 0; c < CN; ++c) {
                    float4 v = make_float4(acc[i][c][0], acc[i][c][1], acc[i][c][2], acc[i][c][3]);
                    const float u[4] = {fabsf(v.x), fabsf(v.y), fabsf(v.z), fabsf(v.w)};
#pragma unroll
                    for (int e = 0; e < 4; ++e) odd |= (uint64_t)(u[e] >= fmaf(least, wide[c][e], bound) && u[e] <= 3.402823466e38f ? 0 : 1) << (i * 4 * CN + c * 4 + e);
                    if (bias) { const float4 b = *(const float4*)(bias + c * 16 + lq * 4); v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w; }
                    *(float4*)(out + r * pitch + c * 16 + lq * 4) = v;
                }
            }
            if (__builtin_amdgcn_ballot_w64(odd != 0)) fa_again<TM>(odd, a.x + m0 * a.K, a.w + (int64_t)n0 * a.K, bias, out, pitch, a.M - m0, a.K, k0, k1);
        }
        s0 = end;
        if (s0 < s1) __syncthreads();
    }
}

// the sums of the tiles that were taken in parts
__global__ __launch_bounds__(256) void f32_ahead_parts_kernel(FaArgs a, int bm) {
    const int t = blockIdx.y, nk = a.K / F3_BK;
    const int64_t steps = (int64_t)a.rest * nk;
    const int b0 = fa_share(steps, a.shares, (int64_t)t * nk), b1 = fa_share(steps, a.shares, (int64_t)(t + 1) * nk - 1);
    if (b0 == b1) return;                                        // one share's
    int tm, tn;
    fa_tile(a.full + t, a.tiles_m, a.tiles_n, tm, tn);
    const int i = blockIdx.x * 1024 + threadIdx.x * 4;
    const int64_t m = (int64_t)tm * bm + i / FA_BN;
    const int n = tn * FA_BN + i % FA_BN;
    if (m >= a.M || n >= a.N) return;
    const bool second = fa_first(steps, a.shares, b0) < (int64_t)t * nk;
    float4 v = *(const float4*)(a.parts + (int64_t)(second ? a.shares + t : b0) * bm * FA_BN + i);
#pragma unroll 4
    for (int b = b0 + 1; b <= b1; ++b) {
        const float4 u = *(const float4*)(a.parts + (int64_t)b * bm * FA_BN + i);
        v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
    }
    if (a.bias) { const float4 b = *(const float4*)(a.bias + n); v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w; }
    *(float4*)(a.y + m * a.N + n) = v;
}

template <int TM, int D>
static int fa_launch(const FaArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((gemm_f32_ahead_kernel<TM, D>), dim3((unsigned)(a.full + a.shares)), dim3(512), 0, st, a);
    return evo_launch_status();
}

static bool fa_ok(int64_t M, int64_t N, int64_t K) {
    return M >= 1 && N >= 32 && K >= 256 && M <= 0xffff0 && N <= 0x7fffff00 && K <= 0x1fffff && N % 32 == 0 && K % 32 == 0 && (double)M * N <= 4e11;
}

// Which tile, and how many tiles are shared out.  A stage of a tile of 16 tm rows takes a CU 0.68 + 0.168 tm us; all CUs together no less than
// (0.58 + 0.202 tm) / CUs a stage (power), and a weight no less than its bytes at 4.3 TB/s.  Tiles behind the last whole round are cut into as many shares as there
// are CUs (or fewer): a share costs 2.7 us, its sums go through memory at 6 TB/s, and as shares of neighbouring tiles are at different k, their operands come from
// beyond the L2 at 6.5 TB/s in all.  Fitted to 190 layers of 33 to 3,000 rows (within 6 % in the mean; the plan taken is 1.8 % behind the best of those measured).
struct FaPlan { int tm; int64_t full, rest; int shares; double us; };
static FaPlan fa_plan(int64_t M, int64_t N, int64_t K) {
    static const int cus = [] {
        int dev = 0, c = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&c, hipDeviceAttributeMultiprocessorCount, dev);
        return c < 8 ? 8 : c;
    }();
    const int64_t rows = (M + 15) / 16, nk = K / F3_BK, tiles_n = (N + FA_BN - 1) / FA_BN;
    const double memory = (double)N * K * 4 / 4.3e6, ahead = 4.8 + (double)rows * 16 * K * 10 / 6e6;
    FaPlan best = {0, 0, 0, 0, 1e300};
    for (int tm = 2; tm <= 8; ++tm) {
        const int64_t tiles_m = (rows + tm - 1) / tm, tiles = tiles_m * tiles_n;
        if (tm > 2 && (rows + tiles_m - 1) / tiles_m < tm) continue;         // (a smaller tile takes no more of them)
        const double step = 0.68 + 0.168 * tm, power = (double)tiles * nk * (0.58 + 0.202 * tm) / cus + 6.3;
        auto consider = [&](int64_t full, int shares) {
            const int64_t rest = tiles - full;
            double busy = 0;
            if (full) busy += (double)((full + cus - 1) / cus) * (nk * step + 2.7);
            if (shares)
                busy += fmax((double)((shares + cus - 1) / cus) * ((double)rest * nk / shares * step + 2.7 * (1 + (double)rest / shares)),
                             (double)rest * nk * (32768 + 3072 * tm) / 6.5e6);
            double us = ahead + fmax(fmax(busy, power), memory);
            if (shares) us += 2.0 + (double)(shares + rest) * tm * 16384 * 2 / 6.0e6;
            if (us < best.us) best = {tm, full, rest, shares, us};
        };
        const int64_t full = tiles / cus * cus, rest = tiles - full;
        if (tiles >= cus / 2 || nk < 8) consider(tiles, 0);
        if (rest)
            for (int q = 1; q <= 4; ++q) {
                const int shares = cus * q / 4;
                if (shares > rest && shares <= rest * nk / 4) consider(full, shares);
            }
        if (best.tm == 0) consider(tiles, 0);
    }
    return best;
}

static int64_t fa_bytes(const FaPlan& p, int64_t M, int64_t K) {
    const int64_t Mp = (M + 15) / 16 * 16;
    return Mp * K * 6 + FA_CHUNKS * Mp * 4 + (p.shares ? (p.shares + p.rest) * p.tm * 16 * FA_BN * 4 : 0);
}

// Taken where its time is the shorter one: weights under 12 M values mostly stay with gemm_f32.hip (1,024 x 4,096: 55 us there at 800 rows, 53 - 61 here).  Above 200 us
// that form's estimate is some 10 % short, below 100 us both are good to 4 % (1,151 x 4,096 x 11,008: 521 for 604); weights of few tiles are faster there up to 128 rows (6,720 x 4,096: 60 -> 66 at 128,
// 55 -> 58 at 96; 8,192 x 4,096 75 -> 64 and 60 -> 56), and 49 to 64 rows are its own tile (59 x 22,016 x 4,096 114 -> 126; 48 rows 105 -> 92, 67 rows 137 -> 106).
extern "C" int evo_linear_f32_ahead_plan(int64_t M, int64_t N, int64_t K, int64_t* out) {
    if (!fa_ok(M, N, K) || !out) return -1;
    const FaPlan p = fa_plan(M, N, K);
    const int64_t row[6] = {p.tm * 16, FA_BN, p.full, p.rest, p.shares, fa_bytes(p, M, K)};
    for (int i = 0; i < 6; ++i) out[i] = row[i];
    return row[5] <= 1ll << 30 && (M > 128 || (N * K >= 32000000 && (M > 64 || M <= 48))) && p.us < (p.us > 200.0 ? 1.1 : p.us < 100.0 ? 0.96 : 1.0) * f3_tiles_us(M, N, K) ? 1 : 0;
}

extern "C" int evo_linear_f32_ahead(const float* x, const float* w, const float* bias, float* y, int64_t M, int64_t N, int64_t K, void* ws, int64_t ws_bytes, void* stream) {
    if (M == 0) return 0;
    if (!fa_ok(M, N, K)) return -1;
    const FaPlan p = fa_plan(M, N, K);
    if (!x || !w || !y || !ws || ws_bytes < fa_bytes(p, M, K) || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)bias | (uintptr_t)y | (uintptr_t)ws) & 15)) return -1;
    const int64_t Mp = (M + 15) / 16 * 16, tiles_m = (M + 16 * p.tm - 1) / (16 * p.tm), tiles_n = (N + FA_BN - 1) / FA_BN;
    if (p.full + p.shares > 0x7fffffff || tiles_m * tiles_n > 0x7fffffff) return -1;
    hipStream_t st = (hipStream_t)stream;
    unsigned char* xs = (unsigned char*)ws;
    float* xmax = (float*)(xs + Mp * K * 6);
    const FaArgs a = {x, xs, xmax, w, bias, y, xmax + FA_CHUNKS * Mp, M, (int)N, (int)K, (int)Mp, (int)tiles_m, (int)tiles_n, (int)p.full, (int)p.rest, p.shares};
    hipLaunchKernelGGL(f32_split_kernel, dim3(FA_CHUNKS, (unsigned)(Mp / 16)), dim3(256), 0, st, x, xs, xmax, M, (int)K, (int)Mp);
    int rc = evo_launch_status();
    if (rc) return rc;
    switch (p.tm) {                                              // (stages ahead: as many as fit the CU's LDS)
        case 2: rc = fa_launch<2, 4>(a, st); break;
        case 3: rc = fa_launch<3, 3>(a, st); break;
        case 4: rc = fa_launch<4, 3>(a, st); break;
        case 5: rc = fa_launch<5, 3>(a, st); break;
        case 6: rc = fa_launch<6, 2>(a, st); break;
        case 7: rc = fa_launch<7, 2>(a, st); break;
        default: rc = fa_launch<8, 2>(a, st); break;
    }
    if (rc || !p.shares) return rc;
    hipLaunchKernelGGL(f32_ahead_parts_kernel, dim3((unsigned)(p.tm * 16 * FA_BN / 1024), (unsigned)p.rest), dim3(256), 0, st, a, p.tm * 16);
    return evo_launch_status();
}
