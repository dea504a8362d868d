// Dense layer on the MFMA pipe, hand-written for gfx950:  Y[M,N] = X[M,K] . W[N,K]^T (+ bias[N]) (+ R[M,N])
// bf16 in, fp32 accumulate, one bf16 rounding.  Both operands are K-contiguous (activations row-major, nn.Linear
// weights [out, in]), so both tiles are plain row slabs.
//
// Workgroup = 8 waves = one 256(M) x 256(N) output tile, K walked in steps of 64; wave (wm, wn) of a 2 x 4 grid
// owns 128(M) x 64(N) = 4 x 2 MFMA tiles of v_mfma_f32_32x32x16_bf16, computed TRANSPOSED (A operand = W rows,
// B operand = X rows) so that a lane's accumulator registers run along N: the epilogue adds bias / residual and
// stores 4 consecutive bf16 (8 bytes) per register group instead of scattering single elements.
//
// Data path.  Operand slabs (256 rows x 128 B = 32 KiB each, one cache line per row) arrive by asynchronous
// global->LDS DMA (global_load_lds_dwordx4) into a ring of FIVE slab slots = all 160 KiB of the CU's LDS; the slab
// sequence is X0 W0 X1 W1 ...  Two slabs are being read, three are in flight.  One raw s_barrier per k-step sits
// between its 3rd and 4th 16-deep sub-step; fragments are double-buffered in registers, so the first fragments of
// the next stage are read right behind the barrier, under the last sub-step of the current one.  The DMA
// instructions are spread between the MFMAs (one per two MFMAs): a burst of 64 KiB right behind the barrier blocks
// every wave on the vector-memory issue queue for ~750 cycles per k-step (measured, independent of data latency).
// LDS rows are XOR-swizzled (granule g of row r at slot g ^ ((r >> 1) & 7)): ds_read_b128 fragment reads are
// bank-conflict free (SQ_LDS_BANK_CONFLICT = 0) and the DMA stays lane-linear on the LDS side.
//
// Everything the compiler would otherwise serialise is inline asm with hand-counted waits: it answers any visible
// LDS-DMA with s_waitcnt vmcnt(0) before the next LDS read, and puts an lgkmcnt wait in front of every other MFMA.
// Workgroups are numbered so that each XCD (private L2) sweeps a contiguous,
// group_m-rastered range of output tiles.
// Entry point and reference citation: include/evo_mi355x.h.
#include <stdlib.h>
#include "gemm_kernel.h"
#include "../../include/evo_mi355x.h"

template <bool BIAS, bool RES>
__global__ __launch_bounds__(512, 1) void gemm_bf16_kernel(GemmArgs a) {
    __shared__ __attribute__((aligned(16))) unsigned char smem[G_NSLOT * G_SLAB];   // the ONLY __shared__ object
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    const int l31 = lane & 31;
    const int wm = wave >> 2, wn = wave & 3;                     // 2 x 4 wave grid

    // XCD-aware tile id: block b runs on XCD b % 8; give every XCD a contiguous run of tiles (bijective for any count)
    int tile;
    {
        const int bid = blockIdx.x, nt = a.n_tiles;
        const int q = nt >> 3, r = nt & 7, xcd = bid & 7, slot = bid >> 3;
        tile = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + slot;
    }
    // grouped raster: consecutive tile ids walk group_m row tiles before the next column tile, so the ~32 tiles an XCD
    // runs at once share group_m X panels and 32/group_m W panels in its L2 instead of 1 + 32
    int tm, tn;
    {
        const int per_group = a.group_m * a.tiles_n;
        const int grp = tile / per_group, in_grp = tile - grp * per_group;
        const int first_m = grp * a.group_m;
        const int gsz = a.tiles_m - first_m < a.group_m ? a.tiles_m - first_m : a.group_m;
        tn = in_grp / gsz;
        tm = first_m + in_grp - tn * gsz;
    }
    const int64_t m0 = (int64_t)tm * GBM;
    const int n0 = tn * GBN;
    const int64_t kb = (int64_t)a.K * 2;                         // bytes per operand row
    const int nk = a.K / GBK;

    // ---- DMA plan: a slab is 32 one-KiB pieces (8 rows each), 4 per wave.  The LDS side of a DMA is lane-linear, so
    //      the swizzle is applied to the global source: the lane that fills slot s of row r fetches granule
    //      s ^ ((r >> 1) & 7) -- still the same 128-byte line.
    const unsigned char* srcx[G_NP];
    const unsigned char* srcw[G_NP];
#pragma unroll
    for (int jj = 0; jj < G_NP; ++jj) {
        const int pos = (wave + 8 * jj) * 1024 + 16 * lane;
        const int r = pos / G_ROW;
        const int col = ((((pos - r * G_ROW) >> 4) ^ (r >> 1)) & 7) * 16;
        int64_t m = m0 + r;
        if (m > a.M - 1) m = a.M - 1;                            // ragged last M tile: clamp (rows never stored)
        srcx[jj] = a.x + m * kb + col;
        srcw[jj] = a.w + (int64_t)(n0 + r) * kb + col;
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
    const uint32_t lds_dma = lds0 + wave * 1024;
    // one piece of slab `H` (even: X of stage H/2, odd: W of stage H/2) -> slot H % 5.  Past the last stage the same
    // instruction re-fetches the last stage into a slot nobody reads: the loop stays branch-free and the vmcnt counts
    // stay constant.
#define G_DMA(SRC, H, JJ)                                                                                     \
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"                             \
                 ::"s"(lds_dma + ((H) % G_NSLOT) * G_SLAB + (JJ) * 8192),                                     \
                   "v"((SRC)[JJ] + (int64_t)(((H) >> 1) < nk ? ((H) >> 1) : nk - 1) * (GBK * 2)) : "memory", "m0")

    // fragment bases (within a slab): B operand = X rows (m), A operand = W rows (n).  Rows 32 apart share
    // (row >> 1) & 7, so one base per k-substep serves all of a wave's tiles (tile offsets are immediates).
    uint32_t x_rd[4], w_rd[4];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
        const int xr = wm * 128 + l31, wr = wn * 64 + l31;
        x_rd[ks] = lds0 + (uint32_t)(xr * G_ROW + (((2 * ks + half) ^ (xr >> 1)) & 7) * 16);
        w_rd[ks] = lds0 + (uint32_t)(wr * G_ROW + (((2 * ks + half) ^ (wr >> 1)) & 7) * 16);
    }

    f32x16_t acc[2][4];                                          // [n tile][m tile]
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    g_u32x4 wf[2][2], xf[2][4];                                  // double-buffered fragments

    // fragments of sub-step KS of the stage whose X / W slabs sit at byte offsets XO / WO
#define G_READ(XO, WO, KS, BUF)                                                                               \
    {                                                                                                         \
        const uint32_t wa_ = (WO) + w_rd[KS], xa_ = (XO) + x_rd[KS];                                          \
        G_DSR(wf[BUF][0], wa_, 0); G_DSR(wf[BUF][1], wa_, 32 * G_ROW);                                        \
        G_DSR(xf[BUF][0], xa_, 0); G_DSR(xf[BUF][1], xa_, 32 * G_ROW);                                        \
        G_DSR(xf[BUF][2], xa_, 64 * G_ROW); G_DSR(xf[BUF][3], xa_, 96 * G_ROW);                               \
    }
    // one counted wait per sub-step, tied to the fragment registers it guards
#define G_LGKM(N, BUF)                                                                                        \
    asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(wf[BUF][0]), "+v"(wf[BUF][1]), "+v"(xf[BUF][0]), "+v"(xf[BUF][1]), \
                 "+v"(xf[BUF][2]), "+v"(xf[BUF][3]) : "n"(N))
    // (the MFMA itself stays a builtin: the compiler must see it to place the MFMA -> accumulator-read wait states)
#define G_MFMA(I, J, BUF)                                                                                     \
    acc[I][J] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, wf[BUF][I]),             \
                                                        __builtin_bit_cast(bf16x8_t, xf[BUF][J]), acc[I][J], 0, 0, 0)
#define G_DMA_PIN(SRC, H, JJ)                                                                                 \
    {                                                                                                         \
        __builtin_amdgcn_sched_barrier(0);                                                                    \
        G_DMA(SRC, H, JJ);                                                                                    \
        __builtin_amdgcn_sched_barrier(0);                                                                    \
    }
    // eight MFMAs of one sub-step with up to four DMA pieces between them (piece index < 0: none)
#define G_MMA_DMA(BUF, SRC, H, JA, JB, JC, JD)                                                                \
    {                                                                                                         \
        G_MFMA(0, 0, BUF); G_MFMA(0, 1, BUF);                                                                 \
        if ((JA) >= 0) G_DMA_PIN(SRC, H, (JA) < 0 ? 0 : (JA));                                                    \
        G_MFMA(0, 2, BUF); G_MFMA(0, 3, BUF);                                                                 \
        if ((JB) >= 0) G_DMA_PIN(SRC, H, (JB) < 0 ? 0 : (JB));                                                    \
        G_MFMA(1, 0, BUF); G_MFMA(1, 1, BUF);                                                                 \
        if ((JC) >= 0) G_DMA_PIN(SRC, H, (JC) < 0 ? 0 : (JC));                                                    \
        G_MFMA(1, 2, BUF); G_MFMA(1, 3, BUF);                                                                 \
        if ((JD) >= 0) G_DMA_PIN(SRC, H, (JD) < 0 ? 0 : (JD));                                                    \
    }

    // ---- pipeline.  Slab h (even: X of stage h/2, odd: W) lives in slot h % 5.  Iteration k:
    //        sub-steps 0,1   MFMAs(k,0..1)  + DMA X(k+2) (slab 2k+4: its slot was freed by barrier k-1)
    //        sub-step  2     MFMAs(k,2)
    //        wait            own pieces of stage k+1 (slabs 2k+2, 2k+3) retired: vmcnt(4) leaves X(k+2) in flight   [RAW]
    //                        lgkmcnt(0): this wave's last reads of stage k retired                                  [WAR]
    //        barrier k       stage k+1 visible to all; slots of slabs 2k, 2k+1 free
    //        sub-step  3     first fragments of stage k+1 are read; MFMAs(k,3) + DMA W(k+2) (slab 2k+5 -> slot of X(k))
    //      A slab is re-filled only behind the barrier that follows the last read of its previous contents, and read
    //      only behind the barrier that follows its own counted vmcnt.
#pragma unroll
    for (int jj = 0; jj < G_NP; ++jj) G_DMA(srcx, 0, jj);
#pragma unroll
    for (int jj = 0; jj < G_NP; ++jj) G_DMA(srcw, 1, jj);
    if (nk > 1) {
#pragma unroll
        for (int jj = 0; jj < G_NP; ++jj) G_DMA(srcx, 2, jj);
#pragma unroll
        for (int jj = 0; jj < G_NP; ++jj) G_DMA(srcw, 3, jj);
        G_VMCNT(2 * G_NP);
    } else {
        G_VMCNT(0);
    }
    G_BARRIER();
    G_READ(0, G_SLAB, 0, 0);
    for (int k = 0; k + 1 < nk; ++k) {                           // (the last k-step is peeled)
        const uint32_t xo = ((2 * k) % G_NSLOT) * G_SLAB, wo = ((2 * k + 1) % G_NSLOT) * G_SLAB;
        G_READ(xo, wo, 1, 1);
        G_LGKM(6, 0);
        __builtin_amdgcn_sched_barrier(0);
        G_MMA_DMA(0, srcx, 2 * k + 4, -1, 0, -1, 1);
        __builtin_amdgcn_sched_barrier(0);
        G_READ(xo, wo, 2, 0);
        G_LGKM(6, 1);
        __builtin_amdgcn_sched_barrier(0);
        G_MMA_DMA(1, srcx, 2 * k + 4, -1, 2, -1, 3);
        __builtin_amdgcn_sched_barrier(0);
        G_READ(xo, wo, 3, 1);
        G_LGKM(6, 0);
        __builtin_amdgcn_sched_barrier(0);
        G_MMA_DMA(0, srcx, 0, -1, -1, -1, -1);
        __builtin_amdgcn_sched_barrier(0);
        G_LGKM(0, 1);                                            // sub-step 3's fragments: stage k is fully read
        G_VMCNT(G_NP);
        G_BARRIER();
        G_READ(((2 * k + 2) % G_NSLOT) * G_SLAB, ((2 * k + 3) % G_NSLOT) * G_SLAB, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        G_MMA_DMA(1, srcw, 2 * k + 5, 0, 1, 2, 3);
        __builtin_amdgcn_sched_barrier(0);
    }
    {
        const int k = nk - 1;
        const uint32_t xo = ((2 * k) % G_NSLOT) * G_SLAB, wo = ((2 * k + 1) % G_NSLOT) * G_SLAB;
        G_READ(xo, wo, 1, 1);
        G_LGKM(6, 0);
        G_MMA_DMA(0, srcx, 0, -1, -1, -1, -1);
        G_READ(xo, wo, 2, 0);
        G_LGKM(6, 1);
        G_MMA_DMA(1, srcx, 0, -1, -1, -1, -1);
        G_READ(xo, wo, 3, 1);
        G_LGKM(6, 0);
        G_MMA_DMA(0, srcx, 0, -1, -1, -1, -1);
        G_LGKM(0, 1);
        G_MMA_DMA(1, srcx, 0, -1, -1, -1, -1);
        G_VMCNT(0);                                              // (tail re-fetches: nothing may land after the LDS is released)
    }

    // ---- epilogue.  D[n][m]: a lane holds column m = lane & 31 and rows n = (r&3) + 8(r>>2) + 4*half, i.e. runs of four
    // consecutive n.  The wave transposes its 128 x 64 tile through its own 18 KiB of the (now idle) LDS -- rows of
    // 128 B + 16 B pad -- so that global traffic moves whole 128-byte row segments, 16 B per lane and eight lanes per
    // output row (the direct 8-byte scatter cost ~10 % of the kernel in partial-line accesses).  The residual tile
    // takes the same way in; bias and residual are added in fp32 before the one rounding.
    G_BARRIER();                                                 // every wave is done with the operand slabs
    {
        constexpr int PITCH = 144;
        unsigned char* tr = smem + wave * (128 * PITCH);
        const int rsub = lane >> 3, cseg = lane & 7;             // 8 rows x 8 segments of 16 B per pass
        const int nseg = n0 + wn * 64 + cseg * 8;
        if (RES) {                                               // residual tile -> LDS, coalesced
#pragma unroll 4
            for (int it = 0; it < 16; ++it) {
                const int row = it * 8 + rsub;
                const int64_t m = m0 + wm * 128 + row;
                uint4 r = make_uint4(0, 0, 0, 0);
                if (m < a.M) r = *(const uint4*)(a.res + m * a.N + nseg);
                *(uint4*)(tr + row * PITCH + cseg * 16) = r;
            }
        }
        asm volatile("" ::: "memory");       // (uint4 rows and uint2 cells are distinct types: keep the passes ordered)
        uint2 bpk[2][4];                                         // this lane's 32 bias values, packed
        if (BIAS) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) bpk[i][g] = *(const uint2*)(a.bias + n0 + wn * 64 + i * 32 + 8 * g + 4 * half);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)                              // one accumulator tile at a time (register pressure)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    unsigned char* cell = tr + (j * 32 + l31) * PITCH + (i * 32 + 8 * g + 4 * half) * 2;
                    float v[4] = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                    if (BIAS) {
                        v[0] += bf_lo(bpk[i][g].x); v[1] += bf_hi(bpk[i][g].x);
                        v[2] += bf_lo(bpk[i][g].y); v[3] += bf_hi(bpk[i][g].y);
                    }
                    if (RES) {
                        const uint2 r = *(const uint2*)cell;
                        v[0] += bf_lo(r.x); v[1] += bf_hi(r.x); v[2] += bf_lo(r.y); v[3] += bf_hi(r.y);
                    }
                    uint2 o;
                    o.x = pack_bf2(v[0], v[1]);                  // the one rounding
                    o.y = pack_bf2(v[2], v[3]);
                    *(uint2*)cell = o;
                }
        asm volatile("" ::: "memory");
#pragma unroll 4
        for (int it = 0; it < 16; ++it) {
            const int row = it * 8 + rsub;
            const int64_t m = m0 + wm * 128 + row;
            const uint4 o = *(const uint4*)(tr + row * PITCH + cseg * 16);
            if (m < a.M) *(uint4*)(a.y + m * a.N + nseg) = o;
        }
    }
}

extern "C" int evo_linear_mfma_bf16(const void* x, const void* w, const void* bias, const void* residual, void* y,
                                    int64_t M, int64_t N, int64_t K, void* stream) {
    return evo_linear_mfma_nf_bf16(x, w, bias, residual, y, nullptr, nullptr, 0, M, N, K, stream);
}

// The same dense layer with the RMSNorm around it folded in (gemmr_bf16_kernel, NF): `row_scale` [ceil(M / 256) * 256] fp32 multiplies the
// accumulators of row m before the bias (the consumer of a normalised stream: w is then W diag(g), no residual); `sumsq`
// [N / 128][ss_ld] fp32 (ss_ld >= ceil(M / 256) * 256) receives the sums of squares of the stored rows per 128-column strip (the
// producer of the stream: residual required).  Both need the persistent form's shape contract (K >= 128, operands < 4 GiB).
extern "C" int evo_linear_mfma_nf_bf16(const void* x, const void* w, const void* bias, const void* residual, void* y,
                                       const float* row_scale, float* sumsq, int64_t ss_ld, int64_t M, int64_t N, int64_t K, void* stream) {
    if (M <= 0 || N <= 0 || K <= 0 || N % GBN != 0 || K % GBK != 0 || N > 0x7fffffff / 2) return -1;
    if ((row_scale && (residual || sumsq)) || (sumsq && (!residual || ss_ld < (M + GBM - 1) / GBM * GBM))) return -1;
    if ((row_scale || sumsq) && !(K >= 2 * GBK && M * K * 2 < 0xffffffffll && N * K * 2 < 0xffffffffll)) return -1;
    GemmArgs a;
    a.rs = row_scale; a.ss = sumsq; a.ss_ld = ss_ld;
    a.x = (const unsigned char*)x; a.w = (const unsigned char*)w; a.bias = (const uint16_t*)bias;
    a.res = (const uint16_t*)residual; a.y = (uint16_t*)y;
    a.M = M; a.N = (int)N; a.K = (int)K;
    a.tiles_n = (int)(N / GBN);
    a.tiles_m = (int)((M + GBM - 1) / GBM);
    // raster width: the ~32 tiles an XCD runs at once cover group_m X panels x 32 / group_m W panels.  Measured on the four layer
    // shapes at M = 65,536 (tools/gemm_ab.py lib.so@G): N = 12,288 / 22,016: 8 is best (98.1 / 98.2 % of hipBLASLt against 97.6 /
    // 96.6 at 4, 88 at 16, 60 at 32); N = 4,096 (16 column tiles): 1-4 tie, 8 loses 1.5-2.5 %.
    const int group_m = (a.tiles_n >= 32 ? 8 : 4);
    a.group_m = group_m;
    const int64_t tiles = ((M + GBM - 1) / GBM) * a.tiles_n;
    if (tiles > 0x7fffffff) return -1;
    a.n_tiles = (int)tiles;
    const dim3 grid((unsigned)tiles), block(512);
    hipStream_t st = (hipStream_t)stream;
    static const int form = [] { const char* e = getenv("EVO_GEMM_FORM"); return e ? atoi(e) : 1; }();   // 1: persistent, 0: tile per workgroup
    if ((row_scale || sumsq) && form != 1) return -1;           // the folded norm exists in the persistent kernel only: never fall through to a launch that ignores it
    if (form == 1 && K >= 2 * GBK && M * K * 2 < 0xffffffffll && N * K * 2 < 0xffffffffll) {
        static const int n_cu = [] {
            int dev = 0, n = 256;
            if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
            n &= ~7;
            return n < 8 ? 8 : n;
        }();
        const dim3 gridp((unsigned)n_cu), block4(256);
        if (row_scale) {
            if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, false, 0, false, 2>), gridp, block4, 0, st, a);
            else hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 0, false, 2>), gridp, block4, 0, st, a);
            return evo_launch_status();
        }
        if (sumsq) {
            if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, true, 0, false, 1>), gridp, block4, 0, st, a);
            else hipLaunchKernelGGL((gemmr_bf16_kernel<false, true, 0, false, 1>), gridp, block4, 0, st, a);
            return evo_launch_status();
        }
        if (bias && residual) hipLaunchKernelGGL((gemmr_bf16_kernel<true, true, 0>), gridp, block4, 0, st, a);
        else if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, false, 0>), gridp, block4, 0, st, a);
        else if (residual) hipLaunchKernelGGL((gemmr_bf16_kernel<false, true, 0>), gridp, block4, 0, st, a);
        else hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 0>), gridp, block4, 0, st, a);
        return evo_launch_status();
    }
    if (bias && residual) hipLaunchKernelGGL((gemm_bf16_kernel<true, true>), grid, block, 0, st, a);
    else if (bias) hipLaunchKernelGGL((gemm_bf16_kernel<true, false>), grid, block, 0, st, a);
    else if (residual) hipLaunchKernelGGL((gemm_bf16_kernel<false, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((gemm_bf16_kernel<false, false>), grid, block, 0, st, a);
    return evo_launch_status();
}

// y [M, N] = act(x . w^T + bias) on columns [0, act_cols), without act behind them: input projections that activate some of their parts, and
// ungated feed-forwards.  act 1: SiLU, 2: GELU (tanh form), 3: square of relu; act_cols % 256 == 0; N % 256 == 0, K % 64 == 0, K >= 128,
// operands below 4 GiB.
extern "C" int evo_linear_act_mfma_bf16(const void* x, const void* w, const void* bias, void* y, int64_t M, int64_t N, int64_t K, int64_t act_cols,
                                        int64_t act, void* stream) {
    if (M <= 0 || N <= 0 || N % GBN != 0 || K % GBK != 0 || K < 2 * GBK || N > 0x7fffffff / 2 || act_cols < 0 || act_cols > N || act_cols % GBN != 0 || act < 1 || act > 3) return -1;
    if (M * K * 2 >= 0xffffffffll || N * K * 2 >= 0xffffffffll) return -1;
    GemmArgs a;
    a.x = (const unsigned char*)x; a.w = (const unsigned char*)w; a.bias = (const uint16_t*)bias; a.res = nullptr; a.y = (uint16_t*)y;
    a.M = M; a.N = (int)N; a.K = (int)K;
    a.act_cols = (int)act_cols;
    a.tiles_n = (int)(N / GBN);
    a.tiles_m = (int)((M + GBM - 1) / GBM);
    a.group_m = a.tiles_n >= 32 ? 8 : 4;
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    if (tiles > 0x7fffffff) return -1;
    a.n_tiles = (int)tiles;
    static const int n_cu = [] {
        int dev = 0, n = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        n &= ~7;
        return n < 8 ? 8 : n;
    }();
#define EVO_ACT(BIAS, ACT) hipLaunchKernelGGL((gemmr_bf16_kernel<BIAS, false, 0, false, 0, ACT>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a)
    if (bias) { if (act == 1) EVO_ACT(true, 1); else if (act == 2) EVO_ACT(true, 2); else EVO_ACT(true, 3); }
    else { if (act == 1) EVO_ACT(false, 1); else if (act == 2) EVO_ACT(false, 2); else EVO_ACT(false, 3); }
#undef EVO_ACT
    return evo_launch_status();
}

// y [M, N] = x . w^T (+ bias) (+ residual) with x in the BLOCKED layout the channel-stationary Hyena operator writes
// ([ceil(M / 128)][K / 16][128][16] bf16): the Hyena block's output projection [REF stripedhyena/model.py ParallelGatedConvBlock.forward:
// out_filter_dense].  M % 256 == 0 (the caller peels the BOS sliver), K % 64 == 0, K >= 128.
extern "C" int evo_linear_xblk_mfma_bf16(const void* x_blk, const void* w, const void* bias, const void* residual, void* y,
                                         int64_t M, int64_t N, int64_t K, void* stream) {
    return evo_linear_xblk_mfma_nf_bf16(x_blk, w, bias, residual, y, nullptr, 0, M, N, K, stream);
}

// ... and with the sums of squares of the stored rows (see evo_linear_mfma_nf_bf16; residual required when sumsq is given)
extern "C" int evo_linear_xblk_mfma_nf_bf16(const void* x_blk, const void* w, const void* bias, const void* residual, void* y,
                                            float* sumsq, int64_t ss_ld, int64_t M, int64_t N, int64_t K, void* stream) {
    if (sumsq && (!residual || ss_ld < M)) return -1;
    if (M <= 0 || M % GBM != 0 || N <= 0 || K <= 0 || N % GBN != 0 || K % GBK != 0 || K < 2 * GBK || N > 0x7fffffff / 2) return -1;
    if (M * K * 2 >= 0xffffffffll || N * K * 2 >= 0xffffffffll) return -1;
    GemmArgs a;
    a.x = (const unsigned char*)x_blk; a.w = (const unsigned char*)w; a.bias = (const uint16_t*)bias;
    a.res = (const uint16_t*)residual; a.y = (uint16_t*)y;
    a.ss = sumsq; a.ss_ld = ss_ld;
    a.M = M; a.N = (int)N; a.K = (int)K;
    a.tiles_n = (int)(N / GBN);
    a.tiles_m = (int)(M / GBM);
    a.group_m = a.tiles_n >= 32 ? 8 : 4;
    const int64_t tiles = (M / GBM) * a.tiles_n;
    if (tiles > 0x7fffffff) return -1;
    a.n_tiles = (int)tiles;
    static const int n_cu = [] {
        int dev = 0, n = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        n &= ~7;
        return n < 8 ? 8 : n;
    }();
    const dim3 gridp((unsigned)n_cu), block4(256);
    if (sumsq) {
        if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, true, 0, true, 1>), gridp, block4, 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL((gemmr_bf16_kernel<false, true, 0, true, 1>), gridp, block4, 0, (hipStream_t)stream, a);
        return evo_launch_status();
    }
    if (bias && residual) hipLaunchKernelGGL((gemmr_bf16_kernel<true, true, 0, true>), gridp, block4, 0, (hipStream_t)stream, a);
    else if (residual) hipLaunchKernelGGL((gemmr_bf16_kernel<false, true, 0, true>), gridp, block4, 0, (hipStream_t)stream, a);
    else if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, false, 0, true>), gridp, block4, 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 0, true>), gridp, block4, 0, (hipStream_t)stream, a);
    return evo_launch_status();
}

// Gated MLP, first half: a[M, I] = act(x W1^T) * (x W2^T), act = gelu (0) or silu (1), in ONE launch of the persistent kernel -- the [M, 2 I] intermediate
// never reaches memory [REF stripedhyena/layers.py ParallelGatedMLP.forward].  w12g = the rows of [W1; W2] regrouped as blocks
// of 64: 32 rows of W1 followed by the same 32 rows of W2 (evo_amd/ops.py pack_gate_weights), 2 I rows in all.
extern "C" int evo_mlp_gate_mfma_bf16(const void* x, const void* w12g, void* a_out, int64_t M, int64_t I, int64_t K, int64_t act, void* stream) {
    return gemmr_gate(x, nullptr, w12g, a_out, M, I, K, act, stream);
}

// ... with the post-mixer RMSNorm folded in: x = the residual stream itself, row_scale [ceil(M / 256) * 256] = 1 / (rms + eps) per row,
// w12g = the regrouped rows of [W1 diag(g); W2 diag(g)] (see evo_linear_mfma_nf_bf16)
extern "C" int evo_mlp_gate_mfma_nf_bf16(const void* x, const float* row_scale, const void* w12g, void* a_out, int64_t M, int64_t I, int64_t K,
                                         void* stream) {
    return gemmr_gate(x, row_scale, w12g, a_out, M, I, K, 0, stream);
}

int gemmr_gate(const void* x, const float* row_scale, const void* w12g, void* a_out, int64_t M, int64_t I, int64_t K, int64_t act, void* stream) {
    const int64_t N = 2 * I;
    if (act != 0 && act != 1) return -1;
    if (M <= 0 || I <= 0 || K <= 0 || N % GBN != 0 || K % GBK != 0 || K < 2 * GBK || N > 0x7fffffff / 2) return -1;
    if (M * K * 2 >= 0xffffffffll || N * K * 2 >= 0xffffffffll) return -1;
    GemmArgs a;
    a.x = (const unsigned char*)x; a.w = (const unsigned char*)w12g; a.bias = nullptr; a.res = nullptr; a.y = (uint16_t*)a_out;
    a.rs = row_scale;
    a.M = M; a.N = (int)N; a.K = (int)K;
    a.tiles_n = (int)(N / GBN);
    a.tiles_m = (int)((M + GBM - 1) / GBM);
    a.group_m = (a.tiles_n >= 32 ? 8 : 4);
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    if (tiles > 0x7fffffff) return -1;
    a.n_tiles = (int)tiles;
    static const int n_cu = [] {
        int dev = 0, n = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        n &= ~7;
        return n < 8 ? 8 : n;
    }();
    // Weights first in up to 16 rounds of tiles: 85.3 -> 81.8 us at 450 rows, 162.4 -> 157.5 at 900, 869 -> 865 at 7,208, 1,433 -> 1,421 at 11,877 (16 rounds of 22,016 columns, K = 4,096);
    // where the power limit has the clock it is level or behind (1,922 : 1,937 at 16,384, 7,547 : 7,568 at 65,536).
#define EVO_GATE(NF, ACT)                                                                                                                                    \
    do {                                                                                                                                                     \
        if (a.n_tiles <= 16 * n_cu) hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 1, false, NF, ACT, 8, true>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a); \
        else hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 1, false, NF, ACT, 8, false>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a); \
    } while (0)
    if (row_scale && act) EVO_GATE(2, 1);
    else if (row_scale) EVO_GATE(2, 0);
    else if (act) EVO_GATE(0, 1);
    else EVO_GATE(0, 0);
#undef EVO_GATE
    return evo_launch_status();
}

// z^T = (x [Mp, K] . w [N, K]^T + bias [N])^T, stored in blocks of 256 positions, zt [Mp / 256][N][256] (element (feature c, position p) at
// ((p / 256) * N + c) * 256 + p % 256): the Hyena projection with a CHANNEL-MAJOR result for csrc/hyena_ct.hip --
// [REF stripedhyena/model.py ParallelGatedConvBlock.forward: projections].  The persistent kernel is launched with its operands
// SWAPPED (its "X" = w: the rows of the result are output features; its "W" = x: the columns are tokens), so a lane's eight
// consecutive output columns are eight consecutive TOKENS of one feature and the epilogue stores whole 128-byte lines of z^T as it
// does for y; the bias is indexed by row (MODE 3).  Bit-identical to evo_linear_mfma_bf16's result, transposed (same k order of
// the same products, one rounding).  Mp % 256 == 0 (the caller pads: every row of x is computed), N % 256 == 0, K % 64 == 0, K >= 128.
extern "C" int evo_linear_t_mfma_bf16(const void* x, const void* w, const void* bias, void* zt, int64_t Mp, int64_t N, int64_t K,
                                      void* stream) {
    return evo_linear_t_mfma_nf_bf16(x, nullptr, w, bias, zt, Mp, N, K, Mp, Mp, 0, stream);
}

// ... with the block's pre-norm folded in: x = the residual stream [x_rows, K] in (batch row, token) order, w = W diag(g), row_scale
// [x_rows] = 1 / (rms + eps) per row; position p = b Tm + t of z^T (Mp = B Tm positions, Tm % 256 == 0) is row p + b row_skip of x -- the
// tail form of z^T (HipOps.zt_layout: Tm = T - row_skip), whose tail tokens the caller projects separately.  row_scale == NULL:
// the plain launch (x_rows = Tm = Mp, row_skip = 0).
extern "C" int evo_linear_t_mfma_nf_bf16(const void* x, const float* row_scale, const void* w, const void* bias, void* zt, int64_t Mp, int64_t N,
                                         int64_t K, int64_t x_rows, int64_t Tm, int64_t row_skip, void* stream) {
    if (row_scale) {
        if (Tm <= 0 || Tm % GBN != 0 || Mp % Tm != 0 || row_skip < 0 || row_skip > 0x7fff || x_rows < Mp + (Mp / Tm - 1) * row_skip
            || x_rows * K * 2 >= 0xffffffffll) return -1;
    } else if (x_rows != Mp || Tm != Mp || row_skip != 0) return -1;
    if (Mp <= 0 || N <= 0 || K <= 0 || Mp % GBN != 0 || N % GBM != 0 || K % GBK != 0 || K < 2 * GBK || Mp > 0x7fffffff / 2) return -1;
    if (Mp * K * 2 >= 0xffffffffll || N * K * 2 >= 0xffffffffll) return -1;
    GemmArgs a;
    a.x = (const unsigned char*)w; a.w = (const unsigned char*)x; a.bias = (const uint16_t*)bias; a.res = nullptr; a.y = (uint16_t*)zt;
    a.M = N; a.N = (int)Mp; a.K = (int)K;
    a.rs = row_scale; a.w_rows = x_rows; a.tm_tiles = (int)(Tm / GBN); a.row_skip = (int)row_skip;
    a.tiles_n = (int)(Mp / GBN);
    a.tiles_m = (int)(N / GBM);
    a.group_m = (a.tiles_m >= 32 ? 8 : 4);      // (column tiles per raster group: see tile_origin, MODE 3)
    const int64_t tiles = (int64_t)a.tiles_m * a.tiles_n;
    if (tiles > 0x7fffffff) return -1;
    a.n_tiles = (int)tiles;
    static const int n_cu = [] {
        int dev = 0, n = 256;
        if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev);
        n &= ~7;
        return n < 8 ? 8 : n;
    }();
    if (row_scale) {
        if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, false, 3, false, 2>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a);
        else hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 3, false, 2>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a);
        return evo_launch_status();
    }
    if (bias) hipLaunchKernelGGL((gemmr_bf16_kernel<true, false, 3>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a);
    else hipLaunchKernelGGL((gemmr_bf16_kernel<false, false, 3>), dim3((unsigned)n_cu), dim3(256), 0, (hipStream_t)stream, a);
    return evo_launch_status();
}
