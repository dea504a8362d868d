// Arguments of the dense-layer kernels (gemm.hip, gemm_tile.hip).
#pragma once
#include "common.h"

struct GemmArgs {
    const unsigned char* x; const unsigned char* w; const uint16_t* bias; const uint16_t* res; uint16_t* y;
    int64_t M; int N; int K;
    int tiles_n; int n_tiles; int tiles_m; int group_m;
    // RMSNorm folded into the dense layers around it
    const float* rs = nullptr;               // SCALE: 1 / (rms + eps) per token row, applied to the accumulators in the epilogue
    float* ss = nullptr;                     // STATS: partial sums of squares of the stored rows, [N / 128 strips][ss_ld] fp32
    int64_t ss_ld = 0;
    int act_cols = 0;                        // ACT, mode 0: columns [0, act_cols) of the result go through the activation (a multiple of 256)
    int turn = 0;                            // gemm_tile.hip: 1: tiles of neighbouring weight rows start one k-step apart
    int64_t w_rows = 0;                      // MODE 3 + SCALE: rows of the token matrix (the kernel's "W" operand): B T; gemm_tile.hip, MODE 1: N where W is [W1; W2] as it is
    int tm_tiles = 0, row_skip = 0;          // MODE 3 + SCALE: a batch row = tm_tiles column tiles of 256; its tokens start row_skip rows further per batch row
};
