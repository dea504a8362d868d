// The persistent dense-layer kernel on tiles of 224 x 256 (gemm_kernel.h; gemm_tile.hip chooses).
#include "gemm_kernel.h"

int gemmr_rows224(const GemmArgs& args, int mode, int act, hipStream_t st) {
    GemmArgs a = args;
    a.tiles_m = (int)((a.M + 223) / 224);
    a.tiles_n = a.N / GBN;
    a.n_tiles = a.tiles_m * a.tiles_n;
    a.group_m = mode == 3 ? gemmr_group(a.tiles_n, a.tiles_m) : gemmr_group(a.tiles_m, a.tiles_n);
    return gemmr_launch<7>(a, mode, act, st);
}
