// Internal header: the bf16-split GEMM kernels (gemm_split.hip) as the GEMM launcher sees them.
#pragma once

#include "gemm_device.h"

namespace mgc {

typedef void (*SplitKernel)(const GemmDev, const unsigned char *planes, long plane_bytes, int kblocks);

// Forms of A beside the AM_* ones of gemm_device.h: row-major but only 4-byte aligned (its row stride
// or K no multiple of four), and a convolution whose channel groups are a multiple of the 32-wide K
// stage, so that a stage reads one window tap.
enum { AM_LOOSE = 4, AM_TAP = 5 };
constexpr bool is_conv(int am) { return am == AM_CONV_VEC || am == AM_TAP; }

// The kernel for bm x bn tiles (128 x 128, 128 x 64, 32 x 64 or 32 x 32) of an A operand of form am
// (AM_VEC, AM_CONV_VEC, AM_CAT, AM_LOOSE or AM_TAP) and
// kchunk k per workgroup.
SplitKernel pick_split(int am, int bm, int bn, int kchunk);

// Tile and K split of a GEMM on the bf16-split kernels; bm 0: the fp32 kernels are faster.
struct SplitChoice {
    int bm, bn, split;
};

__global__ void split_planes_kernel(const float *b, long ldb, int N, int K, int kb, int nb, uint4_t *planes);

}  // namespace mgc
