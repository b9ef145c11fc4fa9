// Internal header: the bf16-split GEMM kernels (gemm_split.hip) as the GEMM launcher sees them.
#pragma once

#include "gemm_device.h"

namespace mgc {

typedef void (*SplitKernel)(const GemmDev, const unsigned char *planes, long plane_bytes, int kblocks);

// The kernel for 128 x bn tiles (bn 128 or 64) of an A operand of form am (AM_VEC, AM_CONV_VEC
// or AM_CAT).
SplitKernel pick_split(int am, int bn);

// Tile and K split of a GEMM on the bf16-split kernels; bm 0: the fp32 kernels are faster.
struct SplitChoice {
    int bm, bn, split;
};

__global__ void split_planes_kernel(const float *b, long ldb, int N, int K, int kb, int nb, uint4_t *planes);
__global__ void tiny_columns_kernel(const float *b, long ldb, int N, int K, unsigned char *flags, int nflags);

}  // namespace mgc
