// Internal header of the GEMM sources: operand forms, the kernel argument block and the device
// helpers the GEMM kernels share (operand loads, activations, the tile epilogue, LDS DMA).
#pragma once

#include "mgc_device.h"

namespace mgc {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));

// A operand forms: strided with unit column stride, NHWC image (implicit im2col), generic
// (register-staged), and a concatenation of a strided matrix (columns < k1) with an NHWC image
// read as a strided 1 x 1 convolution (columns >= k1).
enum { AM_VEC = 0, AM_CONV_VEC = 1, AM_GEN = 2, AM_CAT = 3 };

// 16 zero bytes: the load address of every out-of-range operand element.
static __device__ __attribute__((aligned(16))) float g_zero_page[4] = {0.0f, 0.0f, 0.0f, 0.0f};

// Loads through the global address space. Every operand lives in device memory; saying so
// keeps the compiler from falling back to flat loads, which share a wait counter with LDS.
typedef const __attribute__((address_space(1))) float gfloat;
typedef const __attribute__((address_space(1))) f4 gf4;
__device__ __forceinline__ float ldg(const float *ptr) { return *(gfloat *)ptr; }
__device__ __forceinline__ f4 ldg4(const float *ptr) { return *(gf4 *)ptr; }
enum { BD_NK_VEC = 0, BD_KN_VEC = 1, BD_GEN = 2 };

struct GemmDev {
    int M, N, K;
    mgc_hip_operand a, b;
    float *c;
    long ldc;
    float alpha, beta;
    const float *bias;
    int bias_mode;
    const float *res;
    long ldr;
    int act;
    float lo, hi;
    int batch_rank;
    int bdims[4];
    long a_bs[4], b_bs[4], c_bs[4], r_bs[4];
    int split;    // K splits (1 = none)
    int kchunk;   // K per split, a multiple of 32
    float *ws;    // split partials [split][M][N]
    int tiles_m, tiles_n;
    int vec_out;
    FastDiv div_ow, div_ohw, div_cg, div_kw;  // A as NHWC image: OW, OH * OW, cg, KW
    long a_bytes, b_bytes;  // bytes of A and B reachable from a.p / b.p (all batch elements)
    mgc_hip_operand a2;     // AM_CAT: the image whose 1 x 1 strided window gives columns >= k1
    int k1;
    long a2_bytes;
    int nbatch;   // batch elements
    int nfull = 0x7fffffff;  // gemm_dma_kernel: workgroups from this id on compute quarter tiles
};

__device__ __forceinline__ void batch_offsets(const GemmDev &p, int bz, long &ao, long &bo,
                                              long &co, long &ro) {
    ao = bo = co = ro = 0;
    int rem = bz;
#pragma unroll
    for (int d = 3; d >= 0; --d) {
        if (d < p.batch_rank) {
            int idx = rem % p.bdims[d];
            rem /= p.bdims[d];
            ao += idx * p.a_bs[d];
            bo += idx * p.b_bs[d];
            co += idx * p.c_bs[d];
            ro += idx * p.r_bs[d];
        }
    }
}

__device__ __forceinline__ f4 act4(f4 v, int act, float lo, float hi) {
    switch (act) {
    case MGC_ACT_RELU:
        v[0] = v[0] > 0.0f ? v[0] : 0.0f;
        v[1] = v[1] > 0.0f ? v[1] : 0.0f;
        v[2] = v[2] > 0.0f ? v[2] : 0.0f;
        v[3] = v[3] > 0.0f ? v[3] : 0.0f;
        return v;
    case MGC_ACT_CLIP:
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fminf(fmaxf(v[e], lo), hi);
        return v;
    case MGC_ACT_GELU:
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_erf_f(v[e]);
        return v;
    case MGC_ACT_GELU_TANH:
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_tanh_f(v[e]);
        return v;
    case MGC_ACT_TANH:
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tanh_f(v[e]);
        return v;
    case MGC_ACT_SIGMOID:
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = sigmoid_f(v[e]);
        return v;
    default: return v;
    }
}

// Epilogue shared by the GEMM kernels, pass 2: the BM x BN tile, staged in LDS at Cs with row
// pitch BN + 8 floats, leaves as 16-byte chunks with alpha, bias, residual and activation
// applied, or raw into the split-K workspace. Each thread owns one fixed 16-byte column chunk
// of the tile and the rows r0, r0 + RSTEP, ..., so the column bias is read once per thread.
// Every one of the 256 threads calls it (no barrier inside).
template <int BM, int BN>
__device__ __forceinline__ void gemm_lds_to_global(const GemmDev &p, const float *Cs, int m0, int n0, int ks,
                                                   long co, long ro) {
    constexpr int LDC = BN + 8;
    const f4 zero4 = {0.f, 0.f, 0.f, 0.f};
    const int tid = threadIdx.x;
    constexpr int C4 = BN / 4;
    static_assert(256 % C4 == 0, "column chunks must divide the workgroup");
    constexpr int RSTEP = 256 / C4;
    constexpr int ITERS = BM / RSTEP;
    constexpr int G = ITERS < 4 ? ITERS : 4;
    // Scalars read once: keeps the compiler from copying the argument block to scratch.
    const float alpha = p.alpha, beta = p.beta, lo = p.lo, hi = p.hi;
    const float *const bias = p.bias;
    const int act = p.act, M = p.M, N = p.N;
    const bool split_out = p.split > 1;
    float *const cbase = split_out ? p.ws + (long)ks * M * N : p.c + co;
    const long ldc = split_out ? (long)N : p.ldc;
    const float *const rbase = (!split_out && p.res) ? p.res + ro : nullptr;
    const bool vec = split_out ? (N % 4 == 0) : (p.vec_out != 0);
    const int cl = (tid % C4) * 4;
    const int col = n0 + cl;
    const int r0 = tid / C4;
    const bool col_ok = col < N;
    const int ncol = col_ok ? min(4, N - col) : 0;
    const bool full4 = vec && ncol == 4;
    const int bmode = split_out ? 0 : p.bias_mode;
    f4 cbias = zero4;
    if (bmode == 1 && col_ok) {
        if (full4) {
            cbias = ldg4(bias + col);
        } else {
            for (int e = 0; e < ncol; ++e) cbias[e] = ldg(bias + col + e);
        }
    }
    // pass 2: LDS tile -> epilogue -> memory, 16 bytes per access, G rows per step with their
    // residual chunks (and row biases) requested together.
    if (!col_ok) return;
    const bool pre_res = rbase != nullptr && full4;
#pragma unroll 1
    for (int g = 0; g < ITERS; g += G) {
        f4 rv[G];
        float rb[G];
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int row = m0 + r0 + RSTEP * (g + u);
            const bool ok = row < M;
            rv[u] = zero4;
            rb[u] = 0.0f;
            if (pre_res)
                rv[u] = ldg4(ok ? rbase + (long)row * p.ldr + col
                                                         : g_zero_page);
            if (bmode == 2) rb[u] = ldg(ok ? bias + row : g_zero_page);
        }
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int rl = r0 + RSTEP * (g + u);
            const int row = m0 + rl;
            if (row >= M) break;
            f4 v = *reinterpret_cast<const f4 *>(&Cs[rl * LDC + cl]);
            float *dst = cbase + (long)row * ldc + col;
            if (!split_out) {
                v = v * alpha + cbias;
                if (bmode == 2) v += rb[u];
                if (pre_res) {
                    v += beta * rv[u];
                } else if (rbase) {
                    const float *src = rbase + (long)row * p.ldr + col;
                    for (int e = 0; e < ncol; ++e) v[e] += beta * ldg(src + e);
                }
                v = act4(v, act, lo, hi);
            }
            if (full4) {
                *reinterpret_cast<f4 *>(dst) = v;
            } else {
                for (int e = 0; e < ncol; ++e) dst[e] = v[e];
            }
        }
    }
}


// The whole epilogue: pass 1 moves the accumulators to LDS (smem, at least BM * (BN + 8)
// floats, free when this is called), then gemm_lds_to_global.
template <int BM, int BN, int WGM, int RM, int RN>
__device__ __forceinline__ void gemm_store_tile(const GemmDev &p, float *smem,
                                                     const floatx16 (&acc)[RM][RN], int m0, int n0,
                                                     int ks, long co, long ro) {
    constexpr int WGN = 4 / WGM;
    constexpr int WM = BM / WGM;
    constexpr int WN = BN / WGN;
    constexpr int LDC = BN + 8;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm = wave / WGN, wn = wave - (wave / WGN) * WGN;
    const int li = lane & 31;
    const int lh = lane >> 5;
    // pass 1: registers -> LDS tile. Block (i, j) register r holds tile row
    // 8 * (r / 4) + 4 * lh + r % 4 and column li of that 32x32 block.
    float *const Cs = smem;
#pragma unroll
    for (int i = 0; i < RM; ++i)
#pragma unroll
        for (int j = 0; j < RN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                Cs[(wm * WM + i * 32 + (r >> 2) * 8 + lh * 4 + (r & 3)) * LDC + wn * WN + j * 32 +
                   li] = acc[i][j][r];
    __syncthreads();
    gemm_lds_to_global<BM, BN>(p, Cs, m0, n0, ks, co, ro);
}

// s_waitcnt with only the vector-memory counter constrained (expcnt and lgkmcnt at maximum).
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x70 | 0xF00);
}

// Workgroup barrier for the LDS ring: waits for this wave's own LDS accesses only. The
// __syncthreads() fence would also wait for every outstanding global load, including the
// DMA loads of later pipeline stages, and drain the ring at every step.
__device__ __forceinline__ void barrier_lds() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

typedef __attribute__((address_space(3))) void lds_void;

// 16 bytes at byte offset voff of a buffer resource straight into LDS (lane l of the wave
// writes lds_base + 16 * l); offsets at or past the resource's size read as zeros.
__device__ __forceinline__ void dma16_buf(__amdgpu_buffer_rsrc_t r, unsigned voff, float *lds_base) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_void *)lds_base, 16, (int)voff, 0, 0, 0);
}

}  // namespace mgc
