// fp32 GEMM and implicit-GEMM convolution on the bf16 matrix cores, with 24-bit operands.
//
// gfx950 multiplies fp32 at 157 TFLOP/s (v_mfma_f32_32x32x2_f32) and bf16 at 2.5 PFLOP/s. An fp32
// number is the exact sum of three bf16 numbers, x = h + m + l (each the round-to-nearest bf16 of
// what the ones before leave: 8 + 8 + 8 significant bits), so
//   a b = ah bh + (ah bm + am bh) + (ah bl + am bm + al bh) + O(2^-25 |a b|)
// is six bf16 products, summed in fp32 by v_mfma_f32_32x32x16_bf16: 6 x 32 cycles for 16 k of a
// 32 x 32 block against 8 x 64 cycles in fp32, a ceiling of 416 TFLOP/s. The dropped products
// (am bl, al bm, al bl) are below the rounding of one fp32 product. The leading products and the
// five corrections have an accumulator each, so the corrections are not rounded at the size of
// the whole sum, and the leading sum is rounded once per 16 k instead of once per product:
// against 64 bits a 768-long dot product of normal numbers is 1.5e-7 off (fp32 MFMA: 4.8e-7), a
// 4608-long one 4.3e-7 (1.2e-6).
//
// bf16 has fp32's exponents, so the low parts of a number below 2^-110 would end under bf16's smallest
// subnormal (2^-133). Both operands are therefore split 2^16 times their size, which puts the last
// bit of every fp32 number, subnormals too, at 2^-133 or above (the MFMA keeps bf16 and fp32 subnormals),
// and the sums are multiplied by 2^-32. That is one multiplication per element of A (marking rows and columns of
// small numbers instead cost an instruction per two elements, and a small number beside normal ones
// escaped it): with the recomputation below, ResNet-50 b32 2212 -> 2169 us, the BERT feed-forward b16
// 137.9 -> 135.9, the vocabulary projection, whose MFMAs wait for the split of A, 446 -> 451.
//
// Sums that are not finite (an infinite or NaN operand, operands of 2^112 or sums of 2^96 on, which the
// scaled split overflows to infinities and NaN) are recomputed in fp32 from the operands: a wave that
// holds one runs its part of the tile again on the fp32 MFMA (sums_fp32). An all-NaN 2048 x 768 x 3072
// product takes 205 us, a finite one 83; recomputing each sum in a serial loop took 11500.
#include "gemm_split.h"

namespace mgc {

typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

// Two floats rounded to nearest bf16, packed (v_cvt_pk_bf16_f32).
__device__ __forceinline__ unsigned pack_bf16(float x, float y) {
    const f2 v = {x, y};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf2));
}

// Two floats as three packed bf16 pairs whose exact sums are 2^16 times the floats.
__device__ __forceinline__ void split3(float x, float y, unsigned &h, unsigned &m, unsigned &l) {
    x *= 0x1p16f;
    y *= 0x1p16f;
    h = pack_bf16(x, y);
    x -= __uint_as_float(h << 16);
    y -= __uint_as_float(h & 0xffff0000u);
    m = pack_bf16(x, y);
    x -= __uint_as_float(m << 16);
    y -= __uint_as_float(m & 0xffff0000u);
    l = pack_bf16(x, y);
}

// 16 bytes at byte offset voff of a buffer resource; zeros at or past its end.
__device__ __forceinline__ f4 buf_load4(__amdgpu_buffer_rsrc_t r, unsigned voff) {
    return __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, 0, 0));
}

// Workgroup barrier of a stage: this wave's loads but the last N have landed, its LDS reads too.
// One statement, so that no load moves across the wait that counts it.
template <int N>
__device__ __forceinline__ void barrier_stage() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Split the constant right-hand side b ([N][K] with row stride ldb) into planes. One thread per
// 8 consecutive k of one column (16 bytes of each plane); padding is written as zeros.
__global__ void __launch_bounds__(256) split_planes_kernel(const float *b, long ldb, int N, int K, int kb, int nb,
                                                           uint4_t *planes) {
    const long total = (long)nb * kb * 64;
    for (long t = blockIdx.x * 256L + threadIdx.x; t < total; t += gridDim.x * 256L) {
        const int lane = (int)(t & 63);
        const long block = t >> 6;  // (column block, 16-k block)
        const int n = (int)(block / kb) * 32 + (lane & 31);
        const int k = (int)(block % kb) * 16 + (lane >> 5) * 8;
        uint4_t h, m, l;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float x = n < N && k + 2 * e < K ? b[n * ldb + k + 2 * e] : 0.0f;
            const float y = n < N && k + 2 * e + 1 < K ? b[n * ldb + k + 2 * e + 1] : 0.0f;
            unsigned u, v, w;
            split3(x, y, u, v, w);
            h[e] = u;
            m[e] = v;
            l[e] = w;
        }
        uint4_t *const dst = planes + block * 192 + lane;
        dst[0] = h;
        dst[64] = m;
        dst[128] = l;
    }
}

// One lane's row of A: 8 consecutive k at a time through a buffer resource, masked elements zero.
template <int AMODE>
struct SplitRow {
    static constexpr unsigned OOB = 0x80000000u;  // past every resource's end (extents are < 2^31 bytes)
    unsigned aoff = OOB, aoff2 = OOB;  // byte offset of the row (convolutions: of its window's origin; AM_CAT: in a2)
    int aih = -0x40000000, aiw = -0x40000000;  // fails the window bounds test

    __device__ __forceinline__ SplitRow(const GemmDev &p, int m) {
        if (m >= p.M) return;
        if (AMODE == AM_CAT) {
            const int n = fdiv(m, p.div_ohw), rr = m - n * p.a2.OH * p.a2.OW;
            const int oh = fdiv(rr, p.div_ow), ow = rr - oh * p.a2.OW;
            aoff2 = (unsigned)(((n * p.a2.H + oh * p.a2.SH) * p.a2.W + ow * p.a2.SW) * p.a2.C) * 4u;
        }
        if (is_conv(AMODE)) {
            const int n = fdiv(m, p.div_ohw), rr = m - n * p.a.OH * p.a.OW;
            const int oh = fdiv(rr, p.div_ow), ow = rr - oh * p.a.OW;
            aih = oh * p.a.SH - p.a.PT;
            aiw = ow * p.a.SW - p.a.PL;
            aoff = (unsigned)(((n * p.a.H + aih) * p.a.W + aiw) * p.a.C) * 4u;
        } else {
            aoff = (unsigned)m * (unsigned)p.a.rs * 4u;
        }
    }

    // Four k of a row that is only 4-byte aligned: the load stays inside the row (the last four
    // elements where k is nearer its end) and the elements are moved into place.
    __device__ __forceinline__ f4 load_loose(__amdgpu_buffer_rsrc_t r, int k, int kend) const {
        const int at = min(k, kend - 4), s = k - at;
        const f4 v = buf_load4(r, s < 4 ? aoff + (unsigned)at * 4u : OOB);
        const f4 t = {s & 1 ? v[1] : v[0], s & 1 ? v[2] : v[1], s & 1 ? v[3] : v[2], s & 1 ? 0.0f : v[3]};
        return f4{s & 2 ? t[2] : t[0], s & 2 ? t[3] : t[1], s & 2 ? 0.0f : t[2], s & 2 ? 0.0f : t[3]};
    }

    // x, y: elements k .. k + 3 and k + 4 .. k + 7 (k a multiple of 8) of a stage that starts at `stage`.
    __device__ __forceinline__ void load(const GemmDev &p, int stage, int k, int kend, f4 &x, f4 &y) const {
        const bool k0 = k < kend, k1 = k + 4 < kend;
        if constexpr (AMODE == AM_CAT) {
            // k1 is a multiple of the 32-wide stage, so a whole stage reads one source
            const bool second = stage >= p.k1;
            const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(
                (void *)(second ? p.a2.p : p.a.p), (short)0, (int)(second ? p.a2_bytes : p.a_bytes), 0x00020000);
            const unsigned o = second ? aoff2 + (unsigned)(k - p.k1) * 4u : aoff + (unsigned)k * 4u;
            x = buf_load4(r, k0 ? o : OOB);
            y = buf_load4(r, k1 ? o + 16u : OOB);
        } else {
            const __amdgpu_buffer_rsrc_t r =
                __builtin_amdgcn_make_buffer_rsrc((void *)p.a.p, (short)0, (int)p.a_bytes, 0x00020000);
            if constexpr (AMODE == AM_VEC) {
                const unsigned o = aoff + (unsigned)k * 4u;
                x = buf_load4(r, k0 ? o : OOB);
                y = buf_load4(r, k1 ? o + 16u : OOB);
            } else if constexpr (AMODE == AM_LOOSE) {
                x = load_loose(r, k, kend);
                y = load_loose(r, k + 4, kend);
            } else if constexpr (AMODE == AM_TAP) {
                // The stage's 32 k share a tap: its coordinates are scalar arithmetic, once a stage
                // (211 vector instructions in two stages of 128 columns instead of 286, 24 of them
                // multiplies at a quarter of the rate). ResNet-50 b32 2254 -> 2226 us.
                const int t = fdiv(stage, p.div_cg), kh = fdiv(t, p.div_kw);
                const int dh = kh * p.a.DH, dw = (t - kh * p.a.KW) * p.a.DW;
                const bool ok =
                    (stage < kend) & ((unsigned)(aih + dh) < (unsigned)p.a.H) & ((unsigned)(aiw + dw) < (unsigned)p.a.W);
                const int tap = (dh * p.a.W + dw) * p.a.C + (stage - t * p.a.cg);
                const unsigned o = ok ? aoff + (unsigned)(tap + (k - stage)) * 4u : OOB;
                x = buf_load4(r, o);
                y = buf_load4(r, o + 16u);
            } else {  // cg % 8 == 0: the 8 k share a tap
                const int t = fdiv(k, p.div_cg), kh = fdiv(t, p.div_kw);
                const int dh = kh * p.a.DH, dw = (t - kh * p.a.KW) * p.a.DW;
                const bool ok = k0 && (unsigned)(aih + dh) < (unsigned)p.a.H && (unsigned)(aiw + dw) < (unsigned)p.a.W;
                const unsigned o = ok ? aoff + (unsigned)((dh * p.a.W + dw) * p.a.C + (k - t * p.a.cg)) * 4u : OOB;
                x = buf_load4(r, o);
                y = buf_load4(r, o + 16u);
            }
        }
    }
};

// Eight consecutive k of a row as the three MFMA operands.
__device__ __forceinline__ void split_row(const f4 &x, const f4 &y, bf8 (&a)[3]) {
    uint4_t h, m, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const f4 &v = e < 2 ? x : y;
        unsigned u0, u1, u2;
        split3(v[2 * (e & 1)], v[2 * (e & 1) + 1], u0, u1, u2);
        h[e] = u0;
        m[e] = u1;
        l[e] = u2;
    }
    a[0] = __builtin_bit_cast(bf8, h);
    a[1] = __builtin_bit_cast(bf8, m);
    a[2] = __builtin_bit_cast(bf8, l);
}

// A wave's 32 rows x 32 RN columns (arow, from n0) in fp32, over the 32-wide K stages k0, k0 + step, ...
// straight from the operands. Each half wave's eight k of a 16-k step meet the other half's in eight
// v_mfma_f32_32x32x2_f32.
template <int RN, int AMODE>
__device__ __forceinline__ void sums_fp32(const GemmDev &p, const SplitRow<AMODE> &arow, int n0, int k0, int step,
                                          int kend, floatx16 (&sum)[RN]) {
    const int lane = threadIdx.x & 63, li = lane & 31, lh = lane >> 5;
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[j][r] = 0.0f;
#pragma unroll 1
    for (int stage = k0; stage < kend; stage += step) {
#pragma unroll 1
        for (int k = stage + 8 * lh; k < stage + 32; k += 16) {
            f4 a[2], b[RN][2];
            arow.load(p, stage, k, kend, a[0], a[1]);
#pragma unroll
            for (int j = 0; j < RN; ++j) {
                const int col = n0 + 32 * j + li;
                const float *const src = p.b.p + (long)col * p.b.cs + k;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if constexpr (AMODE == AM_LOOSE) {
#pragma unroll
                        for (int e = 4 * h; e < 4 * h + 4; ++e)
                            b[j][h][e & 3] = ldg(col < p.N && k + e < kend ? src + e : g_zero_page);
                    } else {  // K and the rows' addresses are multiples of four
                        b[j][h] = ldg4(col < p.N && k + 4 * h < kend ? src + 4 * h : g_zero_page);
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int j = 0; j < RN; ++j)
                    sum[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e >> 2][e & 3], b[j][e >> 2][e & 3], sum[j], 0, 0, 0);
        }
    }
}

// The wave's sums from its two accumulators, those that are not finite in fp32 (cor is scratch).
template <int RN, int AMODE>
__device__ __forceinline__ void finish_sums(const GemmDev &p, const SplitRow<AMODE> &arow, int n0, int k0, int step,
                                            int kend, floatx16 (&acc)[RN], floatx16 (&cor)[RN]) {
    float z = 0.0f;  // NaN if a sum is not finite
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            acc[j][r] = (acc[j][r] + cor[j][r]) * 0x1p-32f;
            z = fmaf(acc[j][r], 0.0f, z);
        }
    if (!__any(z != z)) return;
    sums_fp32<RN, AMODE>(p, arow, n0, k0, step, kend, cor);
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = fabsf(acc[j][r]) < __builtin_huge_valf() ? acc[j][r] : cor[j][r];
}

// A workgroup of WAVES waves owns a tile of 32 WAVES rows x 32 RN columns; each wave owns 32 rows and
// all the columns. K advances 32 per stage (two MFMA depths of 16).
//
//  * A: a lane's MFMA operand is 8 consecutive k of one row, so the wave loads its own rows' fp32
//    straight into registers two stages ahead (two 16-byte loads per 16 k through a buffer
//    resource; masked elements read as zero) and splits them there: each element is split once
//    per column tile, and A never goes through LDS.
//  * B: planes split once when the weights are laid out, in fragment order (for a block of 32
//    columns and 16 k the three planes' 64 lanes x 16 bytes), so a stage is copied to LDS by
//    linear 1 KB DMA instructions and read back as linear 16-byte fragments without bank
//    conflicts. A ring of R stages, one barrier per stage, loads two stages ahead.
//
// A wave's 32 x 128 part has 2 x 64 accumulator registers, which two waves per SIMD (two
// workgroups per CU) allow.
template <int RN, int WAVES, int R, int AMODE, bool ORDERED = false>
__global__ void __launch_bounds__(64 * WAVES, RN >= 4 ? 2 : 3)
    gemm_split_kernel(const GemmDev p, const unsigned char *planes, long plane_bytes, int kblocks) {
    constexpr int BK = 32;
    constexpr int BM = 32 * WAVES, BN = 32 * RN;
    constexpr int SLOT = RN * 6 * 1024;             // bytes of one stage of B
    constexpr int DMA = RN * 6 / WAVES;             // 1 KB copies per wave and stage
    static_assert(WAVES == 4 && RN * 6 % WAVES == 0, "the epilogue's workgroup; copies divide among the waves");
    constexpr int EPI = BM * (BN + 8) * 4;
    __shared__ __attribute__((aligned(16))) unsigned char smem[R * SLOT > EPI ? R * SLOT : EPI];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

    // XCD-aware tile order, N fastest (as the fp32 kernels)
    const int nb = gridDim.x;
    const int full = nb & ~7;
    int lin = blockIdx.x;
    if (lin < full) {
        const int per = full >> 3;
        lin = (lin & 7) * per + (lin >> 3);
    }
    const int tm = lin / p.tiles_n;
    const int tn = lin - tm * p.tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    const int ks = blockIdx.z;
    const int kbeg = ks * p.kchunk;
    const int kend = min(p.K, kbeg + p.kchunk);
    const int nk = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
    constexpr unsigned OOB = SplitRow<AMODE>::OOB;

    const int li = lane & 31;
    const int lh = lane >> 5;
    const SplitRow<AMODE> arow(p, m0 + 32 * wave + li);
    f4 va[2][4];    // [set][16-k block, half of the lane's 8 k]
    int ka = kbeg;  // the stage the next A loads fetch
    auto load_a = [&](f4 (&v)[4]) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) arow.load(p, ka, ka + 16 * s + 8 * lh, kend, v[2 * s], v[2 * s + 1]);
        ka += BK;
    };

    // ---- B: 1 KB copy c of a stage is plane c % 3 of 16-k block c / 3 % 2 of column block c / 6 ----
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void *)planes, (short)0, (int)plane_bytes, 0x00020000);
    const unsigned nb_bytes = (unsigned)kblocks * 3072u;
    static_assert(6 % DMA == 0, "a wave's copies lie in one column block");
    const int block = n0 / 32 + wave * DMA / 6;
    // column blocks past N lie past the resource's end, whatever stage is added
    unsigned boff = block * 32 < p.N
                        ? (unsigned)block * nb_bytes + (unsigned)(kbeg >> 4) * 3072u +
                              (unsigned)(wave * DMA % 6) * 1024u + (unsigned)lane * 16u
                        : OOB;
    auto copy_b = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < DMA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_void *)(smem + slot * SLOT + (wave * DMA + i) * 1024), 16,
                                                     (int)boff, i * 1024, 0, 0);
        boff += 6144u;
    };

    floatx16 acc[RN], cor[RN];
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = cor[j][r] = 0.0f;

    constexpr int G = 2;           // column blocks at a time: independent chains, few registers
    constexpr int P = RN / G * 6;  // MFMA pairs of a 16-k step
    static_assert(RN % G == 0, "whole groups of column blocks");
    bf8 b[G][3];
    auto read_b = [&](int q, const unsigned char *bs) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < G; ++j) b[j][q] = *reinterpret_cast<const bf8 *>(bs + j * 6144 + q * 1024 + lane * 16);
    };
    // Stage kt: its copies and A loads have landed once at most the next stage's are outstanding
    // (R = 3), and every wave has read the slot that the new copies overwrite. Loads past the
    // end are masked, so the loop needs no tests.
    //
    // ORDERED (a row-major A): the order inside a stage is written out (sched_barrier). A group's B
    // planes are read as the group before is done with its own, and the next step's A is split and
    // the A of two stages on requested a quarter at a time between MFMA pairs. Left to the compiler,
    // the split and the fragment waits stood in front of each step's MFMAs (1024 x 768 x 50257 476 -> 448 us,
    // BERT feed-forward b16 146 -> 139 us). The other forms of A need more address arithmetic between the loads, which
    // the compiler places better (in this order: bottleneck b32 227 -> 236 us, 1003 x 515 x 1021 36 ->
    // 43 us).
    int slot = 0;
    uint4_t a0[3], a1[3];
    auto stage = [&](f4 (&v)[4], f4 (&w)[4]) __attribute__((always_inline)) {
        constexpr int QA[6] = {0, 2, 1, 1, 0, 0}, QB[6] = {0, 0, 0, 1, 1, 2};
        barrier_stage<(R - 2) * (DMA + 4)>();
        const unsigned char *const bs = smem + slot * SLOT;
        if constexpr (ORDERED) {
#pragma unroll
            for (int q = 0; q < 3; ++q) read_b(q, bs);
            copy_b(slot == 0 ? R - 1 : slot - 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 2 * P; ++t) {
                const int s = t / P, q = t % P, i = t % 6, j0 = q / 6 * G;
                const bf8 a = __builtin_bit_cast(bf8, s ? a1[QA[i]] : a0[QA[i]]);
#pragma unroll
                for (int j = 0; j < G; ++j) {
                    floatx16 &c = i == 0 ? acc[j0 + j] : cor[j0 + j];
                    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[j][QB[i]], c, 0, 0, 0);
                }
                // planes 0, 1 and 2 of the next group after this group's last use of them
                if ((i == 2 || i >= 4) && t + 6 - i < 2 * P) {
                    const int n = t + 6 - i;
                    read_b(i == 2 ? 0 : i - 3, bs + n / P * 3072 + n % P / 6 * G * 6144);
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (q == (e * P + 2) / 4) {
                        const f4 &x = s ? w[e >> 1] : v[2 + (e >> 1)];
                        unsigned h, m, l;
                        split3(x[2 * (e & 1)], x[2 * (e & 1) + 1], h, m, l);
                        uint4_t(&next)[3] = s ? a0 : a1;
                        next[0][e] = h;
                        next[1][e] = m;
                        next[2][e] = l;
                    }
                // v's first half was split in the stage before, its second half in this one's first step
                if (t == P / 2) arow.load(p, ka, ka + 8 * lh, kend, v[0], v[1]);
                if (t == P + P / 3) arow.load(p, ka, ka + 16 + 8 * lh, kend, v[2], v[3]);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            copy_b(slot == 0 ? R - 1 : slot - 1);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                uint4_t(&a)[3] = s ? a1 : a0;
                uint4_t(&next)[3] = s ? a0 : a1;
                bf8 split[3];
                split_row(s ? w[0] : v[2], s ? w[1] : v[3], split);
#pragma unroll
                for (int q = 0; q < 3; ++q) next[q] = __builtin_bit_cast(uint4_t, split[q]);
#pragma unroll
                for (int j0 = 0; j0 < RN; j0 += G) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) read_b(q, bs + s * 3072 + j0 * 6144);
#pragma unroll
                    for (int i = 0; i < 6; ++i)
#pragma unroll
                        for (int j = 0; j < G; ++j) {
                            floatx16 &c = i == 0 ? acc[j0 + j] : cor[j0 + j];
                            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf8, a[QA[i]]), b[j][QB[i]], c, 0, 0, 0);
                        }
                }
                if (s == 0) {
#pragma unroll
                    for (int h = 0; h < 2; ++h) arow.load(p, ka, ka + 16 * h + 8 * lh, kend, v[2 * h], v[2 * h + 1]);
                }
            }
        }
        ka += BK;
        slot = slot == R - 1 ? 0 : slot + 1;
    };

    static_assert(R == 3, "the waits above count for a ring of three");
    copy_b(0);
    load_a(va[0]);
    asm volatile("" ::: "memory");  // the stages' loads stay in order: the waits count them
    copy_b(1);
    load_a(va[1]);
    asm volatile("" ::: "memory");
    {
        bf8 first[3];
        split_row(va[0][0], va[0][1], first);
#pragma unroll
        for (int q = 0; q < 3; ++q) a0[q] = __builtin_bit_cast(uint4_t, first[q]);
    }
    for (int kt = nk >> 1; kt > 0; --kt) {
        stage(va[0], va[1]);
        stage(va[1], va[0]);
    }
    if (nk & 1) stage(va[0], va[1]);
    wait_vmcnt<0>();  // masked copies past the end may still be writing the ring
    __syncthreads();
    finish_sums<RN, AMODE>(p, arow, n0, kbeg, BK, kend, acc, cor);

    float *const Cs = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            Cs[(32 * wave + (r >> 2) * 8 + lh * 4 + (r & 3)) * (BN + 8) + j * 32 + li] = acc[j][r];
    __syncthreads();
    gemm_lds_to_global<BM, BN>(p, Cs, m0, n0, ks, 0, 0);
}

// The same products for GEMMs whose 128-row tiles are too few for the CUs: a tile of 32 rows x 32 RN
// columns per workgroup, whose K stages are dealt to its WAVES waves (wave w takes stages w,
// w + WAVES, ...). Every wave loads its own A rows and B planes straight into registers, two stages
// ahead, so the main loop has neither LDS nor barriers; a stage's B planes are linear 1 KB loads.
// The partial tiles are summed through LDS in wave order, each thread finishing the 16-byte chunks
// whose bias and residual it requested at the start.
template <int RN, int WAVES, int AMODE>
__global__ void __launch_bounds__(64 * WAVES)
    gemm_split_small_kernel(const GemmDev p, const unsigned char *planes, long plane_bytes, int kblocks) {
    constexpr int BK = 32, T = 32;
    constexpr int BN = 32 * RN;
    constexpr int LDC = BN + 8;
    constexpr int CHUNKS = T * BN / 4;                      // 16-byte chunks of the tile
    constexpr int PER = (CHUNKS + 64 * WAVES - 1) / (64 * WAVES);  // per thread
    __shared__ __attribute__((aligned(16))) float slots[WAVES * T * LDC];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nb = gridDim.x;
    const int full = nb & ~7;
    int lin = blockIdx.x;
    if (lin < full) {
        const int per = full >> 3;
        lin = (lin & 7) * per + (lin >> 3);
    }
    // rows fastest: the workgroups that share B planes (the larger operand here) are neighbours
    const int tn = lin / p.tiles_m;
    const int tm = lin - tn * p.tiles_m;
    const int m0 = tm * T, n0 = tn * BN;
    const int ks = blockIdx.z;
    const int kbeg = ks * p.kchunk;
    const int kend = min(p.K, kbeg + p.kchunk);
    const int nk = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
    const int nkw = nk > wave ? (nk - 1 - wave) / WAVES + 1 : 0;  // this wave's stages

    const int li = lane & 31;
    const int lh = lane >> 5;
    const SplitRow<AMODE> arow(p, m0 + li);
    const __amdgpu_buffer_rsrc_t rb =
        __builtin_amdgcn_make_buffer_rsrc((void *)planes, (short)0, (int)plane_bytes, 0x00020000);
    unsigned boff[RN];  // column blocks past N lie past the resource's end, whatever stage is added
#pragma unroll
    for (int j = 0; j < RN; ++j) {
        const int block = n0 / 32 + j;
        boff[j] = block * 32 < p.N ? ((unsigned)block * (unsigned)kblocks + (unsigned)((kbeg >> 4) + 2 * wave)) * 3072u +
                                         (unsigned)lane * 16u
                                   : SplitRow<AMODE>::OOB;
    }
    int ka = kbeg + wave * BK;
    f4 va[2][4], vb[2][RN][6];
    auto load = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
            arow.load(p, ka, ka + 16 * s + 8 * lh, kend, va[set][2 * s], va[set][2 * s + 1]);
        const bool live = ka < kend;  // stages past the end read nothing
#pragma unroll
        for (int j = 0; j < RN; ++j) {
            const unsigned o = live ? boff[j] : SplitRow<AMODE>::OOB;
#pragma unroll
            for (int q = 0; q < 6; ++q)
                vb[set][j][q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)o, q * 1024, 0));
            boff[j] += (unsigned)WAVES * 6144u;
        }
        ka += WAVES * BK;
    };
    load(0);
    load(1);

    // epilogue operands: thread t owns chunks t, t + 64 WAVES, ...
    const bool split_out = p.split > 1;
    const bool vec = split_out ? p.N % 4 == 0 : p.vec_out != 0;
    const f4 zero4 = {0.f, 0.f, 0.f, 0.f};
    f4 ebias[PER], eres[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int c = tid + u * 64 * WAVES;
        const int row = m0 + c / (BN / 4), col = n0 + c % (BN / 4) * 4;
        ebias[u] = eres[u] = zero4;
        if (c < CHUNKS && row < p.M && col + 4 <= p.N && vec && !split_out) {
            if (p.bias && p.bias_mode == 1) ebias[u] = ldg4(p.bias + col);
            if (p.res) eres[u] = ldg4(p.res + (long)row * p.ldr + col);
        }
    }

    floatx16 acc[RN], cor[RN];
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = cor[j][r] = 0.0f;
    auto stage = [&](int set) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            bf8 a[3];
            split_row(va[set][2 * s], va[set][2 * s + 1], a);
#define MGC_MFMA(C, QA, QB)                                                                                        \
    _Pragma("unroll") for (int j = 0; j < RN; ++j) C[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(                 \
        a[QA], __builtin_bit_cast(bf8, vb[set][j][3 * s + QB]), C[j], 0, 0, 0);
            MGC_MFMA(acc, 0, 0)
            MGC_MFMA(cor, 2, 0)
            MGC_MFMA(cor, 1, 0)
            MGC_MFMA(cor, 1, 1)
            MGC_MFMA(cor, 0, 1)
            MGC_MFMA(cor, 0, 2)
#undef MGC_MFMA
        }
        load(set);
    };
    for (int kt = nkw >> 1; kt > 0; --kt) {
        stage(0);
        stage(1);
    }
    if (nkw & 1) stage(0);

    finish_sums<RN, AMODE>(p, arow, n0, kbeg + wave * BK, WAVES * BK, kend, acc, cor);
#pragma unroll
    for (int j = 0; j < RN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
            slots[wave * (T * LDC) + ((r >> 2) * 8 + lh * 4 + (r & 3)) * LDC + j * 32 + li] = acc[j][r];
    __syncthreads();
    const int M = p.M, N = p.N, act = p.act, bias_mode = p.bias ? p.bias_mode : 0;
    const float alpha = p.alpha, beta = p.beta, lo = p.lo, hi = p.hi;
    const float *const bias = p.bias, *const res = p.res;
    const long ldr = p.ldr;
    float *const cbase = split_out ? p.ws + (long)ks * M * N : p.c;
    const long ldc = split_out ? (long)N : p.ldc;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int c = tid + u * 64 * WAVES;
        const int rl = c / (BN / 4), cl = c % (BN / 4) * 4;
        const int row = m0 + rl, col = n0 + cl;
        if (c >= CHUNKS || row >= M || col >= N) continue;
        const int ncol = min(4, N - col);
        const bool full4 = vec && ncol == 4;
        const int o = rl * LDC + cl;
        f4 v = *reinterpret_cast<const f4 *>(&slots[o]);
#pragma unroll
        for (int w = 1; w < WAVES; ++w) v += *reinterpret_cast<const f4 *>(&slots[w * (T * LDC) + o]);
        float *const dst = cbase + (long)row * ldc + col;
        if (!split_out) {
            f4 b = ebias[u], r = eres[u];
            if (!full4) {  // scalar bias and residual reads
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (e < ncol && bias_mode == 1) b[e] = ldg(bias + col + e);
                    if (e < ncol && res) r[e] = ldg(res + (long)row * ldr + col + e);
                }
            }
            v = v * alpha + b;
            if (bias_mode == 2) v += ldg(bias + row);
            if (res) v += beta * r;
            v = act4(v, act, lo, hi);
        }
        if (full4) {
            *reinterpret_cast<f4 *>(dst) = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < ncol) dst[e] = v[e];
        }
    }
}

// The written-out order takes registers (164 instead of 128 at 64 columns, three waves a SIMD instead of
// four), which short loops over many rows miss more than they gain: with K of 64 and 256 in this order
// the bottleneck b32 takes 231 us instead of 228; K of 768 gains (the layers above).
template <int RN>
static SplitKernel pick(int am, int kchunk) {
    return am == AM_VEC     ? (kchunk >= 512 ? &gemm_split_kernel<RN, 4, 3, AM_VEC, true> : &gemm_split_kernel<RN, 4, 3, AM_VEC>)
           : am == AM_CAT   ? &gemm_split_kernel<RN, 4, 3, AM_CAT>
           : am == AM_LOOSE ? &gemm_split_kernel<RN, 4, 3, AM_LOOSE>
           : am == AM_TAP   ? &gemm_split_kernel<RN, 4, 3, AM_TAP>
                            : &gemm_split_kernel<RN, 4, 3, AM_CONV_VEC>;
}

template <int RN, int WAVES>
static SplitKernel pick_small(int am) {
    return am == AM_VEC   ? &gemm_split_small_kernel<RN, WAVES, AM_VEC>
           : am == AM_CAT ? &gemm_split_small_kernel<RN, WAVES, AM_CAT>
           : am == AM_TAP ? &gemm_split_small_kernel<RN, WAVES, AM_TAP>
                          : &gemm_split_small_kernel<RN, WAVES, AM_CONV_VEC>;
}

SplitKernel pick_split(int am, int bm, int bn, int kchunk) {
    if (bm == 32 && am == AM_LOOSE) return &gemm_split_small_kernel<1, 8, AM_LOOSE>;  // bn 32 only: registers
    if (bm == 32) return bn == 64 ? pick_small<2, 8>(am) : pick_small<1, 8>(am);
    return bn == 128 ? pick<4>(am, kchunk) : pick<2>(am, kchunk);
}

}  // namespace mgc
