// The FP32 update Y = Z C on the bf16 matrix cores (gfx950).
//
// The FP32 MFMA runs at 157 TFLOP/s, the bf16 one at 2.5 PFLOP/s.  Every FP32
// value is the exact sum of three bf16 values (8 significant bits each, rounded
// to nearest: x = h + m + l), so a product of two is the sum of nine bf16
// products, each exact in the FP32 accumulator's input.  The three smallest
// (m l, l m, l l: below 2^-26 of the product together, where an FP32 product
// rounds at 2^-24) are left out; the other six are accumulated in FP32.
//
// The bf16 MFMA rounds its sums downward, where the FP32 one rounds to nearest: left
// alone the mean error of all outputs is -0.10 of their rms error at m = 1024, -0.18
// at 3072.  The panels of the second and third quarter of K are therefore summed with
// the other sign (C's values and the accumulators turn there and back), which takes
// out a constant as well as a linearly growing drift: at most 0.01 on inputs of
// mixed or one sign, 0.04 where the terms grow along K.
//
// Measured (before: the FP32 MFMA kernels of blas.hip): 1536 x 1024 over 884,736
// points 21.5 -> 14.0 ms (130 -> 199 TFLOP/s), 384 x 256 over 262,144 points 440 -> 329
// us, 600 x 400 over 157,685 points (no multiple of their tiles) 1128 -> 540 us.  Error
// against 64 bits 2.2e-7 .. 9.9e-7 -> 1.8e-7 .. 8.4e-7 (m = 256 .. 3072).  The matrix
// core is busy for half of the time (at 2.1 GHz); the splits and the barrier of each
// panel take the rest.  Reading each operand a group of products earlier changed
// nothing; 128 columns a workgroup throughout, two workgroups a CU, cost 11 %.
//
// Three bf16 values hold 24 bits from 2^-110 on (the last bit of l is then a bf16
// value).  Both operands are therefore multiplied by 2^40 as they are split, which
// brings FP32's smallest subnormal there, and the sums by 2^-80 as they are stored:
// no value loses bits, also where tiny ones stand beside ordinary ones.  (Before,
// values below 2^-110 did: a column of 1e-36 among ordinary ones was passed on with
// 14 bits.)  What leaves the range at its other end (values from 2^88, sums from 2^48,
// infinities) leaves a sum that is not finite; the workgroup then computes its tile
// again on the FP32 MFMA, so that such inputs give what they always gave.  That takes
// 3.5 times as long (50 ms for the first shape above).  NaN stays NaN in every product.
#include <algorithm>
#include <cmath>
#include <cstdint>

#include "qm_cols.h"
#include "qm_internal.h"

namespace qm {
namespace {

typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
typedef float f2_t __attribute__((ext_vector_type(2)));
typedef float f16_t __attribute__((ext_vector_type(16)));
typedef float f4_t __attribute__((ext_vector_type(4)));

// x scale = h + m + l, 8 values at a time
typedef uint32_t u4_t __attribute__((ext_vector_type(4)));
struct Split {
    u4_t h, m, l;  // 8 bf16 values each
};
__device__ __forceinline__ float wide_lo(bf2_t p) {
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, p) << 16);
}
__device__ __forceinline__ float wide_hi(bf2_t p) {
    return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, p) & 0xffff0000u);
}
__device__ __forceinline__ Split split8(const float (&x)[8], float scale) {
    Split s;
    // in pairs: one conversion instruction each
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
        const f2_t v = {x[e] * scale, x[e + 1] * scale};
        const bf2_t h = __builtin_convertvector(v, bf2_t);
        const f2_t r = {v[0] - wide_lo(h), v[1] - wide_hi(h)};
        const bf2_t m = __builtin_convertvector(r, bf2_t);
        const f2_t t = {r[0] - wide_lo(m), r[1] - wide_hi(m)};
        const bf2_t l = __builtin_convertvector(t, bf2_t);
        s.h[e / 2] = __builtin_bit_cast(uint32_t, h);
        s.m[e / 2] = __builtin_bit_cast(uint32_t, m);
        s.l[e / 2] = __builtin_bit_cast(uint32_t, l);
    }
    return s;
}

__device__ __forceinline__ int xcd_block(int nblk, int per_xcd) {
    const int b = blockIdx.x;
    const int lb = (b & 7) * per_xcd + (b >> 3);
    return lb < nblk ? lb : -1;
}

constexpr float kScale = 0x1p40f, kUnscale = 0x1p-80f;  // of each operand, and of the sums
constexpr int SG_THREADS = 512, SG_K = 16;  // 8 waves; K rows per panel (one MFMA deep)
constexpr int SG_PAD = 8;  // puts the two K halves of an index on different LDS banks

// acc += the six products of one panel; a lane's units: u[split][k half][index]
template <int TA, int TB, int LA, int LB>
__device__ __forceinline__ void panel_products(f16_t (&acc)[TA][TB], const bf8_t (&as)[3][2][LA],
                                               const bf8_t (&bs)[3][2][LB], int wa, int wb, int lane) {
    const int i = lane & 31, kh = lane >> 5;
    bf8_t a[TA], b[3][TB];
    auto load_a = [&](int s) {
#pragma unroll
        for (int t = 0; t < TA; ++t) a[t] = as[s][kh][wa + 32 * t + i];
    };
    auto load_b = [&](int s) {
#pragma unroll
        for (int t = 0; t < TB; ++t) b[s][t] = bs[s][kh][wb + 32 * t + i];
    };
    auto mma = [&](int s) {
#pragma unroll
        for (int x = 0; x < TA; ++x)
#pragma unroll
            for (int y = 0; y < TB; ++y)
                acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[x], b[s][y], acc[x][y], 0, 0, 0);
    };
    load_a(2);
    load_b(0);
    mma(0);
    load_a(1);
    mma(0);
    load_b(1);
    mma(1);
    load_a(0);
    mma(1);
    load_b(2);
    mma(2);
    mma(0);
}
// row of result item r of a 32 x 32 tile (its column is lane % 32)
__device__ __forceinline__ int sg_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }

// Y^T (n x Ng) = C^T (n x m) Z^T (m x Ng): UN columns x 256 points a workgroup, 8
// waves as 2 x 4 of (UN / 2) x 64.  Per panel each thread loads 8 consecutive K of
// one point (8 columns of Z, lanes along the points) and of one column of C,
// splits them and writes 16-byte units [split][k half][index] that are read back
// as whole MFMA operands: reads and writes run through consecutive units.
constexpr int SU_P = 256;
template <int UN>
__global__ __launch_bounds__(SG_THREADS) void split_update_kernel(ColBlocks Z, ColBlocks Y,
                                                                  const float *__restrict__ Cm, int m, int n,
                                                                  int64_t ng, int tiles_n, int nblk, int per_xcd) {
    constexpr int TA = UN / 64, TB = 2;
    __shared__ bf8_t cs[2][3][2][UN + SG_PAD];
    __shared__ bf8_t zs[2][3][2][SU_P];
    const int lb = xcd_block(nblk, per_xcd);
    if (lb < 0) return;
    const int c0 = (lb % tiles_n) * UN;  // column tile fastest: neighbours share Z in one XCD's L2
    const int64_t p0 = (int64_t)(lb / tiles_n) * SU_P;
    const int npanel = (m + SG_K - 1) / SG_K;
    const int turn = npanel / 4;  // panels from turn to 3 turn are summed with the other sign (see the file comment)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int zi = threadIdx.x & (SU_P - 1), zh = wave >> 2;
    const bool cload = 2 * UN == SG_THREADS || threadIdx.x < 2 * UN;  // whole waves
    const int ci = (threadIdx.x >> 1) & (UN - 1), ch = threadIdx.x & 1;
    // points and columns past the end are computed on the last one and not stored
    const int64_t zp = min(p0 + zi, ng - 1);
    const Cols<float> zcols(Z, ng);
    const uint32_t coff = ((uint32_t)min(c0 + ci, n - 1) * m + 8 * ch) * 4u;
    // C through a buffer resource: the last panel may read past a column's end,
    // and past the array's end it gets zeros
    const __amdgpu_buffer_rsrc_t crsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(Cm), 0,
                                                                          (int)((uint32_t)m * n * 4u), 0x20000);
    float zv[8], cv[8];
    // Straight-line: a branch around the loads would make their results meet
    // at its end, and wait there.  K past m is read from column m - 1 (cleared in
    // store), and threads without a column of C read another's again.
    auto fetch = [&](int p) {
        const int kz = p * SG_K + 8 * zh;
        const int end = zcols.end(min(kz, m - 1));
        GlobalPtr<float> zc = zcols.at(min(kz, m - 1));
        const GlobalPtr<float> znext = zcols.at(min(end, m - 1));
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            zv[e] = zc[zp];
            zc = kz + e + 1 == end ? znext : (kz + e + 1 < m ? zc + ng : zc);
        }
        const uint32_t o = coff + p * (SG_K * 4);
        const f4_t v0 = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(crsrc, o, 0, 0));
        const f4_t v1 = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(crsrc, o + 16, 0, 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            cv[e] = v0[e];
            cv[4 + e] = v1[e];
        }
    };
    auto store = [&](int buf, int p) {
        if ((p + 1) * SG_K > m) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                zv[e] = p * SG_K + 8 * zh + e < m ? zv[e] : 0.0f;
                cv[e] = p * SG_K + 8 * ch + e < m ? cv[e] : 0.0f;
            }
        }
        const Split z = split8(zv, kScale);
        zs[buf][0][zh][zi] = __builtin_bit_cast(bf8_t, z.h);
        zs[buf][1][zh][zi] = __builtin_bit_cast(bf8_t, z.m);
        zs[buf][2][zh][zi] = __builtin_bit_cast(bf8_t, z.l);
        if (cload) {
            const Split c = split8(cv, p >= turn && p < 3 * turn ? -kScale : kScale);
            cs[buf][0][ch][ci] = __builtin_bit_cast(bf8_t, c.h);
            cs[buf][1][ch][ci] = __builtin_bit_cast(bf8_t, c.m);
            cs[buf][2][ch][ci] = __builtin_bit_cast(bf8_t, c.l);
        }
    };
    const int wc = (wave & 1) * (UN / 2), wp = (wave >> 1) * 64;
    f16_t acc[TA][TB];
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b) acc[a][b] = f16_t{};
    auto turn_sign = [&]() {
#pragma unroll
        for (int a = 0; a < TA; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b) acc[a][b] = -acc[a][b];
    };
    fetch(0);
    store(0, 0);
    fetch(min(1, npanel - 1));
    __syncthreads();
    for (int p = 0; p < npanel; ++p) {
        const int cur = p & 1;
        if (turn > 0 && (p == turn || p == 3 * turn)) turn_sign();
        // the two waves of a SIMD split the next panel on either side of their
        // products, so that one of them keeps the matrix core busy
        // (the fetch's scheduling apart: mixed with the splits, its results were copied,
        // and waited for, right behind the loads, 15.4 ms instead of 14.0)
        if (wave < 4) {
            store(cur ^ 1, p + 1);
            __builtin_amdgcn_sched_barrier(0);
            fetch(min(p + 2, npanel - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
        panel_products<TA, TB>(acc, cs[cur], zs[cur], wc, wp, lane);
        if (wave >= 4) {
            store(cur ^ 1, p + 1);
            __builtin_amdgcn_sched_barrier(0);
            fetch(min(p + 2, npanel - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
        __syncthreads();
    }
    const int i = lane & 31, kh = lane >> 5;
    const Cols<float> ycols(Y, ng);
    bool finite = true;
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                finite = finite && fabsf(acc[a][b][r]) < HUGE_VALF;
                acc[a][b][r] *= kUnscale;
            }
    if (__syncthreads_or(!finite)) {
#pragma unroll
        for (int a = 0; a < TA; ++a)
#pragma unroll
            for (int b = 0; b < TB; ++b) acc[a][b] = f16_t{};
#pragma unroll 4
        for (int k = 0; k < m; k += 2) {
            const int kk = k + kh;
            float av[TA], bv[TB];
#pragma unroll
            for (int a = 0; a < TA; ++a) {
                const float v = Cm[(int64_t)min(c0 + wc + 32 * a + i, n - 1) * m + min(kk, m - 1)];
                av[a] = kk < m ? v : 0.0f;
            }
            const GlobalPtr<float> zc = zcols.at(min(kk, m - 1));
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                const float v = zc[min(p0 + wp + 32 * b + i, ng - 1)];
                bv[b] = kk < m ? v : 0.0f;
            }
#pragma unroll
            for (int a = 0; a < TA; ++a)
#pragma unroll
                for (int b = 0; b < TB; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[a], bv[b], acc[a][b], 0, 0, 0);
        }
    }
#pragma unroll
    for (int a = 0; a < TA; ++a)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int col = c0 + wc + 32 * a + sg_row(r, lane);
            if (col >= n) continue;
            const GlobalPtr<float> yc = ycols.at(col) + p0;
#pragma unroll
            for (int b = 0; b < TB; ++b)
                if (p0 + wp + 32 * b + i < ng) yc[wp + 32 * b + i] = acc[a][b][r];
        }
}

}  // namespace

// 8 consecutive columns of Z lie in at most two blocks (blocks between others
// are at least 8 columns wide), C's byte offsets fit 32 bits, and the launch has
// 3 workgroups for every 4 CUs
bool split_update_fits(const ColBlocks &Z, int m, int n, int64_t ng) {
    for (int b = 1; b + 1 < Z.nblk; ++b)
        if (Z.ncols[b] < 8) return false;
    return (int64_t)m * n < ((int64_t)1 << 30) && (ng + SU_P - 1) / SU_P * ((n + 255) / 256) >= 192;
}

int split_update(const ColBlocks &Z, const ColBlocks &Y, const float *Cm, int m, int n, int64_t ng, hipStream_t st) {
    const int r = n % 256;
    const int un = r > 0 && r <= 128 ? 128 : 256;
    const int tiles_n = (n + un - 1) / un;
    const int64_t nblk = (ng + SU_P - 1) / SU_P * tiles_n;
    QM_CHECK(nblk < ((int64_t)1 << 30), QM_ERR_ARG, "update: grid too large");
    const int per_xcd = (int)((nblk + 7) / 8);
    if (un == 256)
        hipLaunchKernelGGL(split_update_kernel<256>, dim3((unsigned)(8 * per_xcd)), dim3(SG_THREADS), 0, st, Z, Y, Cm,
                           m, n, ng, tiles_n, (int)nblk, per_xcd);
    else
        hipLaunchKernelGGL(split_update_kernel<128>, dim3((unsigned)(8 * per_xcd)), dim3(SG_THREADS), 0, st, Z, Y, Cm,
                           m, n, ng, tiles_n, (int)nblk, per_xcd);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

}  // namespace qm
