// Cholesky factor and its inverse of the subspace matrices on gfx950:
// A = U^H U and U^-1, real and complex FP64, one launch per 32 columns.
//
// Right-looking by 32 x 32 blocks.  The rows [A | 1] are eliminated together,
// so U^-H = (U^-1)^H comes out of the same launches: step k has one workgroup per
// trailing block (i, j), i <= j, one per block (i, j), j <= k < i, of the right
// hand side, and one per finished block.  Every workgroup eliminates the diagonal
// block again beside the one or two panel blocks that it needs (in registers,
// lanes 0 - 31 of a wave the diagonal block's columns, lanes 32 - 63 a panel
// block's), which costs nothing on an idle chip and leaves no data to wait for
// inside a launch.  Bound by that serial chain of 32 pivots.  The cooperative
// kernel before it held one grid barrier and ~23 us a step, and the triangular
// inverse (or the triangular solves in its place) followed as library launches:
// n = 384 real 275 + 70 -> 155 us (12.9 us a step), n = 135 complex (rocSOLVER,
// rocBLAS before) ~600 -> 86 us.
#include "qm_internal.h"
#include "qm_mfma.h"
#include "qm_wave.h"

namespace qm {
namespace {

constexpr int NB = 32;
constexpr int kCholMaxN = 1024;  // 32 launches; larger orders are for the library

struct cplx {
    double re, im;
};
__device__ __forceinline__ double real_of(double a) { return a; }
__device__ __forceinline__ double real_of(cplx a) { return a.re; }
__device__ __forceinline__ double conj_of(double a) { return a; }
__device__ __forceinline__ cplx conj_of(cplx a) { return {a.re, -a.im}; }
__device__ __forceinline__ double times(double a, double s) { return a * s; }
__device__ __forceinline__ cplx times(cplx a, double s) { return {a.re * s, a.im * s}; }
__device__ __forceinline__ double lane_of(double a, int l) { return lane_value(a, l); }
__device__ __forceinline__ cplx lane_of(cplx a, int l) { return {lane_value(a.re, l), lane_value(a.im, l)}; }
// a - conj(u) x
__device__ __forceinline__ double minus_conj(double a, double u, double x) { return fma(-u, x, a); }
__device__ __forceinline__ cplx minus_conj(cplx a, cplx u, cplx x) {
    return {fma(-u.im, x.im, fma(-u.re, x.re, a.re)), fma(u.im, x.re, fma(-u.re, x.im, a.im))};
}
template <typename T>
__device__ __forceinline__ T value(double re);
template <>
__device__ __forceinline__ double value<double>(double re) { return re; }
template <>
__device__ __forceinline__ cplx value<cplx>(double re) { return {re, 0.0}; }

// 1 / sqrt(x): the hardware's estimate and two Newton steps
__device__ __forceinline__ double inv_sqrt(double x) {
    double y = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int i = 0; i < 2; ++i) y = fma(0.5 * y, fma(-x * y, y, 1.0), y);
    return y;
}

// Step k (see the file comment).  M (k = 0: A, later W) holds the trailing
// matrix in its blocks (i, j), i <= j, and W the right hand side's blocks (i, j), i
// > j, once they differ from the identity.  Blocks of x: 0 the diagonal block, 1
// .. k the finished blocks (k, j) of the right hand side, then the r (r + 1) / 2
// trailing blocks and the r (k + 1) blocks of the right hand side, r = P - 1 - k.
template <typename T>
__global__ __launch_bounds__(256) void chol_step_kernel(const T *__restrict__ A, T *W, T *__restrict__ U,
                                                        T *__restrict__ Ui, int n, int k, int P, int *info) {
    using M = Mfma<double>;
    __shared__ T Ls[NB][NB + 1], Rs[NB][NB + 1];
    const T *src = k == 0 ? A : W;
    const int r = P - 1 - k, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, k0 = k * NB;
    int id = blockIdx.x;
    // block row i and column j of the updated block; i = k: none is updated
    int i = k, j = k;
    bool rhs = true;  // the right block belongs to the right hand side
    if (id >= 1 && id <= k) {
        j = id - 1;
    } else if (id > k) {
        id -= 1 + k;
        if (id < r * (r + 1) / 2) {
            rhs = false;
            int row = 0;
            for (int c = r; id >= c; --c) {  // rows of r, r - 1, .. blocks
                id -= c;
                ++row;
            }
            i = k + 1 + row;
            j = i + id;
        } else {
            id -= r * (r + 1) / 2;
            i = k + 1 + id / (k + 1);
            j = id % (k + 1);
        }
    }
    if (wave < 2) {
        T a[NB];
        // column of the lane: the diagonal block's, or the wave's panel block's
        const bool diag = lane < NB;
        const int l = lane & (NB - 1);
        const int cb = diag ? k : (wave == 0 ? i : j), col = cb * NB + l;
        const bool ident = !diag && wave == 1 && rhs && j == k;
        const T *p = src + (int64_t)min(col, n - 1) * n;
        T raw[NB];
#pragma unroll
        for (int q = 0; q < NB; ++q) raw[q] = p[min(k0 + q, n - 1)];
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            const bool in = k0 + q < n && col < n && (!diag || q <= l);
            T v = in ? raw[q] : value<T>(diag && q == l && col >= n ? 1.0 : 0.0);
            if (ident) v = value<T>(q == l ? 1.0 : 0.0);
            if (diag && q == l) v = value<T>(real_of(v));
            a[q] = v;
        }
        int bad = 0;
#pragma unroll
        for (int q = 0; q < NB; ++q) {
            double piv = lane_value(real_of(a[q]), q);
            if (!(piv > 0.0)) {
                if (bad == 0) bad = k0 + q + 1;
                piv = 1.0;
            }
            const T u = times(a[q], inv_sqrt(piv));
            a[q] = u;
#pragma unroll
            for (int s = q + 1; s < NB; ++s) a[s] = minus_conj(a[s], lane_of(u, s), u);
        }
        if (!diag) {
#pragma unroll
            for (int q = 0; q < NB; ++q) (wave == 0 ? Ls : Rs)[q][l] = a[q];
        }
        if (wave == 0 && blockIdx.x == 0) {
            if (diag && col < n) {
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    if (q <= l && k0 + q < n) U[(int64_t)col * n + k0 + q] = a[q];
            }
            if (tid == 0 && (k == 0 || *info == 0)) *info = bad;
        }
        if (wave == 1 && !diag && col < n) {
            if (i == k) {  // a finished block of U^-H, stored as one of U^-1
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    if (k0 + q < n) {
                        Ui[(int64_t)(k0 + q) * n + col] = conj_of(a[q]);
                        if (j < k) Ui[(int64_t)col * n + k0 + q] = value<T>(0.0);
                    }
            } else if (!rhs && i == j) {
#pragma unroll
                for (int q = 0; q < NB; ++q)
                    if (k0 + q < n) U[(int64_t)col * n + k0 + q] = a[q];
            }
        }
    }
    if (i == k) return;  // the whole workgroup
    __syncthreads();
    // block (i, j) -= Ls^H Rs, a 16 x 16 quadrant a wave
    const int jj = lane & 15, g = lane >> 4, qi = (wave & 1) * 16, qj = (wave >> 1) * 16;
    M::acc_t re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < NB / 4; ++s) {
        const T x = Ls[4 * s + g][qi + jj], y = Rs[4 * s + g][qj + jj];
        if constexpr (sizeof(T) == 8) {
            re = M::mma(x, y, re);
        } else {
            re = M::mma(x.re, y.re, re);
            re = M::mma(x.im, y.im, re);
            im = M::mma(x.re, y.im, im);
            im = M::mma(-x.im, y.re, im);
        }
    }
    const int col = j * NB + qj + jj;
    if (col >= n) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int row = i * NB + qi + M::row(g, q);
        if (row >= n) continue;
        const int64_t at = (int64_t)col * n + row;
        T v = rhs && j == k ? value<T>(0.0) : src[at];
        if constexpr (sizeof(T) == 8) {
            v -= re[q];
        } else {
            v.re -= re[q];
            v.im -= im[q];
        }
        W[at] = v;
    }
}

template <typename T>
int launch(int n, const T *A, T *W, T *U, T *Ui, int *info, hipStream_t st) {
    const int P = (n + NB - 1) / NB;
    for (int k = 0; k < P; ++k) {
        const int r = P - 1 - k;
        hipLaunchKernelGGL(chol_step_kernel<T>, dim3(1 + k + r * (r + 1) / 2 + r * (k + 1)), dim3(256), 0, st, A, W,
                           U, Ui, n, k, P, info);
        QM_HIP(hipGetLastError());
    }
    return QM_OK;
}

}  // namespace

int chol_inverse_supported(int n) { return n >= 1 && n <= kCholMaxN; }

int chol_inverse(int n, bool cplx_, const void *A, void *W, void *U, void *Ui, int *info, hipStream_t st) {
    QM_CHECK(chol_inverse_supported(n), QM_ERR_ARG, "Cholesky: order");
    return cplx_ ? launch<cplx>(n, (const cplx *)A, (cplx *)W, (cplx *)U, (cplx *)Ui, info, st)
                 : launch<double>(n, (const double *)A, (double *)W, (double *)U, (double *)Ui, info, st);
}

}  // namespace qm
