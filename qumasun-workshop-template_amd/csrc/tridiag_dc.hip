// Eigenpairs of a real symmetric tridiagonal matrix by divide and conquer on
// gfx950: all eigenvalues, the nev lowest eigenvectors.
//
// Cuppen's splitting T = diag(T1, T2) + |rho| u u^T with the deflation of
// Dongarra and Sorensen; the secular equation by R.-C. Li's "middle way"
// iteration (LAPACK Working Note 89) safeguarded by bisection, each root held
// as an offset from its nearest pole; eigenvectors from Gu and Eisenstat's
// recomputed z (SIAM J. Matrix Anal. Appl. 16, 1995), so they are orthogonal to
// working precision however close the roots are.
//
// The tree has 2^L leaves of at most kLeaf rows, one wave each, and every
// level is four launches over all of its nodes, with no size read back by the
// host: prep (z, sorting, deflation), roots (a wave per root), zhat (a wave per
// component, and the final order), vectors (the eigenvectors of the rank-one
// problem built in LDS and multiplied onto the node's on MFMA; at the top only
// the nev wanted columns).  Latency bound: ~39 us a level.  rocSOLVER's stedc
// before it solves the merges of a level in one serial kernel, computes every
// vector and reads its status back: n = 384 with 128 vectors 1780 -> 275 us,
// n = 135 with 45 820 -> 190 us (kernel time).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>

#include "qm_internal.h"
#include "qm_mfma.h"
#include "qm_wave.h"
#include "secular.h"

namespace qm {
namespace {

constexpr int kLeaf = 16;
constexpr int kMaxOrder = 1024;         // LDS of the prep and root kernels

// Device arrays of one solve (n values each), in the work buffer after the two
// n x n eigenvector buffers.
struct DcWork {
    double *d, *e;          // scaled diagonal with the split offsets taken off, off-diagonal
    double *val;            // eigenvalues of the level below, ascending inside each node
    double *dl, *zl;        // undeflated poles and z of a node (first k of its range)
    double *tau, *lam;      // root offsets; new eigenvalues (k roots, then the deflated ones)
    double *zh;             // recomputed z
    double *rc, *rs;        // deflating rotations
    double *scal;           // [0]: the power of two T was divided by
    int *col, *org, *src;   // old columns (k undeflated, then deflated); root origins; rank -> index
    int *rp, *rn;           // columns of the rotations
    int *k, *nrot;          // per node
};

// first row of node i at depth l
__host__ __device__ __forceinline__ int node_start(int n, int l, int i) { return (int)(((int64_t)i * n) >> l); }

// scale, split offsets; *info = 1 for a non-finite input (T is then taken as 0)
__global__ __launch_bounds__(256) void dc_init_kernel(DcWork w, const double *__restrict__ d,
                                                      const double *__restrict__ e, int n, int L, int *info) {
    __shared__ double red[256];
    double m = 0.0;
    int bad = 0;
    for (int i = threadIdx.x; i < n; i += 256) {
        const double a = fabs(d[i]), b = i + 1 < n ? fabs(e[i]) : 0.0;
        if (!isfinite(a) || !isfinite(b)) bad = 1;
        m = fmax(m, fmax(a, b));
    }
    red[threadIdx.x] = m;
    bad = __syncthreads_or(bad);
    for (int s = 128; s >= 1; s >>= 1) {
        if ((int)threadIdx.x < s) red[threadIdx.x] = fmax(red[threadIdx.x], red[threadIdx.x + s]);
        __syncthreads();
    }
    m = red[0];
    int ex = 0;
    if (!bad && m > 0.0) (void)frexp(m, &ex);
    ex = min(ex, 1023);  // 2^ex is multiplied back in; entries from 2^1023 on become at most 2
    for (int i = threadIdx.x; i < n; i += 256) {
        double a = bad ? 0.0 : ldexp(d[i], -ex);
        const double b = bad || i + 1 >= n ? 0.0 : ldexp(e[i], -ex);
        // the split before row s takes |e[s-1]| off rows s - 1 and s; rows i and
        // i + 1 are in different leaves when a leaf starts at i + 1
        const int leaf = (int)((((int64_t)(i + 1) << L) - 1) / n);  // last leaf with start <= i
        if (i > 0 && node_start(n, L, leaf) == i) a -= fabs(ldexp(e[i - 1], -ex));
        if (i + 1 < n && node_start(n, L, leaf + 1) == i + 1) a -= fabs(b);
        w.d[i] = bad ? 0.0 : a;
        w.e[i] = b;
    }
    if (threadIdx.x == 0) {
        w.scal[0] = ldexp(1.0, ex);
        *info = bad;
    }
}

__global__ __launch_bounds__(256) void dc_zero_kernel(double *__restrict__ p, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0.0;
}

// column `c`, row `r` of an eigenvector matrix: real, or complex with a zero imaginary part
template <bool CPLX>
__device__ __forceinline__ void put(double *q, int64_t ld, int r, int64_t c, double v) {
    if constexpr (CPLX) {
        q[2 * (r + c * ld)] = v;
        q[2 * (r + c * ld) + 1] = 0.0;
    } else {
        q[r + c * ld] = v;
    }
}

// One leaf by implicit QR steps with Wilkinson's shift (Golub and Van Loan,
// Matrix Computations, 8.3), one wave: every lane runs the scalar recurrence,
// lane r applies the rotations to row r of the vectors, whose running column
// stays in a register.  top: the leaf is the whole matrix (vectors limited to
// nev, eigenvalues scaled back into wout).  A serial chain of ~1.5 m^2 / 2
// rotations; cyclic Jacobi on the same leaves (12 rows) took 149 us, this 79.
template <bool CPLX>
__global__ __launch_bounds__(64) void dc_leaf_kernel(DcWork w, double *__restrict__ q, int ld, int n, int L, int nev,
                                                     double *wout, int max_steps, int *info) {
    __shared__ double V[kLeaf][kLeaf + 1], a[kLeaf + 2], b[kLeaf + 2];
    const int s0 = node_start(n, L, blockIdx.x), m = node_start(n, L, blockIdx.x + 1) - s0;
    const int lane = threadIdx.x, row = lane & (kLeaf - 1);
    if (lane < kLeaf + 2) {
        a[lane] = lane < m ? w.d[s0 + lane] : 0.0;
        b[lane] = lane + 1 < m ? w.e[s0 + lane] : 0.0;
    }
    for (int i = lane; i < kLeaf * kLeaf; i += 64) V[i / kLeaf][i % kLeaf] = i / kLeaf == i % kLeaf ? 1.0 : 0.0;
    __syncthreads();
    int hi = m - 1, steps = 0;
    while (hi > 0 && steps < max_steps) {
        // the unreduced block [lo, hi]: negligible couplings are zeroed
        int lo = hi;
        while (lo > 0 && fabs(b[lo - 1]) > kEps * (fabs(a[lo - 1]) + fabs(a[lo]))) --lo;
        if (lo > 0) b[lo - 1] = 0.0;
        if (lo == hi) {
            --hi;
            continue;
        }
        ++steps;
        const double bl = b[hi - 1], del = 0.5 * (a[hi - 1] - a[hi]);
        const double mu = a[hi] - bl * (bl / (del + copysign(hypot(del, bl), del)));
        double ak = a[lo], bk = b[lo], x = ak - mu, z = bk, vk = V[row][lo];
        double an = a[lo + 1], bn = b[lo + 1], vn = V[row][lo + 1];
        for (int k = lo; k < hi; ++k) {
            // the elements of the next step, requested before this one's chain
            const double an2 = a[min(k + 2, m)], bn2 = b[min(k + 2, m)], vn2 = V[row][min(k + 2, kLeaf - 1)];
            double r = sqrt(fma(x, x, z * z));
            if (!(r > 1.0e-140)) r = hypot(x, z);
            const double ri = 1.0 / r, c = r > 0.0 ? x * ri : 1.0, s = r > 0.0 ? z * ri : 0.0;
            if (k > lo) b[k - 1] = r;
            // rotation in the plane (k, k + 1)
            const double t = s * (an - ak) + 2.0 * c * bk;
            const double dk = ak + s * t, dn = an - s * t;
            const double off = c * t - bk;
            a[k] = dk;
            V[row][k] = c * vk + s * vn;
            vk = c * vn - s * vk;
            x = off;
            z = s * bn;
            ak = dn;
            bk = c * bn;
            if (k + 1 == hi) {
                a[hi] = dn;
                b[k] = off;
                V[row][hi] = vk;
            }
            an = an2;
            bn = bn2;
            vn = vn2;
        }
    }
    __syncthreads();
    if (lane < m) {
        const double v = a[lane];
        int rank = 0;
        for (int i = 0; i < m; ++i) rank += a[i] < v || (a[i] == v && i < lane);
        if (wout) wout[s0 + rank] = v * w.scal[0];
        w.val[s0 + rank] = v;
        if (rank < nev)
            for (int r = 0; r < m; ++r) put<CPLX>(q, ld, s0 + r, s0 + rank, V[r][lane]);
    }
    if (lane == 0 && hi > 0) *info = kDcUnconverged;
}

// exclusive prefix sum of one flag per element over nn <= kMaxOrder elements,
// element i of thread i / 4; returns the total.  cnt: 256 ints of LDS.
__device__ __forceinline__ int flag_scan(const unsigned char *flag, int nn, int *cnt, int (&at)[4]) {
    int c = 0;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int i = threadIdx.x * 4 + u;
        at[u] = c;
        if (i < nn && flag[i]) ++c;
    }
    cnt[threadIdx.x] = c;
    __syncthreads();
    for (int s = 1; s < 256; s <<= 1) {
        const int v = (int)threadIdx.x >= s ? cnt[threadIdx.x - s] : 0;
        __syncthreads();
        cnt[threadIdx.x] += v;
        __syncthreads();
    }
    const int total = cnt[255], base = cnt[threadIdx.x] - c;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) at[u] += base;
    return total;
}

// One workgroup per node: z, the poles sorted, deflation.  A pole deflates when
// its z is negligible, and the lower of two close poles when the rotation that
// zeroes its z leaves a negligible off-diagonal; both tests run for all poles
// at once, and one thread follows the chains of close pairs only.
__global__ __launch_bounds__(256) void dc_prep_kernel(DcWork w, const double *__restrict__ q, int n, int l) {
    __shared__ double d[kMaxOrder], z[kMaxOrder], vals[kMaxOrder];
    __shared__ int col[kMaxOrder], sv[kMaxOrder], cnt[256];
    __shared__ unsigned char keep[kMaxOrder];
    __shared__ unsigned long long close[kMaxOrder / 64];
    __shared__ double red[8];
    const int node = blockIdx.x, s0 = node_start(n, l, node), s1 = node_start(n, l, node + 1),
              mid = node_start(n, l + 1, 2 * node + 1), nn = s1 - s0, n1 = mid - s0, tid = threadIdx.x;
    const double rho_s = w.e[mid - 1], rho = 2.0 * fabs(rho_s), isq2 = 0.70710678118654752440;
    for (int i = tid; i < nn; i += 256) vals[i] = w.val[s0 + i];
    if (tid < kMaxOrder / 64) close[tid] = 0;
    __syncthreads();
    double dm = 0.0, zm = 0.0;
    for (int i = tid; i < nn; i += 256) {
        const double v = vals[i];
        // place in the merged order: values of the other half below v (at or below for the second half)
        int lo = i < n1 ? n1 : 0, hi = i < n1 ? nn : n1;
        const int b = lo;
        while (lo < hi) {
            const int mm = (lo + hi) >> 1;
            if (i < n1 ? vals[mm] < v : vals[mm] <= v) lo = mm + 1;
            else hi = mm;
        }
        const int r = (i < n1 ? i : i - n1) + lo - b;
        const double zz = i < n1 ? q[(mid - 1) + (int64_t)(s0 + i) * n]
                                 : copysign(1.0, rho_s) * q[mid + (int64_t)(s0 + i) * n];
        d[r] = v;
        z[r] = zz * isq2;
        col[r] = s0 + i;
        dm = fmax(dm, fabs(v));
        zm = fmax(zm, fabs(zz * isq2));
    }
    for (int x = 32; x >= 1; x >>= 1) {
        dm = fmax(dm, __shfl_xor(dm, x));
        zm = fmax(zm, __shfl_xor(zm, x));
    }
    if ((tid & 63) == 0) {
        red[tid >> 6] = dm;
        red[4 + (tid >> 6)] = zm;
    }
    __syncthreads();
    dm = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
    zm = fmax(fmax(red[4], red[5]), fmax(red[6], red[7]));
    const double tol = 8.0 * kEps * fmax(dm, zm);
    const bool none = rho * zm <= tol;
    for (int i = tid; i < nn; i += 256) keep[i] = !none && rho * fabs(z[i]) > tol;
    __syncthreads();
    int at[4];
    const int ns = flag_scan(keep, nn, cnt, at);
    for (int u = 0; u < 4; ++u) {
        const int i = tid * 4 + u;
        if (i < nn && keep[i]) sv[at[u]] = i;
    }
    __syncthreads();
    for (int a = tid; a + 1 < ns; a += 256) {
        const int p = sv[a], s = sv[a + 1];
        const double t = d[s] - d[p];
        if (fabs(t * z[p] * z[s]) <= tol * (z[p] * z[p] + z[s] * z[s]))
            atomicOr(&close[a >> 6], 1ull << (a & 63));
    }
    __syncthreads();
    if (tid == 0) {
        int nr = 0;
        bool chain = false;  // the pole before was rotated into this one: its test is no longer the one above
        for (int a = 0; a + 1 < ns;) {
            if (!chain) {  // next flagged pair
                int wd = a >> 6;
                unsigned long long m = close[wd] >> (a & 63) << (a & 63);
                while (m == 0 && ++wd < kMaxOrder / 64) m = close[wd];
                if (m == 0) break;
                a = wd * 64 + __ffsll(m) - 1;
            }
            const int p = sv[a], s = sv[a + 1];
            const double zp = z[p], zs = z[s], dp = d[p], ds = d[s], t = ds - dp;
            chain = fabs(t * zp * zs) <= tol * (zp * zp + zs * zs);
            if (chain) {
                const double tau = hypot(zs, zp), c = zs / tau, sn = -zp / tau;
                z[s] = tau;
                z[p] = 0.0;
                d[p] = dp * c * c + ds * sn * sn;
                d[s] = dp * sn * sn + ds * c * c;
                keep[p] = 0;
                w.rp[s0 + nr] = col[p];
                w.rn[s0 + nr] = col[s];
                w.rc[s0 + nr] = c;
                w.rs[s0 + nr] = sn;
                ++nr;
            }
            ++a;
        }
        w.nrot[node] = nr;
    }
    __syncthreads();
    const int k = flag_scan(keep, nn, cnt, at);
    if (tid == 0) w.k[node] = k;
    for (int u = 0; u < 4; ++u) {
        const int i = tid * 4 + u;
        if (i >= nn) continue;
        if (keep[i]) {
            w.dl[s0 + at[u]] = d[i];
            w.zl[s0 + at[u]] = z[i];
            w.col[s0 + at[u]] = col[i];
        } else {
            const int o = k + i - at[u];
            w.lam[s0 + o] = d[i];
            w.col[s0 + o] = col[i];
        }
    }
}

// Roots of 1/rho + sum z_i^2 / (d_i - x) of every node, a wave each (blocks
// y < yroot, 4 roots a block); the blocks after them apply the node's deflating
// rotations to its old eigenvectors, a thread per row.
__global__ __launch_bounds__(256) void dc_root_kernel(DcWork w, double *__restrict__ q, int n, int l, int yroot,
                                                      int max_steps, int *info) {
    __shared__ double d[kMaxOrder], z2[kMaxOrder];
    const int node = blockIdx.x, s0 = node_start(n, l, node), s1 = node_start(n, l, node + 1), tid = threadIdx.x;
    if ((int)blockIdx.y >= yroot) {
        const int r = s0 + ((int)blockIdx.y - yroot) * 256 + tid, nr = w.nrot[node];
        if (r >= s1) return;
        int last = -1;
        double x = 0.0;
        constexpr int B = 8;  // a rotation's second column is not touched before it: load them together
        for (int t0 = 0; t0 < nr; t0 += B) {
            double y[B];
#pragma unroll
            for (int u = 0; u < B; ++u) y[u] = q[r + (int64_t)w.rn[s0 + min(t0 + u, nr - 1)] * n];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int t = t0 + u;
                if (t >= nr) break;
                const int p = w.rp[s0 + t];
                if (p != last) {
                    if (last >= 0) q[r + (int64_t)last * n] = x;
                    x = q[r + (int64_t)p * n];
                }
                const double c = w.rc[s0 + t], s = w.rs[s0 + t];
                q[r + (int64_t)p * n] = c * x + s * y[u];
                x = c * y[u] - s * x;
                last = w.rn[s0 + t];
            }
        }
        if (last >= 0) q[r + (int64_t)last * n] = x;
        return;
    }
    const int k = w.k[node];
    if ((int)blockIdx.y * 4 >= k) return;
    const int mid = node_start(n, l + 1, 2 * node + 1);
    const double rho = 2.0 * fabs(w.e[mid - 1]);
    for (int i = tid; i < k; i += 256) {
        const double z = w.zl[s0 + i];
        d[i] = w.dl[s0 + i];
        z2[i] = z * z;
    }
    __syncthreads();
    const int j = blockIdx.y * 4 + (tid >> 6), lane = tid & 63;
    if (j >= k) return;  // no barrier below
    int org;
    double tau;
    const bool ok = secular_root(j, k, d, z2, rho, lane, 64, [](double v) { return wave_sum(v); }, max_steps, &org, &tau);
    if (lane == 0) {
        w.tau[s0 + j] = tau;
        w.org[s0 + j] = org;
        w.lam[s0 + j] = d[org] + tau;
        if (!ok) *info = kDcUnconverged;
    }
}

// |zhat_i|^2 = prod_j (lam_j - d_i) / prod_{j != i} (d_j - d_i), a wave per
// component (blocks y < yz); the blocks after them order the node's new
// eigenvalues (top: scaled back into wout).
__global__ __launch_bounds__(256) void dc_zhat_kernel(DcWork w, int n, int l, int yz, double *wout) {
    __shared__ double a[kMaxOrder];
    const int node = blockIdx.x, s0 = node_start(n, l, node), nn = node_start(n, l, node + 1) - s0, tid = threadIdx.x;
    if ((int)blockIdx.y >= yz) {
        for (int i = tid; i < nn; i += 256) a[i] = w.lam[s0 + i];
        __syncthreads();
        const int e = ((int)blockIdx.y - yz) * 256 + tid;
        if (e >= nn) return;
        const double v = a[e];
        int r = 0;
        for (int i = 0; i < nn; ++i) r += a[i] < v || (a[i] == v && i < e);
        w.src[s0 + r] = e;
        w.val[s0 + r] = v;
        if (wout) wout[s0 + r] = v * w.scal[0];
        return;
    }
    const int k = w.k[node];
    if ((int)blockIdx.y * 4 >= k) return;
    for (int i = tid; i < k; i += 256) a[i] = w.dl[s0 + i];
    __syncthreads();
    const int i = blockIdx.y * 4 + (tid >> 6), lane = tid & 63;
    if (i >= k) return;  // no barrier below
    const double di = a[i];
    double p = 1.0;
    for (int j = lane; j < k; j += 64) {
        const double x = (di - a[w.org[s0 + j]]) - w.tau[s0 + j];
        p *= j == i ? x : x / (di - a[j]);
    }
    p = wave_prod(p);
    if (lane == 0) w.zh[s0 + i] = copysign(sqrt(fabs(p)), w.zl[s0 + i]);
}

// 16 new eigenvectors of a node: the rank-one problem's vectors zhat_i / (d_i -
// lam_j) for 16 ranks in LDS, times the node's old undeflated columns (A[row][i]
// = column col_i, 16 rows a wave).  Deflated ranks copy their old column.
// Blocks: x = node, y = column tile, z = group of 4 row tiles.
template <bool CPLX>
__global__ __launch_bounds__(256) void dc_vec_kernel(DcWork w, double *__restrict__ out, int ldo,
                                                     const double *__restrict__ q, int n, int l, int ncols) {
    extern __shared__ __align__(16) double dc_lds[];
    using M = Mfma<double>;
    __shared__ double part[16][16];
    __shared__ int src[16];
    const int node = blockIdx.x, s0 = node_start(n, l, node), nn = node_start(n, l, node + 1) - s0, tid = threadIdx.x;
    const int c0 = blockIdx.y * 16, nc = min(ncols, nn);
    if (c0 >= nc || (int)blockIdx.z * 64 >= nn) return;
    const int k = w.k[node], kp = (k + 3) & ~3;
    double *S = dc_lds;                              // [kp][16]
    int *col = reinterpret_cast<int *>(S + (size_t)kp * 16);
    if (tid < 16) src[tid] = c0 + tid < nc ? w.src[s0 + c0 + tid] : nn;
    for (int i = tid; i < kp; i += 256) col[i] = i < k ? w.col[s0 + i] : s0;
    __syncthreads();
    {
        const int c = tid & 15, j = src[c];
        double s = 0.0, tau = 0.0, dj = 0.0;
        if (j < k) {
            tau = w.tau[s0 + j];
            dj = w.dl[s0 + w.org[s0 + j]];
        }
        for (int i = tid >> 4; i < kp; i += 16) {
            double v = 0.0;
            if (j < k && i < k) v = w.zh[s0 + i] / ((w.dl[s0 + i] - dj) - tau);
            S[(size_t)i * 16 + c] = v;
            s = fma(v, v, s);
        }
        part[tid >> 4][c] = s;
    }
    __syncthreads();
    const int lane = tid & 63, j = lane & 15, g = lane >> 4;
    const int r0 = (blockIdx.z * 4 + (tid >> 6)) * 16;
    if (r0 >= nn) return;  // no barrier below
    double nrm = 0.0;
#pragma unroll
    for (int i = 0; i < 16; ++i) nrm += part[i][j];
    const double inv = 1.0 / sqrt(nrm);
    const int row = s0 + min(r0 + j, nn - 1);
    typename M::acc_t acc = {0, 0, 0, 0};
    for (int i0 = 0; i0 < kp; i0 += 32) {
        double av[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) av[u] = q[row + (int64_t)col[min(i0 + 4 * u + g, kp - 1)] * n];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (i0 + 4 * u < kp) acc = M::mma(av[u], S[(size_t)(i0 + 4 * u + g) * 16 + j], acc);
    }
    const int e = src[j];
    if (c0 + j >= nc) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int x = r0 + M::row(g, r);
        if (x >= nn) continue;
        const double v = e < k ? acc[r] * inv : q[s0 + x + (int64_t)w.col[s0 + e] * n];
        put<CPLX>(out, ldo, s0 + x, s0 + c0 + j, v);
    }
}

int depth_of(int n) {
    int L = 0;
    while (((n + (1 << L) - 1) >> L) > kLeaf) ++L;
    return L;
}

// qm_dc_set_step_limit, process-wide
std::atomic<int> g_dc_step_limit{INT32_MAX};

}  // namespace

int tridiag_dc_max() { return kMaxOrder; }

int tridiag_dc_supported(int n) { return n >= 1 && n <= kMaxOrder; }

size_t tridiag_dc_work_bytes(int n) {
    const size_t m = (size_t)n + 1;
    return sizeof(double) * (2 * (size_t)n * n + 11 * m) + sizeof(int) * 7 * m + 64;
}

template <bool CPLX>
static int solve(int n, int nev, const double *d, const double *e, double *w, double *Z, int ldz, void *work,
                 int *info, hipStream_t st) {
    double *buf[2] = {static_cast<double *>(work), static_cast<double *>(work) + (size_t)n * n};
    const size_t m = (size_t)n + 1;
    double *p = buf[1] + (size_t)n * n;
    DcWork k;
    for (double **a : {&k.d, &k.e, &k.val, &k.dl, &k.zl, &k.tau, &k.lam, &k.zh, &k.rc, &k.rs, &k.scal}) {
        *a = p;
        p += m;
    }
    int *ip = reinterpret_cast<int *>(p);
    for (int **a : {&k.col, &k.org, &k.src, &k.rp, &k.rn, &k.k, &k.nrot}) {
        *a = ip;
        ip += m;
    }
    // steps of a secular root, and of a leaf's QR iteration (~2 a row)
    const int root_steps = std::min(g_dc_step_limit.load(), kMaxSteps);
    const int leaf_steps = std::min(g_dc_step_limit.load(), 40 * kLeaf);
    const int L = depth_of(n);
    hipLaunchKernelGGL(dc_init_kernel, dim3(1), dim3(256), 0, st, k, d, e, n, L, info);
    QM_HIP(hipGetLastError());
    if (L == 0) {
        hipLaunchKernelGGL(dc_leaf_kernel<CPLX>, dim3(1), dim3(64), 0, st, k, Z, ldz, n, 0, nev, w, leaf_steps, info);
        QM_HIP(hipGetLastError());
        return QM_OK;
    }
    // a level writes its nodes' diagonal blocks only: what lies between them stays zero
    hipLaunchKernelGGL(dc_zero_kernel, dim3((unsigned)std::min<int64_t>((2 * (int64_t)n * n + 255) / 256, 2048)),
                       dim3(256), 0, st, buf[0], 2 * (int64_t)n * n);
    QM_HIP(hipGetLastError());
    hipLaunchKernelGGL(dc_leaf_kernel<false>, dim3(1 << L), dim3(64), 0, st, k, buf[0], n, n, L, n, (double *)nullptr,
                       leaf_steps, info);
    QM_HIP(hipGetLastError());
    int cur = 0;
    for (int l = L - 1; l >= 0; --l) {
        const int nodes = 1 << l, nn = (n + nodes - 1) >> l;  // rows of the largest node
        const int y4 = (nn + 3) / 4, y256 = (nn + 255) / 256;
        double *q = buf[cur];
        hipLaunchKernelGGL(dc_prep_kernel, dim3(nodes), dim3(256), 0, st, k, q, n, l);
        QM_HIP(hipGetLastError());
        hipLaunchKernelGGL(dc_root_kernel, dim3(nodes, y4 + y256), dim3(256), 0, st, k, q, n, l, y4, root_steps,
                           info);
        QM_HIP(hipGetLastError());
        hipLaunchKernelGGL(dc_zhat_kernel, dim3(nodes, y4 + y256), dim3(256), 0, st, k, n, l, y4,
                           l == 0 ? w : nullptr);
        QM_HIP(hipGetLastError());
        const size_t lds = (size_t)((nn + 3) & ~3) * (16 * sizeof(double) + sizeof(int));
        const int cols = l == 0 ? nev : nn;
        const dim3 grid(nodes, (cols + 15) / 16, (nn + 63) / 64);
        auto *vk = l == 0 ? dc_vec_kernel<CPLX> : dc_vec_kernel<false>;
        if (lds > (size_t)60 * 1024)
            QM_HIP(hipFuncSetAttribute((const void *)vk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        if (l == 0) hipLaunchKernelGGL(vk, grid, dim3(256), lds, st, k, Z, ldz, (const double *)q, n, l, cols);
        else hipLaunchKernelGGL(vk, grid, dim3(256), lds, st, k, buf[1 - cur], n, (const double *)q, n, l, cols);
        QM_HIP(hipGetLastError());
        cur = 1 - cur;
    }
    return QM_OK;
}

int tridiag_dc(int n, int nev, const double *d, const double *e, double *w, double *Z, int ldz, bool cplx, void *work,
               int *info, hipStream_t st) {
    QM_CHECK(tridiag_dc_supported(n) && nev >= 1 && nev <= n, QM_ERR_ARG, "tridiagonal eigensolve: order or nev");
    return cplx ? solve<true>(n, nev, d, e, w, Z, ldz, work, info, st)
                : solve<false>(n, nev, d, e, w, Z, ldz, work, info, st);
}

}  // namespace qm

extern "C" int qm_dc_set_step_limit(int steps) {
    QM_CHECK(steps >= 0, QM_ERR_ARG, "qm_dc_set_step_limit: steps must be >= 0");
    qm::g_dc_step_limit.store(steps);
    return QM_OK;
}
