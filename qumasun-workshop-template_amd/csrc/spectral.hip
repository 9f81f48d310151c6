// Spectral kinetic operator on gfx950 without a 3-D transform.
//
// |G + k|^2 / 2 is a sum over the axes, so
//   IFFT(|G + k|^2 / 2 FFT psi) = F_xy^-1 ((q_x^2 + q_y^2) / 2) F_xy psi + F_z^-1 (q_z^2 / 2) F_z psi,
// and e^{-i dt |G + k|^2 / 2} is the product of the same two parts.  Each part
// is one kernel that transforms, scales and transforms back inside LDS: no
// spectrum in memory, no packing (OperateKineticInKspace_bundle,
// qumasun_base1.matrix.h:96-130, and mEvolveK_FFT,
// qumasun_symplectic.kinetic_fft.h:65-140, are the operators).  Bound by HBM: 5
// blocks of traffic per kinetic apply (read psi, write out; read psi, read and
// write out) instead of the ~14 of pack, two 3-D library transforms, scaling
// and unpack.  64^3 x 64 complex FP64 (268 MB a block): 737 -> 351 us (3.8 TB/s),
// 128 real FP32 bands 457 -> 191 us.  The error against extended precision (80-bit
// transforms, rms) is smaller too, 64 x 48 x 40 3.0e-16 for 5.1e-16, FP32 1.34e-7 for
// 2.19e-7: a transform's rounding is scaled by its own axes' q^2 only.  (Against a
// 64-bit transform, itself 5e-16 off, it can read larger.)
//
// Transforms are in place in LDS: decimation in frequency forward (natural
// order in, digit-reversed out), the mirrored decimation in time back, so
// nothing is reordered; the scale factor looks its frequency up by position.
// The first forward and the last inverse stage run straight from and to
// global memory, and the last forward stage, the factor and the first inverse
// stage stay in registers.  Lanes run across transforms (columns of the plane
// for y, rows for x at an odd pitch, grid points for z), so every LDS access
// is conflict-free and a stage's twiddles are the same for a whole wave.
//
// Real (Gamma) bands: two real lines of one band are one complex line (planes
// z and z + 1 in the plane kernel, points p and p + C in the line kernel); the
// operator is real there, so the parts do not mix, and bands never share a
// transform.
#include <algorithm>
#include <cmath>
#include <functional>
#include <memory>
#include <vector>

#include "qm_internal.h"

namespace qm {
namespace {

template <typename T>
struct alignas(2 * sizeof(T)) Cx {
    T x, y;
};

constexpr int kMaxStages = 8;
struct Axis {
    int n, ns;
    int r[kMaxStages];  // radices, in forward order; their product is n
    int off;            // of the axis in the twiddle and frequency tables
    double g, k;        // 2 pi / L and the k component
};

template <typename T>
__device__ __forceinline__ Cx<T> cadd(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ Cx<T> csub(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
// a w, or a conj(w)
template <bool CONJ, typename T>
__device__ __forceinline__ Cx<T> ctw(Cx<T> a, Cx<T> w) {
    if constexpr (CONJ) return {a.x * w.x + a.y * w.y, a.y * w.x - a.x * w.y};
    return {a.x * w.x - a.y * w.y, a.x * w.y + a.y * w.x};
}
// -i a forward, +i a inverse
template <bool INV, typename T>
__device__ __forceinline__ Cx<T> crot(Cx<T> a) {
    if constexpr (INV) return {-a.y, a.x};
    return {a.y, -a.x};
}

// cos and sin of 2 pi q / R, q = 1 .. (R - 1) / 2
template <int R> struct Roots;
template <> struct Roots<3> {
    static constexpr double c[1] = {-0.5};
    static constexpr double s[1] = {0.866025403784438646764};
};
template <> struct Roots<5> {
    static constexpr double c[2] = {0.309016994374947424102, -0.809016994374947424102};
    static constexpr double s[2] = {0.951056516295153572116, 0.587785252292473129169};
};
template <> struct Roots<7> {
    static constexpr double c[3] = {0.623489801858733530525, -0.222520933956314404289, -0.900968867902419126236};
    static constexpr double s[3] = {0.781831482468029808708, 0.974927912181823607018, 0.433883739117558120476};
};
template <> struct Roots<11> {
    static constexpr double c[5] = {0.841253532831181168862, 0.415415013001886425529, -0.142314838273285140444,
                                    -0.654860733945285064057, -0.959492973614497389890};
    static constexpr double s[5] = {0.540640817455597582108, 0.909631995354518371412, 0.989821441880932732376,
                                    0.755749574354258283774, 0.281732556841429697711};
};
template <> struct Roots<13> {
    static constexpr double c[6] = {0.885456025653209895900, 0.568064746731155802512, 0.120536680255323053349,
                                    -0.354604887042535625970, -0.748510748171101098635, -0.970941817426052027157};
    static constexpr double s[6] = {0.464723172043768545656, 0.822983865893656394580, 0.992708874098053992801,
                                    0.935016242685414823440, 0.663122658240795202377, 0.239315664287557767149};
};

// a := sum_q a_q e^{-+ 2 pi i p q / R}
template <int R, bool INV, typename T>
__device__ __forceinline__ void dft(Cx<T> (&a)[R]) {
    if constexpr (R == 2) {
        const Cx<T> t = csub(a[0], a[1]);
        a[0] = cadd(a[0], a[1]);
        a[1] = t;
    } else if constexpr (R == 4) {
        const Cx<T> s02 = cadd(a[0], a[2]), d02 = csub(a[0], a[2]), s13 = cadd(a[1], a[3]);
        const Cx<T> d13 = crot<INV>(csub(a[1], a[3]));
        a[0] = cadd(s02, s13);
        a[1] = cadd(d02, d13);
        a[2] = csub(s02, s13);
        a[3] = csub(d02, d13);
    } else if constexpr (R == 8) {
        Cx<T> e[4] = {a[0], a[2], a[4], a[6]}, o[4] = {a[1], a[3], a[5], a[7]};
        dft<4, INV>(e);
        dft<4, INV>(o);
        const T h = T(0.707106781186547524401);
        const Cx<T> r1 = crot<INV>(o[1]), r3 = crot<INV>(o[3]);
        o[1] = {h * (o[1].x + r1.x), h * (o[1].y + r1.y)};
        o[2] = crot<INV>(o[2]);
        o[3] = {h * (r3.x - o[3].x), h * (r3.y - o[3].y)};
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            a[p] = cadd(e[p], o[p]);
            a[p + 4] = csub(e[p], o[p]);
        }
    } else {
        constexpr int H = (R - 1) / 2;
        Cx<T> s[H], d[H];
#pragma unroll
        for (int q = 1; q <= H; ++q) {
            s[q - 1] = cadd(a[q], a[R - q]);
            d[q - 1] = csub(a[q], a[R - q]);
        }
        const Cx<T> a0 = a[0];
#pragma unroll
        for (int q = 0; q < H; ++q) a[0] = cadd(a[0], s[q]);
#pragma unroll
        for (int p = 1; p <= H; ++p) {
            Cx<T> u = a0, v = {T(0), T(0)};
#pragma unroll
            for (int q = 1; q <= H; ++q) {
                const int t = (p * q) % R;
                const T c = T(Roots<R>::c[(t <= H ? t : R - t) - 1]);
                const T sn = t <= H ? T(Roots<R>::s[t <= H ? t - 1 : 0]) : -T(Roots<R>::s[t <= H ? 0 : R - t - 1]);
                u.x += c * s[q - 1].x;
                u.y += c * s[q - 1].y;
                v.x += sn * d[q - 1].x;
                v.y += sn * d[q - 1].y;
            }
            const Cx<T> w = crot<INV>(v);
            a[p] = cadd(u, w);
            a[R - p] = csub(u, w);
        }
    }
}

// One stage of W side-by-side transforms of length n, on sub-blocks of length
// L = R m: element e of transform c is ld(c, e), and st(c, e, value).  Forward:
// R-point transforms at stride m, then the twiddles; inverse: the mirror image.
template <typename T, int R, bool INV, typename Ld, typename St>
__device__ __forceinline__ void stage_r(Ld &&ld, St &&st, int W, int n, int L, const Cx<T> *tw) {
    const int m = L / R, step = n / L, total = W * (n / R);
    for (int i = threadIdx.x; i < total; i += blockDim.x) {
        const int b = (unsigned)i / (unsigned)W, c = i - b * W;
        const int blk = (unsigned)b / (unsigned)m, j = b - blk * m;
        const int e0 = blk * L + j;
        Cx<T> a[R];
#pragma unroll
        for (int q = 0; q < R; ++q) a[q] = ld(c, e0 + q * m);
        if constexpr (INV) {
#pragma unroll
            for (int q = 1; q < R; ++q) a[q] = ctw<true>(a[q], tw[j * q * step]);
        }
        dft<R, INV>(a);
        if constexpr (!INV) {
#pragma unroll
            for (int q = 1; q < R; ++q) a[q] = ctw<false>(a[q], tw[j * q * step]);
        }
#pragma unroll
        for (int q = 0; q < R; ++q) st(c, e0 + q * m, a[q]);
    }
}

// The last forward stage (L = R), f(c, e, value) on the spectrum, and the first
// inverse stage, which works on the same elements
template <typename T, int R, typename Ld, typename St, typename F>
__device__ __forceinline__ void mid_r(Ld &&ld, St &&st, F &&f, int W, int n) {
    const int total = W * (n / R);
    for (int i = threadIdx.x; i < total; i += blockDim.x) {
        const int b = (unsigned)i / (unsigned)W, c = i - b * W, e0 = b * R;
        Cx<T> a[R];
#pragma unroll
        for (int q = 0; q < R; ++q) a[q] = ld(c, e0 + q);
        dft<R, false>(a);
#pragma unroll
        for (int q = 0; q < R; ++q) a[q] = f(c, e0 + q, a[q]);
        dft<R, true>(a);
#pragma unroll
        for (int q = 0; q < R; ++q) st(c, e0 + q, a[q]);
    }
}

// BIG: with the radices 11 and 13.  Grids without them take kernels without
// them, because the widest stage sets a kernel's registers: FP64 plane kernel 83
// VGPRs for 126, line kernel 99 for 175 (4 waves per SIMD for 2).
#define QM_RADIX(r, CALL)                            \
    switch (r) {                                     \
        case 2: CALL(2); break;                      \
        case 3: CALL(3); break;                      \
        case 4: CALL(4); break;                      \
        case 5: CALL(5); break;                      \
        case 7: CALL(7); break;                      \
        case 8: CALL(8); break;                      \
        default:                                     \
            if constexpr (BIG) {                     \
                if (r == 11) CALL(11);               \
                else CALL(13);                       \
            }                                        \
    }

template <typename T, bool BIG, bool INV, typename Ld, typename St>
__device__ __forceinline__ void stage(int r, Ld &&ld, St &&st, int W, int n, int L, const Cx<T> *tw) {
#define QM_CALL(R) stage_r<T, R, INV>(ld, st, W, n, L, tw)
    QM_RADIX(r, QM_CALL)
#undef QM_CALL
}

template <typename T, bool BIG, typename Ld, typename St, typename F>
__device__ __forceinline__ void mid(int r, Ld &&ld, St &&st, F &&f, int W, int n) {
#define QM_CALL(R) mid_r<T, R>(ld, st, f, W, n)
    QM_RADIX(r, QM_CALL)
#undef QM_CALL
}

// value times the factor of the squared wave vector q2 = sum of q_d^2 over the
// part's axes.  MODE 0: q2 / 2 * scale (kinetic operator); MODE 1:
// e^{-i dt q2 / 2} * scale (kinetic propagator).  The factor is FP64 in both precisions.
template <typename T, int MODE>
__device__ __forceinline__ Cx<T> kfactor(Cx<T> v, double q2, double scale, double dt) {
    if constexpr (MODE == 0) {
        const T f = (T)(0.5 * q2 * scale);
        return {v.x * f, v.y * f};
    }
    double sn, cs;
    sincos(-dt * (0.5 * q2), &sn, &cs);
    return ctw<false>(v, Cx<T>{(T)(cs * scale), (T)(sn * scale)});
}

// The xy part: one workgroup per complex plane (ny rows of nx at LDS pitch
// `pitch`).  Complex bands: plane z of a band's (re, im) columns; real bands:
// planes z, z + 1 of one column.  out = part psi + V psi (MODE 0), or psi <-
// part psi in place (MODE 1, out == psi: a workgroup has read its plane before
// it writes).  NC: components per band.  Workgroup size and LDS: plane_shape.
template <typename T, int MODE, int NC, bool BIG>
__global__ __launch_bounds__(1024) void spectral_plane_kernel(T *out, const T *psi, const T *__restrict__ vloc,
                                                              const Cx<T> *__restrict__ twt,
                                                              const int *__restrict__ freq, int64_t ng, int nz,
                                                              int pitch, Axis ax, Axis ay, double scale, double dt) {
    extern __shared__ __align__(16) unsigned char spectral_lds[];
    Cx<T> *twx = reinterpret_cast<Cx<T> *>(spectral_lds), *twy = twx + ax.n, *s = twy + ay.n;
    const int nx = ax.n, ny = ay.n, plane = nx * ny;
    const int npl = NC == 2 ? nz : (nz + 1) / 2;
    const int u = blockIdx.x;
    const int band = u / npl, z = (u - band * npl) * (NC == 2 ? 1 : 2);
    const int64_t re = (int64_t)band * NC * ng + (int64_t)z * plane;
    const int64_t im = re + (NC == 2 ? ng : plane);
    const bool has_im = NC == 2 || z + 1 < nz;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) twx[i] = twt[ax.off + i];
    for (int i = threadIdx.x; i < ny; i += blockDim.x) twy[i] = twt[ay.off + i];
    __syncthreads();
    const int *fx = freq + ax.off, *fy = freq + ay.off;
    // transforms along y: c is the column, e the row; along x: c the row, e the column
    auto ldg = [&](int c, int e) -> Cx<T> {
        const int i = e * nx + c;
        return {psi[re + i], has_im ? psi[im + i] : T(0)};
    };
    auto stg = [&](int c, int e, Cx<T> v) {
        const int i = e * nx + c;
        if constexpr (MODE == 0) {
            const T *vp = vloc + (int64_t)z * plane;
            v.x += vp[i] * psi[re + i];
            if (has_im) v.y += vp[(NC == 2 ? 0 : plane) + i] * psi[im + i];
        }
        out[re + i] = v.x;
        if (has_im) out[im + i] = v.y;
    };
    auto ldy = [&](int c, int e) { return s[e * pitch + c]; };
    auto sty = [&](int c, int e, Cx<T> v) { s[e * pitch + c] = v; };
    auto ldx = [&](int c, int e) { return s[c * pitch + e]; };
    auto stx = [&](int c, int e, Cx<T> v) { s[c * pitch + e] = v; };
    int L = ny;
    for (int q = 0; q < ay.ns; ++q) {
        if (q == 0) stage<T, BIG, false>(ay.r[q], ldg, sty, nx, ny, L, twy);
        else stage<T, BIG, false>(ay.r[q], ldy, sty, nx, ny, L, twy);
        L /= ay.r[q];
        __syncthreads();
    }
    L = nx;
    for (int q = 0; q < ax.ns - 1; ++q) {
        stage<T, BIG, false>(ax.r[q], ldx, stx, ny, nx, L, twx);
        L /= ax.r[q];
        __syncthreads();
    }
    mid<T, BIG>(ax.r[ax.ns - 1], ldx, stx,
           [&](int c, int e, Cx<T> v) {
               const double qx = ax.g * (double)fx[e] + ax.k, qy = ay.g * (double)fy[c] + ay.k;
               return kfactor<T, MODE>(v, qx * qx + qy * qy, scale, dt);
           },
           ny, nx);
    __syncthreads();
    for (int q = ax.ns - 2; q >= 0; --q) {
        L *= ax.r[q];
        stage<T, BIG, true>(ax.r[q], ldx, stx, ny, nx, L, twx);
        __syncthreads();
    }
    L = 1;
    for (int q = ay.ns - 1; q >= 0; --q) {
        L *= ay.r[q];
        if (q == 0) stage<T, BIG, true>(ay.r[q], ldy, stg, nx, ny, L, twy);
        else stage<T, BIG, true>(ay.r[q], ldy, sty, nx, ny, L, twy);
        __syncthreads();
    }
}

// The z part: one workgroup per C complex lines along z.  Complex bands: C grid
// points of a band's (re, im) columns; real bands: points p .. p + C - 1 and
// p + C .. p + 2 C - 1 of one column.  out += part psi (MODE 0), or psi <- part
// psi in place (MODE 1).
template <typename T, int MODE, int NC, bool BIG>
__global__ __launch_bounds__(256) void spectral_line_kernel(T *out, const T *psi, const Cx<T> *__restrict__ twt,
                                                            const int *__restrict__ freq, int64_t ng, int plane,
                                                            int tiles, int C, Axis az, double scale, double dt) {
    extern __shared__ __align__(16) unsigned char spectral_lds[];
    Cx<T> *tw = reinterpret_cast<Cx<T> *>(spectral_lds), *s = tw + az.n;
    const int n = az.n;
    const int band = blockIdx.x / tiles;
    const int p0 = (blockIdx.x - band * tiles) * (NC == 2 ? C : 2 * C);
    const int64_t re = (int64_t)band * NC * ng + p0;
    const int64_t im = NC == 2 ? re + ng : re + C;
    const int nre = min(C, plane - p0), nim = NC == 2 ? nre : plane - p0 - C;  // lanes with a point
    for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = twt[az.off + i];
    __syncthreads();
    const int *fz = freq + az.off;
    auto ldg = [&](int c, int e) -> Cx<T> {
        const int64_t i = (int64_t)e * plane + c;
        return {c < nre ? psi[re + i] : T(0), c < nim ? psi[im + i] : T(0)};
    };
    auto stg = [&](int c, int e, Cx<T> v) {
        const int64_t i = (int64_t)e * plane + c;
        if (c < nre) out[re + i] = MODE == 0 ? out[re + i] + v.x : v.x;
        if (c < nim) out[im + i] = MODE == 0 ? out[im + i] + v.y : v.y;
    };
    auto lds = [&](int c, int e) { return s[e * C + c]; };
    auto sts = [&](int c, int e, Cx<T> v) { s[e * C + c] = v; };
    auto fac = [&](int c, int e, Cx<T> v) {
        const double q = az.g * (double)fz[e] + az.k;
        return kfactor<T, MODE>(v, q * q, scale, dt);
    };
    if (az.ns == 1) {
        mid<T, BIG>(az.r[0], ldg, stg, fac, C, n);
        return;
    }
    int L = n;
    for (int q = 0; q < az.ns - 1; ++q) {
        if (q == 0) stage<T, BIG, false>(az.r[q], ldg, sts, C, n, L, tw);
        else stage<T, BIG, false>(az.r[q], lds, sts, C, n, L, tw);
        L /= az.r[q];
        __syncthreads();
    }
    mid<T, BIG>(az.r[az.ns - 1], lds, sts, fac, C, n);
    __syncthreads();
    for (int q = az.ns - 2; q >= 0; --q) {
        L *= az.r[q];
        if (q == 0) stage<T, BIG, true>(az.r[q], lds, stg, C, n, L, tw);
        else stage<T, BIG, true>(az.r[q], lds, sts, C, n, L, tw);
        __syncthreads();
    }
}

// ---- Poisson solve ---------------------------------------------------------
// 4 pi / |G|^2 is no sum over the axes, so the spectrum of the one real FP64
// field goes through memory, and three kernels take the place of a library
// transform pair and the scaling pass.  Latency bound (64^3 is 4 MB of spectrum):
// 28 us of kernels for 31, two launches fewer, and the first solve of a context
// builds small tables instead of library plans (4.4 -> 0.35 ms for the fields'
// first pass); the fields' sequence 137 -> 125 us.

// spec plane z = F_xy of real plane z, in the transforms' output positions
template <bool BIG>
__global__ __launch_bounds__(1024) void poisson_forward_kernel(Cx<double> *__restrict__ spec,
                                                               const double *__restrict__ rho,
                                                               const Cx<double> *__restrict__ twt, int pitch, Axis ax,
                                                               Axis ay) {
    using T = double;
    extern __shared__ __align__(16) unsigned char spectral_lds[];
    Cx<T> *twx = reinterpret_cast<Cx<T> *>(spectral_lds), *twy = twx + ax.n, *s = twy + ay.n;
    const int nx = ax.n, ny = ay.n, plane = nx * ny;
    const int64_t base = (int64_t)blockIdx.x * plane;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) twx[i] = twt[ax.off + i];
    for (int i = threadIdx.x; i < ny; i += blockDim.x) twy[i] = twt[ay.off + i];
    __syncthreads();
    auto ldg = [&](int c, int e) -> Cx<T> { return {rho[base + e * nx + c], 0.0}; };
    auto ldy = [&](int c, int e) { return s[e * pitch + c]; };
    auto sty = [&](int c, int e, Cx<T> v) { s[e * pitch + c] = v; };
    auto ldx = [&](int c, int e) { return s[c * pitch + e]; };
    auto stx = [&](int c, int e, Cx<T> v) { s[c * pitch + e] = v; };
    int L = ny;
    for (int q = 0; q < ay.ns; ++q) {
        if (q == 0) stage<T, BIG, false>(ay.r[q], ldg, sty, nx, ny, L, twy);
        else stage<T, BIG, false>(ay.r[q], ldy, sty, nx, ny, L, twy);
        L /= ay.r[q];
        __syncthreads();
    }
    L = nx;
    for (int q = 0; q < ax.ns; ++q) {
        stage<T, BIG, false>(ax.r[q], ldx, stx, ny, nx, L, twx);
        L /= ax.r[q];
        __syncthreads();
    }
    for (int i = threadIdx.x; i < plane; i += blockDim.x) {
        const int y = (unsigned)i / (unsigned)nx;
        spec[base + i] = s[y * pitch + i - y * nx];
    }
}

// C lines along z of the spectrum: forward, 4 pi / |G|^2 / N (0 at G = 0), back
template <bool BIG>
__global__ __launch_bounds__(256) void poisson_line_kernel(Cx<double> *__restrict__ spec,
                                                           const Cx<double> *__restrict__ twt,
                                                           const int *__restrict__ freq, int plane, int C, Axis ax,
                                                           Axis ay, Axis az, double scale) {
    using T = double;
    extern __shared__ __align__(16) unsigned char spectral_lds[];
    Cx<T> *tw = reinterpret_cast<Cx<T> *>(spectral_lds), *s = tw + az.n;
    const int n = az.n, p0 = blockIdx.x * C, nc = min(C, plane - p0);
    for (int i = threadIdx.x; i < n; i += blockDim.x) tw[i] = twt[az.off + i];
    __syncthreads();
    auto ldg = [&](int c, int e) -> Cx<T> {
        return c < nc ? spec[(int64_t)e * plane + p0 + c] : Cx<T>{0.0, 0.0};
    };
    auto stg = [&](int c, int e, Cx<T> v) {
        if (c < nc) spec[(int64_t)e * plane + p0 + c] = v;
    };
    auto lds = [&](int c, int e) { return s[e * C + c]; };
    auto sts = [&](int c, int e, Cx<T> v) { s[e * C + c] = v; };
    auto fac = [&](int c, int e, Cx<T> v) -> Cx<T> {
        const int p = min(p0 + c, plane - 1), y = (unsigned)p / (unsigned)ax.n, x = p - y * ax.n;
        const double qx = ax.g * (double)freq[ax.off + x], qy = ay.g * (double)freq[ay.off + y],
                     qz = az.g * (double)freq[az.off + e];
        const double e2 = 0.5 * (qx * qx + qy * qy + qz * qz);
        const double f = e2 == 0.0 ? 0.0 : 2.0 * M_PI / e2 * scale;
        return {v.x * f, v.y * f};
    };
    if (az.ns == 1) {
        mid<T, BIG>(az.r[0], ldg, stg, fac, C, n);
        return;
    }
    int L = n;
    for (int q = 0; q < az.ns - 1; ++q) {
        if (q == 0) stage<T, BIG, false>(az.r[q], ldg, sts, C, n, L, tw);
        else stage<T, BIG, false>(az.r[q], lds, sts, C, n, L, tw);
        L /= az.r[q];
        __syncthreads();
    }
    mid<T, BIG>(az.r[az.ns - 1], lds, sts, fac, C, n);
    __syncthreads();
    for (int q = az.ns - 2; q >= 0; --q) {
        L *= az.r[q];
        if (q == 0) stage<T, BIG, true>(az.r[q], lds, stg, C, n, L, tw);
        else stage<T, BIG, true>(az.r[q], lds, sts, C, n, L, tw);
        __syncthreads();
    }
}

// plane z of V_H = the real part of F_xy^-1 of spectrum plane z
template <bool BIG>
__global__ __launch_bounds__(1024) void poisson_inverse_kernel(double *__restrict__ vh,
                                                               const Cx<double> *__restrict__ spec,
                                                               const Cx<double> *__restrict__ twt, int pitch, Axis ax,
                                                               Axis ay) {
    using T = double;
    extern __shared__ __align__(16) unsigned char spectral_lds[];
    Cx<T> *twx = reinterpret_cast<Cx<T> *>(spectral_lds), *twy = twx + ax.n, *s = twy + ay.n;
    const int nx = ax.n, ny = ay.n, plane = nx * ny;
    const int64_t base = (int64_t)blockIdx.x * plane;
    for (int i = threadIdx.x; i < nx; i += blockDim.x) twx[i] = twt[ax.off + i];
    for (int i = threadIdx.x; i < ny; i += blockDim.x) twy[i] = twt[ay.off + i];
    for (int i = threadIdx.x; i < plane; i += blockDim.x) {
        const int y = (unsigned)i / (unsigned)nx;
        s[y * pitch + i - y * nx] = spec[base + i];
    }
    __syncthreads();
    auto stg = [&](int c, int e, Cx<T> v) { vh[base + e * nx + c] = v.x; };
    auto ldy = [&](int c, int e) { return s[e * pitch + c]; };
    auto sty = [&](int c, int e, Cx<T> v) { s[e * pitch + c] = v; };
    auto ldx = [&](int c, int e) { return s[c * pitch + e]; };
    auto stx = [&](int c, int e, Cx<T> v) { s[c * pitch + e] = v; };
    int L = 1;
    for (int q = ax.ns - 1; q >= 0; --q) {
        L *= ax.r[q];
        stage<T, BIG, true>(ax.r[q], ldx, stx, ny, nx, L, twx);
        __syncthreads();
    }
    L = 1;
    for (int q = ay.ns - 1; q >= 0; --q) {
        L *= ay.r[q];
        if (q == 0) stage<T, BIG, true>(ay.r[q], ldy, stg, nx, ny, L, twy);
        else stage<T, BIG, true>(ay.r[q], ldy, sty, nx, ny, L, twy);
        __syncthreads();
    }
}

// Radices of n, largest first so that few stages touch LDS and the middle
// stage, whose elements stay in registers, is a small one; false when a prime
// factor above 13 remains.
bool factor(int n, Axis &a) {
    a.n = n;
    a.ns = 0;
    int twos = 0, rest = n;
    while (rest % 2 == 0) {
        rest /= 2;
        ++twos;
    }
    int odd[kMaxStages * 4], no = 0;
    for (int p : {13, 11, 7, 5, 3})
        while (rest % p == 0) {
            if (no >= kMaxStages) return false;
            odd[no++] = p;
            rest /= p;
        }
    if (rest != 1) return false;
    std::vector<int> r(odd, odd + no);
    for (; twos > 4 || twos == 3; twos -= 3) r.push_back(8);
    if (twos == 4) r.insert(r.end(), {4, 4});
    if (twos == 2) r.push_back(4);
    if (twos == 1) r.push_back(2);
    if ((int)r.size() > kMaxStages) return false;
    std::sort(r.begin(), r.end(), std::greater<int>());
    a.ns = (int)r.size();
    for (int i = 0; i < a.ns; ++i) a.r[i] = r[i];
    return true;
}

constexpr size_t kPlaneLds = 160 * 1024;  // the plane kernel may take a CU's whole LDS
constexpr size_t kLineLds = 64 * 1024;

// Workgroup of the plane kernel: 2 waves per SIMD for each workgroup that fits
// a CU's LDS beside it, so that a CU holds 16 waves at any plane size.
template <typename T>
bool plane_shape(int nx, int ny, int *pitch, size_t *lds, int *threads) {
    *pitch = nx | 1;
    *lds = sizeof(Cx<T>) * ((size_t)*pitch * ny + nx + ny);
    *threads = *lds > kPlaneLds / 2 ? 1024 : (*lds > kPlaneLds / 4 ? 512 : 256);
    return *lds <= kPlaneLds;
}

// Lines per workgroup of the line kernel: 512 bytes of consecutive points where
// their transforms fit the LDS limit, less for long axes.
template <typename T>
bool line_shape(int nz, int *C, size_t *lds) {
    for (*C = 512 / (int)sizeof(Cx<T>); *C >= 8; *C /= 2) {
        *lds = sizeof(Cx<T>) * ((size_t)nz * *C + nz);
        if (*lds <= kLineLds) return true;
    }
    return false;
}

}  // namespace

// Tables of the three axes: twiddles e^{-2 pi i t / n} and the frequency at
// each position of a forward transform's output (i > n/2 -> i - n).
struct SpectralTables {
    Axis ax[3];
    bool ok = false;   // every axis has a factorisation
    bool big = false;  // some axis has a radix above 8
    Cx<double> *d_tw64 = nullptr;
    Cx<float> *d_tw32 = nullptr;
    int *d_freq = nullptr;
};

void spectral_destroy(SpectralTables *t) {
    if (!t) return;
    for (void *p : {(void *)t->d_tw64, (void *)t->d_tw32, (void *)t->d_freq})
        if (p) (void)hipFree(p);
    delete t;
}

// The context's tables, built on first use (not inside a capture, where the
// caller keeps the library transforms): *out is null where the axes, or the
// plane's size, do not fit these kernels.
template <typename T>
int spectral_tables(qm_ctx *ctx, bool capturing, SpectralTables **out) {
    *out = nullptr;
    int pitch, threads, C;
    size_t lds;
    if (!plane_shape<T>(ctx->nx, ctx->ny, &pitch, &lds, &threads) || !line_shape<T>(ctx->nz, &C, &lds)) return QM_OK;
    if (!ctx->spectral) {
        if (capturing) return QM_OK;
        std::unique_ptr<SpectralTables, void (*)(SpectralTables *)> t(new SpectralTables(), spectral_destroy);
        const int n[3] = {ctx->nx, ctx->ny, ctx->nz};
        const double h[3] = {ctx->hx, ctx->hy, ctx->hz};
        t->ok = true;
        for (int d = 0; d < 3; ++d) t->ok = factor(n[d], t->ax[d]) && t->ok;
        if (t->ok) {
            std::vector<Cx<double>> tw;
            std::vector<Cx<float>> tw32;
            std::vector<int> freq;
            for (int d = 0; d < 3; ++d) {
                Axis &a = t->ax[d];
                t->big = t->big || a.r[0] > 8;
                a.off = (int)freq.size();
                a.g = 2.0 * M_PI / (h[d] * n[d]);
                a.k = 0.0;
                for (int i = 0; i < n[d]; ++i) {
                    const long double ph = 2.0L * 3.14159265358979323846264338327950288L * i / n[d];
                    tw.push_back({(double)cosl(ph), (double)-sinl(ph)});
                    tw32.push_back({(float)cosl(ph), (float)-sinl(ph)});
                    // position = sum_s p_s m_s with m_s = n / (r_0 .. r_s): frequency sum_s p_s (r_0 .. r_{s-1})
                    int f = 0, rem = i, m = n[d], w = 1;
                    for (int s = 0; s < a.ns; ++s) {
                        m /= a.r[s];
                        f += (rem / m) * w;
                        rem %= m;
                        w *= a.r[s];
                    }
                    freq.push_back(2 * f > n[d] ? f - n[d] : f);
                }
            }
            QM_HIP(hipMalloc((void **)&t->d_tw64, sizeof(Cx<double>) * tw.size()));
            QM_HIP(hipMalloc((void **)&t->d_tw32, sizeof(Cx<float>) * tw32.size()));
            QM_HIP(hipMalloc((void **)&t->d_freq, sizeof(int) * freq.size()));
            QM_HIP(hipMemcpy(t->d_tw64, tw.data(), sizeof(Cx<double>) * tw.size(), hipMemcpyHostToDevice));
            QM_HIP(hipMemcpy(t->d_tw32, tw32.data(), sizeof(Cx<float>) * tw32.size(), hipMemcpyHostToDevice));
            QM_HIP(hipMemcpy(t->d_freq, freq.data(), sizeof(int) * freq.size(), hipMemcpyHostToDevice));
        }
        ctx->spectral = t.release();
    }
    if (ctx->spectral->ok) *out = ctx->spectral;
    return QM_OK;
}
template int spectral_tables<double>(qm_ctx *, bool, SpectralTables **);
template int spectral_tables<float>(qm_ctx *, bool, SpectralTables **);

namespace {

template <typename T, int MODE, int NC, bool BIG>
int launch_parts(const qm_ctx *ctx, const SpectralTables *t, T *out, const T *psi, int nb, const double k[3],
                 double dt, hipStream_t st) {
    Axis a[3];
    for (int d = 0; d < 3; ++d) {
        a[d] = t->ax[d];
        a[d].k = k[d];
    }
    const Cx<T> *tw;
    const T *v;
    if constexpr (sizeof(T) == 8) {
        tw = t->d_tw64;
        v = ctx->d_vloc64;
    } else {
        tw = t->d_tw32;
        v = ctx->d_vloc32;
    }
    const int nx = ctx->nx, ny = ctx->ny, nz = ctx->nz, plane = nx * ny;
    int pitch = 0, threads = 0, C = 0;
    size_t plds = 0, llds = 0;
    QM_CHECK(plane_shape<T>(nx, ny, &pitch, &plds, &threads) && line_shape<T>(nz, &C, &llds), QM_ERR_STATE,
             "spectral kinetic: the grid does not fit the kernels");
    const int64_t planes = (int64_t)nb * (NC == 2 ? nz : (nz + 1) / 2);
    const int tile = NC == 2 ? C : 2 * C, tiles = (plane + tile - 1) / tile;
    QM_CHECK(planes < INT32_MAX && (int64_t)nb * tiles < INT32_MAX, QM_ERR_ARG,
             "spectral kinetic: too many bands per call");
    auto *pk = spectral_plane_kernel<T, MODE, NC, BIG>;
    if (plds > (size_t)64 * 1024)
        QM_HIP(hipFuncSetAttribute((const void *)pk, hipFuncAttributeMaxDynamicSharedMemorySize, (int)plds));
    hipLaunchKernelGGL(pk, dim3((unsigned)planes), dim3(threads), plds, st, out, psi, v, tw, t->d_freq, ctx->ng, nz,
                       pitch, a[0], a[1], 1.0 / ((double)nx * ny), dt);
    QM_HIP(hipGetLastError());
    hipLaunchKernelGGL((spectral_line_kernel<T, MODE, NC, BIG>), dim3((unsigned)(nb * tiles)), dim3(256), llds, st, out,
                       MODE == 0 ? psi : out, tw, t->d_freq, ctx->ng, plane, tiles, C, a[2], 1.0 / nz, dt);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

template <bool BIG>
int launch_poisson(const qm_ctx *ctx, const SpectralTables *t, Cx<double> *spec, double *vh, const double *rho,
                   hipStream_t st) {
    const int nx = ctx->nx, ny = ctx->ny, nz = ctx->nz, plane = nx * ny;
    int pitch = 0, threads = 0, C = 0;
    size_t plds = 0, llds = 0;
    QM_CHECK(plane_shape<double>(nx, ny, &pitch, &plds, &threads) && line_shape<double>(nz, &C, &llds), QM_ERR_STATE,
             "Poisson solve: the grid does not fit the kernels");
    auto *fk = poisson_forward_kernel<BIG>;
    auto *ik = poisson_inverse_kernel<BIG>;
    if (plds > (size_t)64 * 1024)
        for (const void *f : {(const void *)fk, (const void *)ik})
            QM_HIP(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)plds));
    hipLaunchKernelGGL(fk, dim3(nz), dim3(threads), plds, st, spec, rho, t->d_tw64, pitch, t->ax[0], t->ax[1]);
    QM_HIP(hipGetLastError());
    hipLaunchKernelGGL(poisson_line_kernel<BIG>, dim3((plane + C - 1) / C), dim3(256), llds, st, spec, t->d_tw64,
                       t->d_freq, plane, C, t->ax[0], t->ax[1], t->ax[2], 1.0 / (double)ctx->ng);
    QM_HIP(hipGetLastError());
    hipLaunchKernelGGL(ik, dim3(nz), dim3(threads), plds, st, vh, spec, t->d_tw64, pitch, t->ax[0], t->ax[1]);
    QM_HIP(hipGetLastError());
    return QM_OK;
}

}  // namespace

template <typename T>
int spectral_kinetic(const qm_ctx *ctx, const SpectralTables *t, T *out, const T *psi, int nb, int ncomp,
                     const double k[3], hipStream_t st) {
    if (t->big)
        return ncomp == 2 ? launch_parts<T, 0, 2, true>(ctx, t, out, psi, nb, k, 0.0, st)
                          : launch_parts<T, 0, 1, true>(ctx, t, out, psi, nb, k, 0.0, st);
    return ncomp == 2 ? launch_parts<T, 0, 2, false>(ctx, t, out, psi, nb, k, 0.0, st)
                      : launch_parts<T, 0, 1, false>(ctx, t, out, psi, nb, k, 0.0, st);
}
template int spectral_kinetic<double>(const qm_ctx *, const SpectralTables *, double *, const double *, int, int,
                                      const double *, hipStream_t);
template int spectral_kinetic<float>(const qm_ctx *, const SpectralTables *, float *, const float *, int, int,
                                     const double *, hipStream_t);

template <typename T>
int spectral_step(const qm_ctx *ctx, const SpectralTables *t, T *psi, int nb, const double k[3], double dt,
                  hipStream_t st) {
    return t->big ? launch_parts<T, 1, 2, true>(ctx, t, psi, psi, nb, k, dt, st)
                  : launch_parts<T, 1, 2, false>(ctx, t, psi, psi, nb, k, dt, st);
}
template int spectral_step<double>(const qm_ctx *, const SpectralTables *, double *, int, const double *, double,
                                   hipStream_t);
template int spectral_step<float>(const qm_ctx *, const SpectralTables *, float *, int, const double *, double,
                                  hipStream_t);

int spectral_poisson(const qm_ctx *ctx, const SpectralTables *t, void *spec, double *vh, const double *rho,
                     hipStream_t st) {
    Cx<double> *z = static_cast<Cx<double> *>(spec);
    return t->big ? launch_poisson<true>(ctx, t, z, vh, rho, st) : launch_poisson<false>(ctx, t, z, vh, rho, st);
}

}  // namespace qm
