// Adjoint of H.psi with respect to the local potential: the band density.
//
//   rho(r) += sum_n occ_n |psi_n(r)|^2      (dE_band/dV_loc(r) = rho(r) dV)
//
// Mathematics: SetDensityOne (qumasun_SetDensityOne.h:9-41), which sums the
// SoA re and im rows of every band with the band's occupancy.  One thread per
// grid point walks all bands (coalesced along x) and accumulates in FP64.
#include <algorithm>

#include "qm_internal.h"

namespace qm {
namespace {

// Occupations of one launch, by value (no staging buffer, no upload): bands
// beyond kDensityBands take further launches.
constexpr int kDensityBands = 256;
struct DensityOcc {
    double occ[kDensityBands];
};

// One read of psi and one update of rho: bound by HBM (64^3 x 64 FP64: 134 MB
// in 27 us).  Four bands' values are requested together.
template <typename T, int NC>
__global__ __launch_bounds__(256) void band_density_kernel(double *__restrict__ rho, const T *__restrict__ psi,
                                                            DensityOcc occ, int64_t ng, int nb) {
    constexpr int U = 4;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= ng) return;
    const T *p = psi + i;
    double s = 0.0;
    int n = 0;
    for (; n + U <= nb; n += U) {
        T v[U][NC];
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int c = 0; c < NC; ++c) v[u][c] = p[((int64_t)(n + u) * NC + c) * ng];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            double t = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c) t += (double)v[u][c] * (double)v[u][c];
            s += occ.occ[n + u] * t;
        }
    }
    for (; n < nb; ++n) {
        double t = 0.0;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const double v = (double)p[((int64_t)n * NC + c) * ng];
            t += v * v;
        }
        s += occ.occ[n] * t;
    }
    rho[i] += s;
}

template <typename T>
int launch_density(const qm_ctx *ctx, double *rho, const T *psi, const double *occ, int nb, int ncomp,
                   hipStream_t st) {
    QM_CHECK(ncomp == 1 || ncomp == 2, QM_ERR_ARG, "ncomp must be 1 or 2");
    const int64_t blocks = (ctx->ng + 255) / 256;
    for (int n0 = 0; n0 < nb; n0 += kDensityBands) {
        const int n = std::min(kDensityBands, nb - n0);
        DensityOcc o;
        for (int i = 0; i < kDensityBands; ++i) o.occ[i] = i < n ? occ[n0 + i] : 0.0;
        const T *src = psi + (int64_t)n0 * ncomp * ctx->ng;
        if (ncomp == 1)
            hipLaunchKernelGGL((band_density_kernel<T, 1>), dim3((unsigned)blocks), dim3(256), 0, st, rho, src, o,
                               ctx->ng, n);
        else
            hipLaunchKernelGGL((band_density_kernel<T, 2>), dim3((unsigned)blocks), dim3(256), 0, st, rho, src, o,
                               ctx->ng, n);
        QM_HIP(hipGetLastError());
    }
    return QM_OK;
}

}  // namespace

int launch_band_density_f64(const qm_ctx *ctx, double *rho, const double *psi, const double *occ, int nb,
                            int ncomp, hipStream_t st) {
    return launch_density<double>(ctx, rho, psi, occ, nb, ncomp, st);
}
int launch_band_density_f32(const qm_ctx *ctx, double *rho, const float *psi, const double *occ, int nb,
                            int ncomp, hipStream_t st) {
    return launch_density<float>(ctx, rho, psi, occ, nb, ncomp, st);
}

}  // namespace qm
