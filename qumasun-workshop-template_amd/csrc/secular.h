// One root of the secular equation f(x) = 1/rho + sum_i z_i^2 / (d_i - x), rho > 0,
// d ascending: root j lies between d_j and d_{j+1}, the last one above d_{k-1}.
//
// It is held as an offset from its nearest pole, so that differences to the poles
// keep their relative accuracy.  R.-C. Li's "middle way" steps (LAPACK Working Note
// 89) inside a bracket whose ends have one sign: the far end is the middle of the
// interval, the near end a lower bound of the offset's size, from f's terms of the
// other sign where they are largest.  From step kFreeSteps on every fourth step
// halves the bracket (its logarithm while the ends are more than a factor of 4
// apart), so that the iteration ends whatever the other steps do: with z_i^2 of
// undeflated poles above 2^-114 and their gaps above 2^-54 the ends of a bracket
// are less than 2^256 apart, and 8 + 54 halvings bring them within two units of
// each other.  kMaxSteps covers them.  (Few roots get there: of 3.3 million random
// ones, clustered and graded, 12,000, and 56 steps at most; every second step
// instead of every fourth takes them 47 steps instead of 29 on average.)
#pragma once

#include <cmath>

#ifdef __HIPCC__
#define QM_HD __host__ __device__ __forceinline__
#else
#define QM_HD inline
#endif

namespace qm {

constexpr double kEps = 0x1p-53;  // unit roundoff
constexpr int kFreeSteps = 16;
constexpr int kMaxSteps = kFreeSteps + 4 * 64;

// The rational step from tau: the zero of the interpolating function with the poles
// at a1 and a2 from tau (last root: the one pole at a1); f, its derivative's parts
// from the poles up to j and above, and their sum.
struct RationalStep {
    QM_HD double operator()(bool last, double a1, double a2, double f, double dpsi, double dphi, double df) const {
        if (last) {
            const double c = f - a1 * dpsi;
            return a1 + a1 * a1 * dpsi / c;
        }
        const double c = f - a1 * dpsi - a2 * dphi, a = (a1 + a2) * f - a1 * a2 * df, b = a1 * a2 * f;
        const double s = sqrt(fabs(a * a - 4.0 * b * c));
        if (c == 0.0) return b / a;
        return a <= 0.0 ? (a - s) / (2.0 * c) : 2.0 * b / (a + s);
    }
};

// Root j of k: its origin (a pole) and offset.  The terms are summed by `lanes`
// callers together, this one taking every lanes-th from `lane` on; sum(v) is the
// total over them, the same in each.  False where max_steps did not do.
template <typename Sum, typename Step = RationalStep>
QM_HD bool secular_root(int j, int k, const double *d, const double *z2, double rho, int lane, int lanes, Sum &&sum,
                        int max_steps, int *origin, double *offset, Step step = Step()) {
    const double rinv = 1.0 / rho;
    const bool last = j == k - 1;
    double lo, hi, tau;
    int org = j;
    if (!last) {
        const double del = d[j + 1] - d[j], h = 0.5 * del;
        double c0 = 0.0, below = 0.0;  // below: the terms of the poles under d_j at d_j + h
        for (int i = lane; i < k; i += lanes) {
            if (i == j || i == j + 1) continue;
            const double t = z2[i] / ((d[i] - d[j]) - h);
            c0 += t;
            if (i < j) below += t;
        }
        below = sum(below);
        c0 = sum(c0);
        const double above = c0 - below;
        c0 = rinv + c0;
        const double f = c0 + (z2[j + 1] - z2[j]) / h;
        if (f > 0.0) {
            // z_j^2 / tau = the other terms, at most the positive ones at h
            lo = 0.25 * z2[j] / (rinv + fabs(above) + z2[j + 1] / h);
            hi = h;
            const double a = c0 * del + z2[j] + z2[j + 1], b = z2[j] * del, s = sqrt(fabs(a * a - 4.0 * b * c0));
            tau = a > 0.0 ? 2.0 * b / (a + s) : (a - s) / (2.0 * c0);
        } else {
            org = j + 1;
            lo = -h;
            hi = -0.25 * z2[j + 1] / (fabs(below) + z2[j] / h);
            const double a = c0 * del - z2[j] - z2[j + 1], b = z2[j + 1] * del, s = sqrt(fabs(a * a + 4.0 * b * c0));
            tau = a < 0.0 ? 2.0 * b / (a - s) : -(a + s) / (2.0 * c0);
        }
    } else {
        double s = 0.0;
        for (int i = lane; i < k; i += lanes) s += z2[i];
        hi = rho * sum(s) * (1.0 + 8.0 * kEps);
        lo = 0.25 * z2[j] * rho;  // every other term is negative
        double c0 = 0.0;
        for (int i = lane; i < k - 1; i += lanes) c0 += z2[i] / ((d[i] - d[j]) - hi);
        c0 = rinv + sum(c0);
        tau = c0 > 0.0 ? z2[j] / c0 : hi;
    }
    if (!(tau > lo && tau < hi)) tau = 0.5 * (lo + hi);
    const double d0 = d[org];
    const double dj = d[j] - d0, dj1 = last ? 0.0 : d[j + 1] - d0;
    bool ok = false;
    for (int it = 0; it < max_steps; ++it) {
        double psi = 0.0, dpsi = 0.0, phi = 0.0, dphi = 0.0;
        for (int i = lane; i < k; i += lanes) {
            const double g = 1.0 / ((d[i] - d0) - tau), t = z2[i] * g;
            if (i <= j) {
                psi += t;
                dpsi += t * g;
            } else {
                phi += t;
                dphi += t * g;
            }
        }
        psi = sum(psi);
        dpsi = sum(dpsi);
        phi = sum(phi);
        dphi = sum(dphi);
        const double f = rinv + psi + phi, df = dpsi + dphi;
        if (fabs(f) <= kEps * (8.0 * (phi - psi) + rinv + fabs(tau) * df)) {
            ok = true;
            break;
        }
        if (f > 0.0) hi = fmin(hi, tau);
        else lo = fmax(lo, tau);
        double eta = step(last, dj - tau, dj1 - tau, f, dpsi, dphi, df);
        if (!(f * eta < 0.0)) eta = -f / df;
        double x = tau + eta;
        if (!(x > lo && x < hi) || (it >= kFreeSteps && it % 4 == 3)) {
            const double a = fmin(fabs(lo), fabs(hi)), b = fmax(fabs(lo), fabs(hi));
            x = copysign(b > 4.0 * a ? sqrt(a) * sqrt(b) : 0.5 * (a + b), lo + hi);
        }
        if (x == tau || hi - lo <= 2.0 * kEps * fmax(fabs(lo), fabs(hi))) {
            ok = true;
            break;
        }
        tau = x;
    }
    *origin = org;
    *offset = tau;
    return ok;
}

}  // namespace qm
