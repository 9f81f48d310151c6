// CPU check of the secular equation's root finder (csrc/secular.h), built with
// AddressSanitizer and UndefinedBehaviorSanitizer by tests/test_secular_bound.py.
// Random poles and weights (clustered, graded, paired, tiny), inside the range
// that deflation leaves: every root is found within the step bound, also when the
// rational steps are taken away (they then move by 1e-9 of a Newton step, so that
// only the bracket ends the iteration), and both ways agree.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "secular.h"

using namespace qm;

struct Stuck {
    double operator()(bool, double, double, double f, double, double, double df) const { return -1e-9 * f / df; }
};

int main() {
    std::mt19937_64 gen(20260923u);
    std::uniform_real_distribution<double> u(0.0, 1.0);
    int fails = 0, worst = 0, worst_stuck = 0;
    long roots = 0;
    for (int trial = 0; trial < 4000; ++trial) {
        const int k = 1 + (int)(u(gen) * u(gen) * 60);
        std::vector<double> d(k), z2(k);
        const double spread = std::pow(10.0, -16.0 * u(gen));
        double x = u(gen) - 0.5, top = 0.0, total = 0.0;
        for (int i = 0; i < k; ++i) {
            double gap = 0.0;
            switch (trial % 6) {
                case 0: gap = u(gen); break;
                case 1: gap = std::pow(10.0, -15.0 * u(gen)); break;
                case 2: gap = i % 5 == 0 ? u(gen) : spread * u(gen); break;
                case 3: gap = std::pow(2.0, -(double)i * u(gen)); break;
                case 4: gap = i % 2 ? u(gen) : 1e-15; break;
                default: gap = 1.0 / k;
            }
            x += gap + 4e-16 * std::fabs(x);
            d[i] = x;
            top = std::fmax(top, std::fabs(x));
            const double e = u(gen);
            switch (trial / 6 % 5) {
                case 0: z2[i] = e; break;
                case 1: z2[i] = std::pow(10.0, -30.0 * e); break;
                case 2: z2[i] = i == k / 2 ? 1.0 : 1e-15 * (1.0 + e); break;
                case 3: z2[i] = i % 2 ? 1.0 : 1e-14 * e + 1e-16; break;
                default: z2[i] = std::pow(10.0, -30.0 * i / k);
            }
            total += z2[i];
        }
        bool ascending = true;
        for (int i = 0; i < k; ++i) {
            d[i] /= top;
            z2[i] /= total;
            ascending = ascending && (i == 0 || d[i] > d[i - 1]);
        }
        if (!ascending) continue;
        const double rho = 2.0 * std::pow(10.0, -14.0 * u(gen) * (u(gen) < 0.5));
        for (int j = 0; j < k; ++j) {
            int o1 = -1, o2 = -1;
            double t1 = 0.0, t2 = 0.0;
            long sums = 0;
            auto sum = [&](double v) {
                ++sums;
                return v;
            };
            const bool ok1 = secular_root(j, k, d.data(), z2.data(), rho, 0, 1, sum, kMaxSteps, &o1, &t1);
            worst = std::max(worst, (int)(sums / 4));
            sums = 0;
            const bool ok2 = secular_root(j, k, d.data(), z2.data(), rho, 0, 1, sum, kMaxSteps, &o2, &t2, Stuck());
            worst_stuck = std::max(worst_stuck, (int)(sums / 4));
            ++roots;
            // inside its interval, on the near side of the middle
            bool in = std::isfinite(t1) && t1 != 0.0 && (o1 == j ? t1 > 0.0 : o1 == j + 1 && t1 < 0.0);
            if (j + 1 < k) in = in && std::fabs(t1) <= 0.5 * (d[j + 1] - d[j]);
            // both stop where f is within its rounding, or one unit apart: the
            // offsets differ by the sum of both residuals over f', small against the
            // nearest pole's distance wherever f is not flat
            double df = 0.0, mag = 1.0 / rho;
            for (int i = 0; i < k; ++i) {
                const double g = 1.0 / ((d[i] - d[o1]) - t1);
                df += z2[i] * g * g;
                mag += 8.0 * z2[i] * std::fabs(g);
            }
            const double tol = 8.0 * kEps * (mag / df + std::fabs(t1));
            const bool same = o1 == o2 && std::fabs(t1 - t2) <= tol;
            if (!(ok1 && ok2 && in && same) && fails++ < 10)
                std::fprintf(stderr, "trial %d root %d of %d: ok %d %d in %d offsets %g %g (tol %g)\n", trial, j, k, ok1,
                             ok2, in, t1, t2, tol);
        }
    }
    if (fails) {
        std::fprintf(stderr, "%d roots failed\n", fails);
        return 1;
    }
    std::printf("secular: %ld roots ok, at most %d steps, %d by the bracket alone, bound %d\n", roots, worst, worst_stuck,
                kMaxSteps);
    return 0;
}
