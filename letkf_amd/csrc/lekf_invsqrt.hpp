// lekf_invsqrt.hpp -- nodes of a rational form of x^(-1/2) on [1, kappa].
//
// x^(-1/2) = (2/pi) Int_0^inf dt / (t^2 + x).  With t = sc(u | k'), k^2 = 1/kappa
// and k' = sqrt(1 - k^2), the integrand is periodic in u and the N-point midpoint
// rule over (0, K') converges geometrically, error ~ exp(-2 pi^2 N / (ln kappa + 2.8))
// (Hale, Higham and Trefethen, SIAM J. Numer. Anal. 46, 2008):
//   x^(-1/2) ~ sum_j om_j / (x + sg_j),  sg_j = sc(u_j)^2,
//   om_j = (2/pi) (K'/N) sc'(u_j),       u_j = (j - 1/2) K' / N.
// Every term is positive, so the sum loses nothing to cancellation.  sc is taken
// from its theta functions at an imaginary argument, whose nome is tiny here.
// The tables hold N = 8, 12, .., 40 nodes for kappa = 4 * 8^i, up to 2^26, where an
// eigenvalue is small enough to be truncated: the largest relative error over [1, kappa]
// is below 4e-16 in each.  Evaluated at compile time.
#pragma once

namespace lekf_invsqrt {

constexpr int kLevels = 9;
constexpr int kMaxNodes = 8 + 4 * (kLevels - 1);

struct Table {
    double sg[kLevels][kMaxNodes];
    double om[kLevels][kMaxNodes];
};

constexpr double c_sqrt(double x)
{
    double r = x > 1.0 ? x : 1.0;
    for (int i = 0; i < 60; ++i) {
        const double n = 0.5 * (r + x / r);
        if (n == r) break;
        r = n;
    }
    return r;
}

constexpr double c_exp(double x)
{
    // x = n ln 2 + f, |f| <= ln 2 / 2; ln 2 in two parts, the first of 16 bits so that
    // n times it is exact
    const double hi = 45426.0 / 65536.0, lo = 1.4286068203094172321e-6;
    int n = (int)(x / (hi + lo) + (x >= 0 ? 0.5 : -0.5));
    const double f = (x - n * hi) - n * lo;
    double s = 1.0, t = 1.0;
    for (int i = 1; i < 24; ++i) {
        t *= f / i;
        s += t;
    }
    for (; n <= -32; n += 32) s *= 1.0 / 4294967296.0;
    for (; n < 0; ++n) s *= 0.5;
    for (; n > 0; --n) s *= 2.0;
    return s;
}

constexpr double c_agm(double a, double b)
{
    for (int i = 0; i < 40 && !(a - b <= 1e-16 * a && b - a <= 1e-16 * a); ++i) {
        const double m = 0.5 * (a + b);
        b = c_sqrt(a * b);
        a = m;
    }
    return 0.5 * (a + b);
}

constexpr Table make_table()
{
    Table T{};
    const double pi = 3.14159265358979323846;
    double kappa = 4.0;
    for (int l = 0; l < kLevels; ++l, kappa *= 8.0) {
        const int N = 8 + 4 * l;
        const double K = 0.5 * pi / c_agm(1.0, c_sqrt(1.0 - 1.0 / kappa));
        const double Kp = 0.5 * pi / c_agm(1.0, c_sqrt(1.0 / kappa));
        const double lnq = -pi * Kp / K;  // the nome's logarithm
        double th2 = 0.0, th3 = 1.0;
        for (int n = 0; n < 6; ++n) th2 += 2.0 * c_exp(lnq * (n + 0.5) * (n + 0.5));
        for (int n = 1; n < 6; ++n) th3 += 2.0 * c_exp(lnq * n * n);
        for (int j = 0; j < N; ++j) {
            const double y = (j + 0.5) / N * (-0.5 * lnq);
            double S = 0.0, dS = 0.0, C = 1.0, dC = 0.0;
            for (int n = 0; n < 6; ++n) {
                const double sg = (n & 1) ? -1.0 : 1.0;
                const double g = lnq * (n + 0.5) * (n + 0.5);
                const double p = c_exp(g + (2 * n + 1) * y), m = c_exp(g - (2 * n + 1) * y);
                S += sg * (p - m);
                dS += sg * (2 * n + 1) * (p + m);
                if (n > 0) {
                    const double h = lnq * n * n;
                    const double p2 = c_exp(h + 2 * n * y), m2 = c_exp(h - 2 * n * y);
                    C += sg * (p2 + m2);
                    dC += sg * 2 * n * (p2 - m2);
                }
            }
            const double sc = th3 / th2 * S / C;
            const double dsc = pi / (2.0 * K) * th3 / th2 * (dS * C - S * dC) / (C * C);
            T.sg[l][j] = sc * sc;
            T.om[l][j] = 2.0 / pi * Kp / N * dsc;
        }
    }
    return T;
}

}  // namespace lekf_invsqrt
