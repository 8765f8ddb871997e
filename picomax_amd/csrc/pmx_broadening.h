/*
 * pmx_broadening.h -- the broadening's expansion over a frequency bin: its
 * order, its economised coefficients and the kernel tables of the convolution
 * (plain C++, on the host).
 */
#ifndef PMX_BROADENING_H
#define PMX_BROADENING_H

#include "pmx_internal.h"

#include <algorithm>
#include <cmath>
#include <complex>

namespace pmx {

constexpr int MAX_NT = 20; /* 4 waves x 5 orders in the MFMA kernel */

/* Taylor order for a truncation below tol relative to the peak: with
 * r = (df/2)/epsilon the Lorentzian terms fall like r^n (its poles sit at
 * distance >= epsilon from every expansion point), the Gaussian ones like
 * r^n / sqrt(n!) (Hermite-function bound). */
inline int taylor_order(int delta, double eps, double df, double tol) {
    const double r = 0.5 * df / eps;
    if (r >= 0.6) return -1;
    double term = 1.0;
    for (int n = 1; n <= MAX_NT; n++) {
        term *= (delta == 0) ? r / std::sqrt((double)n) : r;
        if (term < tol) return n;
    }
    return -1;
}

/* one row of Taylor coefficients h^n delta^(n)(x)/n!, n < NT */
inline void taylor_row(int delta, double eps, double h, double x, int NT, double *row) {
    if (delta == 1) {
        /* (1/pi) Im[(-1)^n / (x - i eps)^(n+1)] h^n */
        std::complex<double> z(x, -eps), inv = 1.0 / z, pw = inv;
        double hn = 1.0, sg = 1.0;
        for (int n = 0; n < NT; n++) {
            row[n] = sg * hn * pw.imag() / PMX_PI;
            pw *= inv;
            hn *= h;
            sg = -sg;
        }
    } else {
        /* a_{n+1} = -(x a_n + a_{n-1}) / (eps^2 (n+1)), a_0 = g(x) */
        double am1 = 0.0, a0 = std::exp(-0.5 * x * x / (eps * eps)) / (eps * std::sqrt(2.0 * PMX_PI));
        double hn = 1.0;
        for (int n = 0; n < NT; n++) {
            row[n] = hn * a0;
            double a1 = -(x * a0 + am1) / (eps * eps * (n + 1));
            am1 = a0;
            a0 = a1;
            hn *= h;
        }
    }
}

/* the expansion of delta over a bin, economised.  The Taylor series
 * about the bin centre needs NT orders because it spends its accuracy at
 * s = 0; rewritten in Chebyshev polynomials T_n(s) on |s| <= 1 its
 * coefficients fall like (1/r + sqrt(1/r^2 + 1))^-n instead of r^n
 * (Lorentzian, r = (df/2)/epsilon), so M < NT of them leave no larger an rms
 * error.  The kept part is written back in powers of s, so moments and
 * convolution run as before with M orders in place of NT (Lorentzian r = 0.2:
 * 12 for 16 in FP64, 8 for 9 on the mixed paths; the rank update, the
 * convolution and the moments' memory are all linear in it). */
struct Economised {
    int M, NX;             /* orders kept; Taylor orders the coefficients are taken from */
    std::vector<double> E; /* [M][NX]: Taylor coefficients -> kept powers */
};

/* NT: the order count of the plain series, whose rms error over a bin, where it
 * is largest, is the one kept to */
inline Economised economise(int delta, double eps, double df, int NT) {
    const double r = 0.5 * df / eps, h = 0.5 * df;
    Economised ec;
    int NX = NT + 4;
    for (double t = std::pow(r, NX); t > 1e-16 && NX < 64; t *= r) NX++;
    /* A[k][n]: the T_k coefficient of s^n; B[n][k]: the s^n coefficient of T_k */
    std::vector<long double> A((size_t)NX * NX, 0.0L), B((size_t)NX * NX, 0.0L);
    A[0] = 1.0L;
    for (int n = 1; n < NX; n++) /* s T_k = (T_{k+1} + T_{|k-1|}) / 2 */
        for (int k = 0; k < n; k++) {
            const long double v = A[(size_t)k * NX + n - 1];
            if (k == 0) A[(size_t)1 * NX + n] += v;
            else {
                A[(size_t)(k + 1) * NX + n] += 0.5L * v;
                A[(size_t)(k - 1) * NX + n] += 0.5L * v;
            }
        }
    B[0] = 1.0L;
    if (NX > 1) B[(size_t)1 * NX + 1] = 1.0L;
    for (int k = 2; k < NX; k++)
        for (int n = 0; n < NX; n++)
            B[(size_t)n * NX + k] = (n > 0 ? 2.0L * B[(size_t)(n - 1) * NX + k - 1] : 0.0L) - B[(size_t)n * NX + k - 2];
    /* the offsets near the peak, where both series are at their worst */
    const int Dm = (int)(4.0 * eps / df) + 1;
    const int step = std::max(1, Dm / 32);
    /* squares are averaged over the bin at s = cos(angle), angles equally spaced, weights sin(angle) */
    constexpr int S = 20;
    double s[S], wt[S];
    std::vector<double> T((size_t)NX * S, 1.0); /* T_k(s) */
    for (int i = 0; i < S; i++) {
        const double angle = PMX_PI * (i + 0.5) / S;
        s[i] = std::cos(angle);
        wt[i] = std::sin(angle);
        for (int k = 1; k < NX; k++)
            T[(size_t)k * S + i] = k == 1 ? s[i] : 2.0 * s[i] * T[(size_t)(k - 1) * S + i] - T[(size_t)(k - 2) * S + i];
    }
    std::vector<double> row(NX), tail(NT, 0.0);
    double worst = 0.0;
    for (int D = -1; D <= Dm; D += (D < 8 ? 1 : step)) { /* delta is even: D and -1 - D mirror each other */
        taylor_row(delta, eps, h, (D + 0.5) * df, NX, row.data());
        double p[S] = {}, t = 0.0;
        for (int n = NX - 1; n > 0; n--) { /* the terms from n on */
            long double a = 0.0L;
            for (int m = n; m < NX; m += 2) a += A[(size_t)n * NX + m] * row[m];
            double t2 = 0.0;
            for (int i = 0; i < S; i++) {
                p[i] += (double)a * T[(size_t)n * S + i];
                t2 += wt[i] * p[i] * p[i];
            }
            if (n < NT) tail[n] = std::max(tail[n], t2);
        }
        for (int i = 0; i < S; i++) { /* the Taylor terms from NT on */
            double q = 0.0;
            for (int m = NX - 1; m >= NT; m--) q = q * s[i] + row[m];
            q *= std::pow(s[i], NT);
            t += wt[i] * q * q;
        }
        worst = std::max(worst, t);
    }
    ec.NX = NX;
    ec.M = NT;
    for (int m = 1; m < NT; m++)
        if (tail[m] <= 1.04 * worst) { /* the same to 2%; the largest error is then a quarter of the plain series' */
            ec.M = m;
            break;
        }
    ec.E.assign((size_t)ec.M * NX, 0.0);
    for (int n = 0; n < ec.M; n++)
        for (int m = 0; m < NX; m++) {
            long double v = 0.0L;
            for (int k = n; k < ec.M && k <= m; k++) v += B[(size_t)n * NX + k] * A[(size_t)k * NX + m];
            ec.E[(size_t)n * NX + m] = (double)v;
        }
    return ec;
}

/* kernel table K_n(D), n < ec.M, for the W offsets D = f0 - f =
 * Dlo .. Dlo + W - 1 (row D - Dlo) */
inline void kernel_table(int delta, double eps, double df, int Dlo, int W, const Economised &ec, std::vector<double> &Kt) {
    Kt.assign((size_t)W * ec.M, 0.0);
    std::vector<double> row(ec.NX);
    for (int Dd = Dlo; Dd < Dlo + W; Dd++) {
        taylor_row(delta, eps, 0.5 * df, (Dd + 0.5) * df, ec.NX, row.data()); /* x = c_b - w_f */
        for (int n = 0; n < ec.M; n++) {
            double v = 0.0;
            for (int m = ec.NX - 1; m >= n; m--) v += ec.E[(size_t)n * ec.NX + m] * row[m];
            Kt[(size_t)(Dd - Dlo) * ec.M + n] = v;
        }
    }
}

} // namespace pmx

#endif
