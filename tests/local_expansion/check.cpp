// The far cells' local expansion (csrc/pgrav_local.h) against the cells' own fields in
// FP64: for each order, softening and nearest distance, the largest error of the pull at
// any sink over the root mean square pull, one line each.
#include <array>
#include <cmath>
#include <cstdio>
#include <random>
#include <vector>

#include "pgrav_local.h"

using namespace pgrav;

namespace {

// psi = sum_k P_k(x) (|x|^2 + eps^2)^-(k+1/2) of a prepared record at x: grad psi, -psi
void field(const double *M, int order, const double *X, double eps2, double *out) {
    const double x = X[0], y = X[1], z = X[2], x2 = x * x, y2 = y * y, z2 = z * z;
    const double b2[3][3] = {{M[4], M[5], M[6]}, {M[5], M[7], M[8]}, {M[6], M[8], M[9]}};
    const double b3[5] = {x2 - z2, y2 - z2, x * y, x * z, y * z};
    const double b4[7] = {x * (x2 - 3 * z2), y * (y2 - 3 * z2), y * (x2 - z2), z * (3 * x2 - z2),
                          x * (y2 - z2), x * y * z, z * (3 * y2 - z2)};
    double G[5][3] = {}, P[5] = {M[3], 0, 0, 0, 0};
    for (int r = 0; r < 3; r++) {
        for (int c = 0; c < 3; c++) G[2][r] += b2[r][c] * X[c];
        for (int k = 0; k < 5; k++) G[3][r] += M[10 + 5 * r + k] * b3[k];
        for (int k = 0; k < 7; k++) G[4][r] += M[25 + 7 * r + k] * b4[k];
        for (int k = 2; k <= 4; k++) P[k] += G[k][r] * X[r];
    }
    const double ri2 = 1 / (x2 + y2 + z2 + eps2);
    double f = sqrt(ri2);
    for (int k = 0; k <= order; k++, f *= ri2) {
        out[3] -= f * P[k];
        for (int r = 0; r < 3; r++) out[r] += f * (k * G[k][r] - (2 * k + 1) * ri2 * P[k] * X[r]);
    }
}

// the prepared record of points about their mean, of masses m (sum 1), through traceless moments
void record(const std::vector<std::array<double, 3>> &points, const std::vector<double> &m, double size,
            int order, double *M) {
    std::vector<std::array<double, 3>> p = points;
    const int n = (int)p.size();
    double mean[3] = {0, 0, 0};
    for (int i = 0; i < n; i++)
        for (int k = 0; k < 3; k++) mean[k] += m[i] * p[i][k];
    double q[29] = {0};
    q[0] = 1;
    q[4] = size;
    auto dl = [](int i, int j) { return i == j ? 1.0 : 0.0; };
    for (int i0 = 0; i0 < n; i0++) {
        double x[3], r2 = 0;
        for (int k = 0; k < 3; k++) {
            x[k] = (p[i0][k] - mean[k]) / size;
            r2 += x[k] * x[k];
        }
        const int i2[5][2] = {{0, 0}, {0, 1}, {1, 1}, {0, 2}, {1, 2}};
        const int i3[7][3] = {{0, 0, 0}, {0, 0, 1}, {0, 1, 1}, {1, 1, 1}, {0, 0, 2}, {0, 1, 2}, {1, 1, 2}};
        const int i4[9][4] = {{0, 0, 0, 0}, {0, 0, 0, 1}, {0, 0, 1, 1}, {0, 1, 1, 1}, {1, 1, 1, 1},
                              {0, 0, 0, 2}, {0, 0, 1, 2}, {0, 1, 1, 2}, {1, 1, 1, 2}};
        for (int t = 0; t < 5; t++) {
            const int i = i2[t][0], j = i2[t][1];
            q[8 + t] += m[i0] * (x[i] * x[j] - r2 / 3 * dl(i, j));
        }
        for (int t = 0; t < 7; t++) {
            const int i = i3[t][0], j = i3[t][1], l = i3[t][2];
            q[13 + t] += m[i0] * (x[i] * x[j] * x[l] -
                                  r2 / 5 * (dl(i, j) * x[l] + dl(i, l) * x[j] + dl(j, l) * x[i]));
        }
        for (int t = 0; t < 9; t++) {
            const int i = i4[t][0], j = i4[t][1], l = i4[t][2], k = i4[t][3];
            q[20 + t] += m[i0] *
                         (x[i] * x[j] * x[l] * x[k] -
                          r2 / 7 * (dl(i, j) * x[l] * x[k] + dl(i, l) * x[j] * x[k] + dl(i, k) * x[j] * x[l] +
                                    dl(j, l) * x[i] * x[k] + dl(j, k) * x[i] * x[l] + dl(l, k) * x[i] * x[j]) +
                          r2 * r2 / 35 * (dl(i, j) * dl(l, k) + dl(i, l) * dl(j, k) + dl(i, k) * dl(j, l)));
        }
    }
    prep_record<double>(q, order, 0, M);
}

// a cell of 20 points of one mass, anywhere in a box
void cell(std::mt19937_64 &g, double size, int order, double *M) {
    std::uniform_real_distribution<double> U(-0.5, 0.5);
    std::vector<std::array<double, 3>> p(20);
    for (auto &q : p)
        for (int k = 0; k < 3; k++) q[k] = size * U(g);
    record(p, std::vector<double>(20, 0.05), size, order, M);
}

// One cell of two points at distance at most b from their mean, anywhere around the group
// and turned any way: the largest error in units of the cell's pull as a point, m / d^2.
template <int ORDER>
void run_two(double rho, double bd) {
    std::mt19937_64 g(2);
    std::normal_distribution<double> N;
    double worst = 0;
    for (int c = 0; c < 400; c++) {
        auto unit = [&](double *n) {
            double r = 0;
            for (int k = 0; k < 3; k++) {
                n[k] = N(g);
                r += n[k] * n[k];
            }
            for (int k = 0; k < 3; k++) n[k] /= sqrt(r);
        };
        double n[3], t[3];
        unit(n);
        unit(t);
        if (c < 100)  // along the line of sight
            for (int k = 0; k < 3; k++) t[k] = c % 2 ? n[k] : -n[k];
        const double f = 0.5 + 0.1 * (c % 5);  // the share of the point nearer to the mean
        double M[PREC4];
        record({{t[0] * bd, t[1] * bd, t[2] * bd},
                {-t[0] * bd * (1 - f) / f, -t[1] * bd * (1 - f) / f, -t[2] * bd * (1 - f) / f}},
               {1 - f, f}, bd, ORDER, M);
        std::vector<double> A(LX_ALL, 0.0);
        lx_add_cell<ORDER, false, double>(M, 1.0, n[0], n[1], n[2], 0.0, rho, A.data());
        for (int i = 0; i < 64; i++) {
            double u[3], o[4], r[4] = {0, 0, 0, 0}, e = 0;
            unit(u);
            if (i < 2)  // towards the cell and away from it
                for (int k = 0; k < 3; k++) u[k] = i ? n[k] : -n[k];
            lx_evaluate<false, 0, double>(A.data(), u[0], u[1], u[2], 1 / rho, o);
            const double X[3] = {rho * u[0] - n[0], rho * u[1] - n[1], rho * u[2] - n[2]};
            field(M, ORDER, X, 0.0, r);
            for (int k = 0; k < 3; k++) e += (o[k] - r[k]) * (o[k] - r[k]);
            worst = std::max(worst, sqrt(e));
        }
    }
    printf("two %d %g %g %.3e\n", ORDER, rho, bd, worst);
}

template <int ORDER, bool SOFT, typename T>
void run(double rho, double eta) {
    std::mt19937_64 g(1);
    std::normal_distribution<double> N;
    std::uniform_real_distribution<double> U(0, 1);
    const double rs = 0.37, dmin = rs / rho, eps2 = SOFT ? eta * dmin * dmin : 0.0;
    std::vector<std::array<double, 3>> s(64);
    std::vector<std::array<double, 4>> ref(64, {0, 0, 0, 0});
    for (int i = 0; i < 64; i++) {
        const double v[3] = {N(g), N(g), N(g)};
        const double f = (i < 8 ? rs : rs * cbrt(U(g))) / sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        s[i] = {v[0] * f, v[1] * f, v[2] * f};
    }
    std::vector<T> A(LX_ALL, T(0));
    for (int c = 0; c < 6; c++) {
        // on the z axis either way, beside it, and anywhere
        double n[3] = {N(g), N(g), N(g)};
        if (c < 2)
            n[0] = n[1] = 0, n[2] = c ? 1 : -1;
        if (c == 2)
            n[0] = 1e-9, n[1] = -1e-10, n[2] = 1;
        const double d = dmin * (c < 3 ? 1 : 1 + U(g)), f = d / sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
        const double C[3] = {n[0] * f, n[1] * f, n[2] * f};
        double M[PREC4];
        cell(g, 0.6 * d, ORDER, M);
        T rec[PREC4];
        for (int k = 0; k < PREC4; k++) rec[k] = (T)M[k];
        lx_add_cell<ORDER, SOFT, T>(rec, T(1), (T)C[0], (T)C[1], (T)C[2], (T)eps2, (T)rs, A.data());
        for (int i = 0; i < 64; i++) {
            const double X[3] = {s[i][0] - C[0], s[i][1] - C[1], s[i][2] - C[2]};
            field(M, ORDER, X, eps2, ref[i].data());
        }
    }
    double worst = 0, rms = 0, wphi = 0, rphi = 0;
    for (int i = 0; i < 64; i++) {
        T o[4];
        lx_evaluate<SOFT, 0, T>(A.data(), (T)(s[i][0] / rs), (T)(s[i][1] / rs), (T)(s[i][2] / rs), (T)(1 / rs), o);
        double e = 0;
        for (int k = 0; k < 3; k++) {
            e += (o[k] - ref[i][k]) * (o[k] - ref[i][k]);
            rms += ref[i][k] * ref[i][k] / 64;
        }
        worst = std::max(worst, sqrt(e));
        wphi = std::max(wphi, std::fabs(o[3] - ref[i][3]));
        rphi += ref[i][3] * ref[i][3] / 64;
    }
    printf("%d %d %d %g %g %.3e %.3e\n", ORDER, (int)SOFT, (int)sizeof(T), rho, eta, worst / sqrt(rms),
           wphi / sqrt(rphi));
}

}  // namespace

int main() {
    for (double rho : {0.01, 0.05, 0.17}) {
        run<0, false, double>(rho, 0);
        run<2, false, double>(rho, 0);
        run<4, false, double>(rho, 0);
        run<0, false, float>(rho, 0);
        run<2, false, float>(rho, 0);
        run<4, false, float>(rho, 0);
        for (double eta : {1e-8, 1e-4}) {
            run<0, true, double>(rho, eta);
            run<2, true, double>(rho, eta);
            run<4, true, double>(rho, eta);
            run<0, true, float>(rho, eta);
            run<2, true, float>(rho, eta);
            run<4, true, float>(rho, eta);
        }
    }
    for (double rho : {0.05, 0.17})
        for (double bd : {0.0, 0.2, 0.4, 0.5, 0.6}) {
            if (bd == 0.0)
                run_two<0>(rho, 1e-3);
            else {
                run_two<2>(rho, bd);
                run_two<4>(rho, bd);
            }
        }
    return 0;
}
