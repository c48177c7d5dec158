// A sink group's local expansion of its far cells: the sum of their multipole
// fields about the group centre, to degree LX_P, built one cell per lane and
// evaluated once per sink.  No HIP dependency: host tests compile the same code.
//
// The pair kernels take a cell's field psi = sum_k P_k(x) / w^(2k+1), x = sink -
// cell, w^2 = |x|^2 + eps^2, P_k the record's harmonic polynomial of degree k
// (pgrav_device.h; phi = -psi, a = grad psi), sink by sink.  For a cell at c = d n
// from the group centre, d well above the sinks' distance r_s from it, the same
// field is
//   psi(s) = sum_{l <= LX_P} sum_m A_lm H_lm(s) + |s|^2 sum_{l <= 3} sum_m B_lm H_lm(s)
//            + |s|^4 sum_{l <= 1} sum_m C_lm H_lm(s)
// with H the real solid harmonics below.  B and C belong to softened cells, whose
// field is not harmonic: they are kept to first order in (eps / d)^2 and to total
// degree 5 in s.
//
// Harmonics: E_l^m = C_l^m + i S_l^m, the coefficients of t^m in
// (u(t).x)^l / l!, u = ((t - 1/t)/2, i (t + 1/t)/2, 1), that is
//   E_0^0 = 1, E_m^m = (x + iy)/(2m) E_{m-1}^{m-1},
//   E_l^m = ((2l-1) z E_{l-1}^m - r^2 E_{l-2}^m) / ((l+m)(l-m)),
//   dE_l^m/dz = E_{l-1}^m, (d/dx -+ i d/dy) E_l^m = +-E_{l-1}^{m-+1},
//   E_l^{-m} = (-1)^m conj(E_l^m).
// Coefficient order: degree l at l^2: C_l^0, C_l^1, S_l^1, C_l^2, ...
//
// Translation: the moments are turned so that the cell lies on the z axis, where
//   E_k^m(s - d z) / |s - d z|^(2k+1) = sum_l (-1)^(k+m) (k+l)! / ((k+m)! (k-m)!)
//                                       E_l^m(s) / d^(k+l+1)
// couples only equal m, and the result is turned back.  A turn about z is one
// complex product per m; the turn about y is a turn about z between two exchanges of
// the axes y and z, whose constant matrices (LX_SWAP) are three quarters zeros.
#pragma once
#include <math.h>

#include <type_traits>

#include "pgrav_record.h"

namespace pgrav {

constexpr int LX_P = 8;  // degree of the expansion
constexpr int LX_N = (LX_P + 1) * (LX_P + 1);
constexpr int LX_NB = 16, LX_NC = 4;  // coefficients with |s|^2 and |s|^4 (softened cells)
constexpr int LX_ALL = LX_N + LX_NB + LX_NC;  // A, B, C one after another

PGRAV_HD constexpr int lx_c(int l, int m) { return l * l + (m ? 2 * m - 1 : 0); }
PGRAV_HD constexpr int lx_s(int l, int m) { return l * l + 2 * m; }

// f(0), f(1), ... with compile-time indices
template <int B, int E, class F>
PGRAV_HD inline __attribute__((always_inline)) void lx_for(F &&f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        lx_for<B + 1, E>(f);
    }
}
#define LX_I __attribute__((always_inline))

// H_i(x, z, y) = sum_j b[l][i][j] H_j(x, y, z) within degree l.  With y and z
// exchanged, u(t) becomes c u(t'), c = i (t^2 + 1)/(2t), t' = -i (t - i)/(t + i), so
// E_l^m(x, z, y) = sum_m' K_mm' E_l^m', K_mm' = (i/2)^l (-i)^m' times the coefficient
// of t^(l+m) in (t - i)^(l+m') (t + i)^(l-m').
struct LxSwap {
    double b[LX_P + 1][2 * LX_P + 1][2 * LX_P + 1];
};
constexpr LxSwap lx_make_swap() {
    LxSwap w{};
    for (int l = 0; l <= LX_P; l++) {
        double kr[2 * LX_P + 1][2 * LX_P + 1] = {}, ki[2 * LX_P + 1][2 * LX_P + 1] = {};
        for (int mp = -l; mp <= l; mp++) {
            double re[2 * LX_P + 2] = {}, im[2 * LX_P + 2] = {};
            re[0] = 1;
            for (int f = 0; f < 2 * l; f++) {
                const double a = f < l + mp ? -1.0 : 1.0;  // times (t + i a)
                for (int q = 2 * l; q >= 0; q--) {
                    const double r0 = re[q], i0 = im[q];
                    re[q] = (q ? re[q - 1] : 0.0) - a * i0;
                    im[q] = (q ? im[q - 1] : 0.0) + a * r0;
                }
            }
            double sc = 1.0;
            for (int f = 0; f < l; f++) sc *= 0.5;
            const int ph = ((l - mp) % 4 + 4) % 4;  // i^(l - m')
            for (int m = -l; m <= l; m++) {
                const double r0 = sc * re[l + m], i0 = sc * im[l + m];
                kr[l + m][l + mp] = ph == 0 ? r0 : (ph == 1 ? -i0 : (ph == 2 ? -r0 : i0));
                ki[l + m][l + mp] = ph == 0 ? i0 : (ph == 1 ? r0 : (ph == 2 ? -i0 : -r0));
            }
        }
        for (int m = 0; m <= l; m++)
            for (int mp = 0; mp <= l; mp++) {
                const double sg = mp % 2 ? -1.0 : 1.0;
                const double pr = kr[l + m][l + mp], pi = ki[l + m][l + mp];
                const double nr = mp ? sg * kr[l + m][l - mp] : 0.0, ni = mp ? sg * ki[l + m][l - mp] : 0.0;
                const int ic = m ? 2 * m - 1 : 0, jc = mp ? 2 * mp - 1 : 0;
                w.b[l][ic][jc] = pr + nr;
                if (mp)
                    w.b[l][ic][2 * mp] = ni - pi;
                if (m) {
                    w.b[l][2 * m][jc] = pi + ni;
                    if (mp)
                        w.b[l][2 * m][2 * mp] = pr - nr;
                }
            }
    }
    return w;
}
constexpr LxSwap LX_SWAP = lx_make_swap();

// The axial translation in units of D = sqrt(d^2 + eps^2), eta = (eps / D)^2:
// E_k^m(s - d z) w^-(2k+1) = sum_l (t + a eta + |s|^2 b eta + |s|^4 c eta + ...) E_l^m(s)
// to first order in eta.  Built by multiplying the shift of E_k^m,
// sum_j E_{k-j}^m(s) (-kappa)^j / j!, kappa = d / D, with the Gegenbauer series of
// (1 - 2 kappa z + |s|^2)^-(k+1/2), both as polynomials in z and u = |s|^2, and
// sorting each total degree n into E_n^m, u E_{n-2}^m, ...
struct LxAxial {
    double t[LX_P + 1][5][5], a[LX_P + 1][5][5], b[4][5][5], c[2][5][5];
};
constexpr LxAxial lx_make_axial() {
    constexpr int N = LX_P + 8;
    LxAxial r{};
    for (int m = 0; m <= 4; m++) {
        // e[l][j]: E_l^m / (x + iy)^m = sum_j e[l][j] z^(l-m-2j) u^j
        double e[N][N] = {};
        double d = 1;
        for (int q = 1; q <= m; q++) d *= 2.0 * q;
        e[m][0] = 1 / d;
        for (int l = m + 1; l < N; l++)
            for (int j = 0; 2 * j <= l - m; j++) {
                double v = 2 * j <= l - 1 - m ? (2 * l - 1) * e[l - 1][j] : 0.0;
                if (j && l - 2 >= m)
                    v -= e[l - 2][j - 1];
                e[l][j] = v / ((double)(l + m) * (l - m));
            }
        for (int k = m; k <= 4; k++) {
            // Gegenbauer terms, value and d/d eta (kappa = 1 - eta/2)
            const double lam = k + 0.5;
            double g[N][N] = {}, gd[N][N] = {};
            g[0][0] = 1;
            for (int q = 1; q < N; q++)
                for (int j = 0; 2 * j <= q; j++) {
                    const double f = 2 * (q + lam - 1) / q, h = (q + 2 * lam - 2) / q;
                    const double p = 2 * j <= q - 1 ? g[q - 1][j] : 0.0, pd = 2 * j <= q - 1 ? gd[q - 1][j] : 0.0;
                    g[q][j] = f * p - (j && q >= 2 ? h * g[q - 2][j - 1] : 0.0);
                    gd[q][j] = f * (pd - 0.5 * p) - (j && q >= 2 ? h * gd[q - 2][j - 1] : 0.0);
                }
            for (int n = m; n <= LX_P + 2; n++) {
                double F[N] = {}, Fd[N] = {};
                double fac = 1;  // (-1)^j / j!
                for (int s = 0; s <= k - m; s++) {
                    if (s)
                        fac *= -1.0 / s;
                    const int l = k - s, q = n - l;
                    if (q < 0)
                        continue;
                    for (int j = 0; 2 * j <= l - m; j++)
                        for (int i = 0; 2 * i <= q; i++) {
                            F[i + j] += fac * e[l][j] * g[q][i];
                            Fd[i + j] += fac * e[l][j] * (gd[q][i] - 0.5 * s * g[q][i]);
                        }
                }
                const double x0 = F[0] / e[n][0], x0d = Fd[0] / e[n][0];
                if (n <= LX_P) {
                    r.t[n][k][m] = x0;
                    r.a[n][k][m] = x0d;
                }
                if (n - 2 < m)
                    continue;
                const double x1d = (Fd[1] - x0d * e[n][1]) / e[n - 2][0];
                if (n - 2 <= 3)
                    r.b[n - 2][k][m] = x1d;
                if (n - 4 >= m && n - 4 <= 1)
                    r.c[n - 4][k][m] = (Fd[2] - x0d * e[n][2] - x1d * e[n - 2][1]) / e[n - 4][0];
            }
        }
    }
    return r;
}
constexpr LxAxial LX_AX = lx_make_axial();
constexpr int LX_SOFT_L = 5;  // degrees whose softening terms are kept: of a point, at (eps / d)^2
                              // = FAR_ETA and r_s = FAR_RHO d (pgrav_far.h), degree 6's is 2.6e-7
                              // of the pull and 7's 6e-8

template <typename T>
PGRAV_HD inline T lx_rsqrt(T x) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (sizeof(T) == 4)
        return __builtin_amdgcn_rsqf(x);
#endif
    return T(1) / sqrt(x);
}

// out_j += sum_i in_i b[l][i][j] over in_0 .. in_{NI-1}
template <int L, int NI, typename T>
PGRAV_HD inline LX_I void lx_swap(const T *in, T *out) {
    lx_for<0, 2 * L + 1>([&](auto j) LX_I {
        T v = T(0);
        lx_for<0, NI>([&](auto i) LX_I {
            constexpr double b = LX_SWAP.b[L][decltype(i)::value][decltype(j)::value];
            if constexpr (b != 0.0)
                v += T(b) * in[i];
        });
        out[j] = v;
    });
}

// (c_m, s_m) turned by m times the angle with cosines co[m] and sines si[m] * SG
template <int L, int SG, typename T>
PGRAV_HD inline LX_I void lx_turn(T *v, const T *co, const T *si) {
    lx_for<1, L + 1>([&](auto mm) LX_I {
        constexpr int m = decltype(mm)::value;
        const T c = v[2 * m - 1], s = v[2 * m];
        if constexpr (SG > 0) {
            v[2 * m - 1] = c * co[m] - s * si[m];
            v[2 * m] = c * si[m] + s * co[m];
        } else {
            v[2 * m - 1] = c * co[m] + s * si[m];
            v[2 * m] = s * co[m] - c * si[m];
        }
    });
}

// degree L of an expansion about the turned z axis (orders m <= M), turned back and
// added to acc
template <int L, int M, typename T>
PGRAV_HD inline LX_I void lx_turn_back(const T *in, const T *cp, const T *sp, const T *ct, const T *st,
                                       T *acc) {
    constexpr int NI = 2 * (M < L ? M : L) + 1;
    T v[2 * L + 1], w[2 * L + 1];
    lx_swap<L, NI>(in, v);
    lx_turn<L, -1>(v, ct, st);
    lx_swap<L, 2 * L + 1>(v, w);
    acc[0] += w[0];
    lx_for<1, L + 1>([&](auto mm) LX_I {
        constexpr int m = decltype(mm)::value;
        acc[2 * m - 1] += w[2 * m - 1] * cp[m];
        acc[2 * m - 1] -= w[2 * m] * sp[m];
        acc[2 * m] += w[2 * m - 1] * sp[m];
        acc[2 * m] += w[2 * m] * cp[m];
    });
}

// Adds to A the expansion of one cell at (cx, cy, cz) from the centre, in units of
// the length lam: the coefficients of H_lm(s / lam) and, SOFT, of |s / lam|^2 H_lm and
// |s / lam|^4 H_lm.  rec: the cell's prepared record
// (entries 4 .. 45 for orders 2 and 4), m its mass.
template <int ORDER, bool SOFT, typename T>
PGRAV_HD inline LX_I void lx_add_cell(const T *rec, T mass, T cx, T cy, T cz, T eps2, T lam,
                                      T *A) {
    T *B = A + LX_N, *C = B + LX_NB;
    const T d2 = cx * cx + cy * cy + cz * cz;
    const T iD = lx_rsqrt(SOFT ? d2 + eps2 : d2);
    const T rho = lam * iD;
    const T eta = SOFT ? (eps2 * iD) * iD : T(0);
    if constexpr (ORDER == 0) {
        // 1/w: coefficients (l+m)! (l-m)! E_l^m(c) / D^(2l+1) (twice for m > 0): by
        // J_m^m = (2m-1) (x+iy) J_{m-1}^{m-1}, J_l^m = (2l-1) z J_{l-1}^m -
        // ((l-1)^2 - m^2) r^2 J_{l-2}^m with (x, y, z) = c / D
        const T x = cx * iD, y = cy * iD, z = cz * iD;
        const T r2 = SOFT ? T(1) - eta : T(1);
        T wt[LX_P + 1];  // m / D (lam / D)^l
        wt[0] = mass * iD;
        lx_for<1, LX_P + 1>([&](auto l) LX_I { wt[l] = wt[l - 1] * rho; });
        const T eb = eta * rho * rho;
        T jc = T(1), js = T(0);
        lx_for<0, LX_P + 1>([&](auto mm) LX_I {
            constexpr int m = decltype(mm)::value;
            if constexpr (m > 0) {
                const T c = jc * x - js * y;
                js = T(2 * m - 1) * (jc * y + js * x);
                jc = T(2 * m - 1) * c;
            }
            T c1 = jc, s1 = js, c2 = T(0), s2 = T(0);
            lx_for<m, LX_P + 1>([&](auto ll) LX_I {
                constexpr int l = decltype(ll)::value;
                if constexpr (l > m) {
                    const T g = T(2 * l - 1) * z;
                    constexpr T h = T((l - 1) * (l - 1) - m * m);
                    const T c = g * c1 - h * r2 * c2, s = g * s1 - h * r2 * s2;
                    c2 = c1;
                    s2 = s1;
                    c1 = c;
                    s1 = s;
                }
                const T w = m ? T(2) * wt[l] : wt[l];
                A[lx_c(l, m)] += w * c1;
                if constexpr (m > 0)
                    A[lx_s(l, m)] += w * s1;
                if constexpr (SOFT && l <= 3) {
                    const T v = w * eb * T(LX_AX.b[l][0][0] / LX_AX.t[l][0][0]);
                    B[lx_c(l, m)] += v * c1;
                    if constexpr (m > 0)
                        B[lx_s(l, m)] += v * s1;
                }
                if constexpr (SOFT && l <= 1) {
                    const T v = w * (eb * rho * rho) * T(LX_AX.c[l][0][0] / LX_AX.t[l][0][0]);
                    C[lx_c(l, m)] += v * c1;
                    if constexpr (m > 0)
                        C[lx_s(l, m)] += v * s1;
                }
            });
        });
        return;
    } else {
        constexpr int M = ORDER;  // highest order m of the moments
        const T id = SOFT ? lx_rsqrt(d2) : iD;
        const T nx = cx * id, ny = cy * id, nz = cz * id;
        const T t2 = nx * nx + ny * ny;
        const bool tilt = t2 > T(1e-24);
        const T it = lx_rsqrt(tilt ? t2 : T(1));
        // cosines and sines of m phi and m theta
        T cp[LX_P + 1], sp[LX_P + 1], ct[LX_P + 1], st[LX_P + 1];
        cp[1] = tilt ? nx * it : T(1);
        sp[1] = tilt ? ny * it : T(0);
        ct[1] = nz;
        st[1] = tilt ? t2 * it : T(0);
        lx_for<2, LX_P + 1>([&](auto m) LX_I {
            cp[m] = cp[m - 1] * cp[1] - sp[m - 1] * sp[1];
            sp[m] = sp[m - 1] * cp[1] + cp[m - 1] * sp[1];
            ct[m] = ct[m - 1] * ct[1] - st[m - 1] * st[1];
            st[m] = st[m - 1] * ct[1] + ct[m - 1] * st[1];
        });
        // moments on E_k^m: derivatives d/dz^(k-m) (d/dx - i d/dy)^m of P_k (whose
        // gradient is k G_k), doubled and conjugated for m > 0
        T q2[5], q3[7], q4[9];
        const T *o = rec + 10, *h = rec + 25;
        q2[0] = T(2) * rec[9];
        q2[1] = T(4) * rec[6];
        q2[2] = T(4) * rec[8];
        q2[3] = T(4) * (rec[4] - rec[7]);
        q2[4] = T(8) * rec[5];
        if constexpr (ORDER == 4) {
            q3[0] = T(-6) * (o[10] + o[11]);
            q3[1] = T(6) * o[13];
            q3[2] = T(6) * o[14];
            q3[3] = T(12) * (o[10] - o[11]);
            q3[4] = T(12) * o[12];
            q3[5] = T(12) * (o[0] - o[1] - o[7]);
            q3[6] = T(12) * (o[2] + o[5] - o[6]);
            q4[0] = T(-24) * (h[17] + h[20]);
            q4[1] = T(-16) * (T(3) * h[14] + h[18]);
            q4[2] = T(-16) * (T(3) * h[15] + h[16]);
            q4[3] = T(48) * (h[17] - h[20]);
            q4[4] = T(16) * h[19];
            q4[5] = T(48) * (h[14] - h[18]);
            q4[6] = T(48) * (h[16] - h[15]);
            q4[7] = T(48) * ((h[0] - h[4]) + (h[8] - h[9]));
            q4[8] = T(48) * ((h[7] - h[11]) - (h[1] - h[2]));
        }
        // into the turned frame, scaled by D^-(k+1) (no power of 1/D beyond the third is
        // formed, as in the pair kernels, so the range of usable units is theirs)
        T a[5][9];  // a[k]: the order-k moments there
        const T iD2 = iD * iD, f3 = iD * iD2;
        a[0][0] = mass * iD;
        {
            T v[5], w[5];
            lx_turn<2, -1>(q2, cp, sp);
            lx_swap<2, 5>(q2, v);
            lx_turn<2, 1>(v, ct, st);
            lx_swap<2, 5>(v, w);
            lx_for<0, 5>([&](auto i) LX_I { a[2][i] = w[i] * f3; });
        }
        if constexpr (ORDER == 4) {
            T v[7], w[7];
            lx_turn<3, -1>(q3, cp, sp);
            lx_swap<3, 7>(q3, v);
            lx_turn<3, 1>(v, ct, st);
            lx_swap<3, 7>(v, w);
            lx_for<0, 7>([&](auto i) LX_I { a[3][i] = (w[i] * iD) * f3; });
            T y[9], z[9];
            lx_turn<4, -1>(q4, cp, sp);
            lx_swap<4, 9>(q4, y);
            lx_turn<4, 1>(y, ct, st);
            lx_swap<4, 9>(y, z);
            lx_for<0, 9>([&](auto i) LX_I { a[4][i] = (z[i] * iD2) * f3; });
        }
        T pw = T(1);  // (lam / D)^l
        lx_for<0, LX_P + 1>([&](auto ll) LX_I {
            constexpr int l = decltype(ll)::value;
            constexpr int ML = M < l ? M : l;
            T v[2 * ML + 1];
            lx_for<0, 2 * ML + 1>([&](auto ii) LX_I {
                constexpr int i = decltype(ii)::value, m = (i + 1) / 2;
                T s = T(0);
                lx_for<0, ORDER + 1>([&](auto kk) LX_I {
                    constexpr int k = decltype(kk)::value;
                    if constexpr (k != 1 && k >= m) {
                        constexpr T t = T(LX_AX.t[l][k][m]), e = T(LX_AX.a[l][k][m]);
                        if constexpr (SOFT && l <= LX_SOFT_L && e != T(0))
                            s += (t + e * eta) * a[k][i];
                        else
                            s += t * a[k][i];
                    }
                });
                v[i] = s * pw;
            });
            lx_turn_back<l, M>(v, cp, sp, ct, st, A + l * l);
            if constexpr (SOFT && l <= 3) {
                const T f = eta * pw * rho * rho;
                lx_for<0, 2 * ML + 1>([&](auto ii) LX_I {
                    constexpr int i = decltype(ii)::value, m = (i + 1) / 2;
                    T s = T(0);
                    lx_for<0, ORDER + 1>([&](auto kk) LX_I {
                        constexpr int k = decltype(kk)::value;
                        if constexpr (k != 1 && k >= m)
                            s += T(LX_AX.b[l][k][m]) * a[k][i];
                    });
                    v[i] = s * f;
                });
                lx_turn_back<l, M>(v, cp, sp, ct, st, B + l * l);
                if constexpr (l <= 1) {
                    lx_for<0, 2 * ML + 1>([&](auto ii) LX_I {
                        constexpr int i = decltype(ii)::value, m = (i + 1) / 2;
                        T s = T(0);
                        lx_for<0, ORDER + 1>([&](auto kk) LX_I {
                            constexpr int k = decltype(kk)::value;
                            if constexpr (k != 1 && k >= m)
                                s += T(LX_AX.c[l][k][m]) * a[k][i];
                        });
                        v[i] = s * (f * rho * rho);
                    });
                    lx_turn_back<l, M>(v, cp, sp, ct, st, C + l * l);
                }
            }
            pw *= rho;
        });
    }
}

// The expansion at s = lam (x, y, z): out = grad psi (3) and -psi, with ilam = 1 / lam;
// degrees LMIN.. of A only (a caller may add the lower ones in higher precision).
template <bool SOFT, int LMIN = 0, typename T>
PGRAV_HD inline LX_I void lx_evaluate(const T *A, T x, T y, T z, T ilam, T *out) {
    const T *B = A + LX_N, *C = B + LX_NB;
    const T r2 = x * x + y * y + z * z;
    T psi = T(0), gx = T(0), gy = T(0), gz = T(0);
    T bp = T(0), bx = T(0), by = T(0), bz = T(0);  // the |s|^2 and |s|^4 factors
    T ep = T(0), ex = T(0), ey = T(0), ez = T(0);
    T pc[LX_P + 2], ps[LX_P + 2], p2c[LX_P + 1], p2s[LX_P + 1];  // degrees l - 1 and l - 2
    lx_for<0, LX_P + 1>([&](auto ll) LX_I {
        constexpr int l = decltype(ll)::value;
        T c[LX_P + 1], s[LX_P + 1];
        lx_for<0, l + 1>([&](auto mm) LX_I {
            constexpr int m = decltype(mm)::value;
            if constexpr (l == 0) {
                c[0] = T(1);
                s[0] = T(0);
            } else if constexpr (m == l) {
                constexpr T f = T(1.0 / (2.0 * m));
                c[m] = f * (x * pc[m - 1] - y * ps[m - 1]);
                s[m] = f * (x * ps[m - 1] + y * pc[m - 1]);
            } else {
                constexpr T f = T(1.0 / ((double)(l + m) * (l - m)));
                const T g = T(2 * l - 1) * z;
                if constexpr (l - 2 >= m) {
                    c[m] = f * (g * pc[m] - r2 * p2c[m]);
                    s[m] = f * (g * ps[m] - r2 * p2s[m]);
                } else {
                    c[m] = f * (g * pc[m]);
                    s[m] = f * (g * ps[m]);
                }
            }
        });
        // value and gradient terms of degree l (the gradient through degree l - 1)
        auto add = [&](const T *K, T &p, T &vx, T &vy, T &vz) LX_I {
            lx_for<0, l + 1>([&](auto mm) LX_I {
                constexpr int m = decltype(mm)::value;
                const T a = K[lx_c(l, m)];
                p += a * c[m];
                if constexpr (m == 0) {
                    if constexpr (l >= 1)
                        vz += a * pc[0];
                    if constexpr (l >= 2) {
                        vx -= a * pc[1];
                        vy -= a * ps[1];
                    }
                } else {
                    const T b = K[lx_s(l, m)];
                    p += b * s[m];
                    const T ha = T(0.5) * a, hb = T(0.5) * b;
                    vx += ha * pc[m - 1];
                    vy += hb * pc[m - 1];
                    if constexpr (m > 1) {
                        vx += hb * ps[m - 1];
                        vy -= ha * ps[m - 1];
                    }
                    if constexpr (m <= l - 1) {
                        vz += a * pc[m];
                        vz += b * ps[m];
                    }
                    if constexpr (m + 1 <= l - 1) {
                        vx -= ha * pc[m + 1];
                        vx -= hb * ps[m + 1];
                        vy -= ha * ps[m + 1];
                        vy += hb * pc[m + 1];
                    }
                }
            });
        };
        if constexpr (l >= LMIN)
            add(A, psi, gx, gy, gz);
        if constexpr (SOFT && l <= 3)
            add(B, bp, bx, by, bz);
        if constexpr (SOFT && l <= 1)
            add(C, ep, ex, ey, ez);
        lx_for<0, l + 1>([&](auto m) LX_I {
            if constexpr (decltype(m)::value < l) {
                p2c[m] = pc[m];
                p2s[m] = ps[m];
            }
            pc[m] = c[m];
            ps[m] = s[m];
        });
    });
    if constexpr (SOFT) {
        // |s|^2 (b + |s|^2 e)
        const T q = bp + r2 * ep, f = T(2) * (q + r2 * ep);
        psi += r2 * q;
        gx += r2 * (bx + r2 * ex) + x * f;
        gy += r2 * (by + r2 * ey) + y * f;
        gz += r2 * (bz + r2 * ez) + z * f;
    }
    out[0] = gx * ilam;
    out[1] = gy * ilam;
    out[2] = gz * ilam;
    out[3] = -psi;
}

}  // namespace pgrav
