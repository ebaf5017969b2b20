// One-electron integrals and gradient terms of one primitive pair (onee_kernels.hip).
//
// sum_ab D_ab dH_ab/dR - W_ab dS_ab/dR, H = T + V, for the primitive pair (pi, pj) of the shell pair
// (si, sj) (overlap_derivative_matrix, scf/gradient.rs:188, and hcore_derivative_matrix
// :355, contracted as in rhf_gradient :930-950).  Basis-function derivatives:
// d/dA_x phi_i = 2 alpha phi_(i+1) - i phi_(i-1); for V the operator centre C gets -(dA + dB) by
// translational invariance of each three-centre integral.
#pragma once
#include <cmath>

#include "eri_device.h"
#include "qcg_common.h"
#include "rys.h"

namespace qcg {

// Plain-pointer view of a basis (host vectors or device copies).
struct BasisView {
    int nshell, nbf, natom;
    const int *l, *nprim, *prim_off, *shell_atom, *bf_off, *Z;
    const double *exps, *coefs, *centers, *xyz;
};

// Radial normalisation (2a/pi)^(3/4) (4a)^(l/2) of one primitive (cartesian_gaussian_normalization
// without the component factor, integrals/overlap.rs:343-377).
QCG_HD double onee_norm_radial(double a, int l) {
    const double two_a_pi = 2.0 * a / kPi;
    const double base = sqrt(sqrt(two_a_pi * two_a_pi * two_a_pi));
    const double fa = 4.0 * a;
    double num = 1.0;
    if (l == 1) num = sqrt(fa);
    else if (l == 2) num = fa;
    else if (l > 2) num = pow(fa, l / 2.0);
    return base * num;
}

QCG_HD double onee_norm_comp(int l, int c) {
    return 1.0 / sqrt(dfact_odd(cart_x(l, c)) * dfact_odd(cart_y(l, c)) * dfact_odd(cart_z(l, c)));
}

// 1-D overlap table s[i][j], i <= imax, j <= jmax (Obara-Saika), without the exp/sqrt prefactor.
QCG_HD void onee_overlap_1d(double PA, double PB, double oo2p, int imax, int jmax, double* s, int ld) {
    s[0] = 1.0;
    for (int i = 0; i <= imax; ++i)
        for (int j = 0; j <= jmax; ++j) {
            if (i == 0 && j == 0) continue;
            double v;
            if (i > 0) {
                v = PA * s[(i - 1) * ld + j];
                if (i > 1) v += (i - 1) * oo2p * s[(i - 2) * ld + j];
                if (j > 0) v += j * oo2p * s[(i - 1) * ld + j - 1];
            } else {
                v = PB * s[i * ld + j - 1];
                if (j > 1) v += (j - 1) * oo2p * s[i * ld + j - 2];
            }
            s[i * ld + j] = v;
        }
}

// Rys rule of n <= 3 nodes (the most the one-electron terms of s, p, d shells need, derivatives
// included): only these orders are instantiated, which keeps the kernels' registers down.
QCG_HD void onee_rys(int n, double T, const double* rys_tab, double* x, double* w) {
    static_assert(kMaxL <= 2, "one-electron Rys orders above 3");
    if (n == 1) rys_eval<double, 1>(T, rys_tab, x, w);
    else if (n == 2) rys_eval<double, 2>(T, rys_tab, x, w);
    else rys_eval<double, 3>(T, rys_tab, x, w);
}

// Geometry and contraction data of one primitive pair.
struct OneePair {
    int la, lb, na, nb, atA, atB, bfa, bfb;
    double a, b, p, oo2p, kab, ca, cb;
    double AB[3], P[3], PA[3], PB[3];
};

QCG_HD OneePair onee_pair_setup(const BasisView& B, int si, int sj, int pi, int pj) {
    OneePair q;
    q.la = B.l[si];
    q.lb = B.l[sj];
    q.na = ncart(q.la);
    q.nb = ncart(q.lb);
    q.atA = B.shell_atom[si];
    q.atB = B.shell_atom[sj];
    q.bfa = B.bf_off[si];
    q.bfb = B.bf_off[sj];
    const double* A = &B.centers[3 * si];
    const double* Bc = &B.centers[3 * sj];
    for (int x = 0; x < 3; ++x) q.AB[x] = A[x] - Bc[x];
    const double ab2 = q.AB[0] * q.AB[0] + q.AB[1] * q.AB[1] + q.AB[2] * q.AB[2];
    q.a = B.exps[B.prim_off[si] + pi];
    q.b = B.exps[B.prim_off[sj] + pj];
    q.ca = B.coefs[B.prim_off[si] + pi] * onee_norm_radial(q.a, q.la);
    q.cb = B.coefs[B.prim_off[sj] + pj] * onee_norm_radial(q.b, q.lb);
    q.p = q.a + q.b;
    q.oo2p = 0.5 / q.p;
    q.kab = exp(-(q.a * q.b / q.p) * ab2);
    for (int x = 0; x < 3; ++x) {
        q.P[x] = (q.a * A[x] + q.b * Bc[x]) / q.p;
        q.PA[x] = q.P[x] - A[x];
        q.PB[x] = q.P[x] - Bc[x];
    }
    return q;
}

// Density element (or sum of the mirrored ones) of a component pair of the unordered shell pair.
QCG_HD double onee_weight(const double* M, int nbf, int i, int j, bool mirror) {
    const double v = M[(size_t)i * nbf + j];
    return mirror ? v + M[(size_t)j * nbf + i] : v;
}

// Overlap and kinetic terms of the primitive pair (pi, pj) of the shell pair (si, sj) of angular momenta
// LA, LB; mirror: the pair stands for (sj, si) too.  gA, gB: the derivative sums of the two centres.
template <int LA, int LB>
QCG_HD void onee_grad_overlap_kinetic(const BasisView& B, int si, int sj, int pi, int pj, bool mirror, const double* D,
                                      const double* W, double* gA, double* gB) {
    constexpr int NB = ncart(LB), NQ = ncart(LA) * NB, LD = LB + 3;
    const OneePair q = onee_pair_setup(B, si, sj, pi, pj);
    const double a = q.a, b = q.b;
    // per axis S(i, j), i <= LA + 2, j <= LB + 2, and T(i, j), i <= LA + 1, j <= LB + 1
    double s[3][(LA + 3) * LD], t[3][(LA + 2) * LD];
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        double* sx = s[x];
        sx[0] = 1.0;
        static_for<(LA + 3) * LD - 1>([&](auto ec) {
            constexpr int e = decltype(ec)::value + 1, i = e / LD, j = e % LD;
            double v;
            if constexpr (i > 0) {
                v = q.PA[x] * sx[e - LD];
                if constexpr (i > 1) v += (i - 1) * q.oo2p * sx[e - 2 * LD];
                if constexpr (j > 0) v += j * q.oo2p * sx[e - LD - 1];
            } else {
                v = q.PB[x] * sx[e - 1];
                if constexpr (j > 1) v += (j - 1) * q.oo2p * sx[e - 2];
            }
            sx[e] = v;
        });
        static_for<(LA + 2) * (LB + 2)>([&](auto ec) {
            constexpr int i = decltype(ec)::value / (LB + 2), j = decltype(ec)::value % (LB + 2), e = i * LD + j;
            double v = 4.0 * a * b * sx[e + LD + 1];
            if constexpr (i > 0) v -= 2.0 * b * i * sx[e - LD + 1];
            if constexpr (j > 0) v -= 2.0 * a * j * sx[e + LD - 1];
            if constexpr (i > 0 && j > 0) v += (double)(i * j) * sx[e - LD - 1];
            t[x][e] = 0.5 * v;
        });
    }
    const double pre = q.kab * (kPi / q.p) * sqrt(kPi / q.p) * q.ca * q.cb;
    static_for<NQ>([&](auto kc) {
        constexpr int k = decltype(kc)::value, ca = k / NB, cb = k % NB;
        constexpr int ip[3] = {cart_x(LA, ca), cart_y(LA, ca), cart_z(LA, ca)};
        constexpr int jp[3] = {cart_x(LB, cb), cart_y(LB, cb), cart_z(LB, cb)};
        constexpr int e[3] = {ip[0] * LD + jp[0], ip[1] * LD + jp[1], ip[2] * LD + jp[2]};
        const double nrm = pre * cnorm(LA, ca) * cnorm(LB, cb);
        const double dv = nrm * onee_weight(D, B.nbf, q.bfa + ca, q.bfb + cb, mirror);
        const double wv = nrm * onee_weight(W, B.nbf, q.bfa + ca, q.bfb + cb, mirror);
        static_for<3>([&](auto xc) {
            constexpr int x = decltype(xc)::value, y = (x + 1) % 3, z = (x + 2) % 3;
            const double sy = s[y][e[y]], sz = s[z][e[z]], syz = sy * sz, tyz = t[y][e[y]] * sz + sy * t[z][e[z]];
            // derivative with respect to A_x and B_x of S and T
            double dsA = 2.0 * a * s[x][e[x] + LD], dsB = 2.0 * b * s[x][e[x] + 1];
            double dtA = 2.0 * a * t[x][e[x] + LD], dtB = 2.0 * b * t[x][e[x] + 1];
            if constexpr (ip[x] > 0) {
                dsA -= ip[x] * s[x][e[x] - LD];
                dtA -= ip[x] * t[x][e[x] - LD];
            }
            if constexpr (jp[x] > 0) {
                dsB -= jp[x] * s[x][e[x] - 1];
                dtB -= jp[x] * t[x][e[x] - 1];
            }
            gA[x] += dv * (dtA * syz + dsA * tyz) - wv * dsA * syz;
            gB[x] += dv * (dtB * syz + dsB * tyz) - wv * dsB * syz;
        });
    });
}

// Nuclear attraction terms of nucleus cnuc for the primitive pair (pi, pj) of the shell pair (si, sj) of
// angular momenta LA, LB; mirror: the pair stands for (sj, si) too.  gA, gB: the derivative sums of the
// two centres.  One Rys node at a time, everything in registers: per axis the 1-D factors I(i, j) for
// i <= LA + 1, j <= LB, and I(i, j+1) = I(i+1, j) + AB I(i, j).
template <int LA, int LB>
QCG_HD void onee_grad_nuclear(const BasisView& B, int si, int sj, int pi, int pj, int cnuc, bool mirror,
                              const double* D, const double* rys_tab, double* gA, double* gB) {
    constexpr int N = (LA + LB + 1) / 2 + 1, NB = ncart(LB), NQ = ncart(LA) * NB, NM = LA + LB + 1;
    const OneePair q = onee_pair_setup(B, si, sj, pi, pj);
    const double* C = &B.xyz[3 * cnuc];
    const double PC[3] = {q.P[0] - C[0], q.P[1] - C[1], q.P[2] - C[2]};
    double rx[N], rw[N];
    rys_eval<double, N>(q.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]), rys_tab, rx, rw);
    const double pz = -(double)B.Z[cnuc] * 2.0 * kPi / q.p * q.kab * q.ca * q.cb;
    double W[NQ];
    static_for<NQ>([&](auto kc) {
        constexpr int k = decltype(kc)::value, a = k / NB, b = k % NB;
        W[k] = pz * cnorm(LA, a) * cnorm(LB, b) * onee_weight(D, B.nbf, q.bfa + a, q.bfb + b, mirror);
    });
    const double two_a = 2.0 * q.a, two_b = 2.0 * q.b;
#pragma unroll
    for (int r = 0; r < N; ++r) {
        const double u = rx[r], bb = (1.0 - u) * q.oo2p;
        double I[3][(LA + 2) * (LB + 1)];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            double h[NM + 1], t[NM + 1];
            const double c0 = q.PA[x] - u * PC[x];
            h[0] = 1.0;
            h[1] = c0;
#pragma unroll
            for (int n = 1; n < NM; ++n) h[n + 1] = c0 * h[n] + n * bb * h[n - 1];
#pragma unroll
            for (int j = 0; j <= LB; ++j) {
#pragma unroll
                for (int n = 0; n + j <= NM; ++n) {
                    t[n] = j == 0 ? h[n] : h[n + 1] + q.AB[x] * h[n];
                    if (n <= LA + 1) I[x][n * (LB + 1) + j] = t[n];
                }
#pragma unroll
                for (int n = 0; n + j <= NM; ++n) h[n] = t[n];
            }
        }
        static_for<NQ>([&](auto kc) {
            constexpr int k = decltype(kc)::value, a = k / NB, b = k % NB;
            constexpr int ip[3] = {cart_x(LA, a), cart_y(LA, a), cart_z(LA, a)};
            constexpr int jp[3] = {cart_x(LB, b), cart_y(LB, b), cart_z(LB, b)};
            constexpr int e[3] = {ip[0] * (LB + 1) + jp[0], ip[1] * (LB + 1) + jp[1], ip[2] * (LB + 1) + jp[2]};
            const double w = rw[r] * W[k];
            static_for<3>([&](auto xc) {
                constexpr int x = decltype(xc)::value, y = (x + 1) % 3, z = (x + 2) % 3;
                const double oth = w * (I[y][e[y]] * I[z][e[z]]);
                const double up = I[x][e[x] + LB + 1];
                double dA = two_a * up, dB = two_b * (up + q.AB[x] * I[x][e[x]]);
                if constexpr (ip[x] > 0) dA -= ip[x] * I[x][e[x] - (LB + 1)];
                if constexpr (jp[x] > 0) dB -= jp[x] * I[x][e[x] - 1];
                gA[x] += oth * dA;
                gB[x] += oth * dB;
            });
        });
    }
}

// One term of S, T, V for the Cartesian component pair (ia, jb) of the ordered shell pair (si, sj)
// and its primitive pair (pi, pj) (overlap_matrix, integrals/overlap.rs:647; kinetic,
// integrals/kinetic.rs; nuclear attraction, integrals/nuclear.rs:226), component norms left out:
// cnuc < 0: overlap and kinetic into out[0], out[1]; cnuc >= 0: the attraction to nucleus cnuc
// into out[2].  Overlap and kinetic from the Obara-Saika 1-D tables; V by Rys quadrature, the 1-D
// moments h_n = <(x-A)^n> by their two-term recurrence and (x-B)^j moved onto A binomially.
QCG_HD void onee_element_term(const BasisView& B, int si, int sj, int ia, int jb, int pi, int pj, int cnuc,
                              const double* rys_tab, double* out) {
    constexpr int LD = kMaxL + 3;
    const int la = B.l[si], lb = B.l[sj];
    const int ip[3] = {cart_x(la, ia), cart_y(la, ia), cart_z(la, ia)};
    const int jp[3] = {cart_x(lb, jb), cart_y(lb, jb), cart_z(lb, jb)};
    const OneePair q = onee_pair_setup(B, si, sj, pi, pj);
    if (cnuc < 0) {
        const double a = q.a, b = q.b;
        double s1[LD * LD];
        double sx[3], tx[3];
        for (int x = 0; x < 3; ++x) {
            const int i = ip[x], j = jp[x];
            onee_overlap_1d(q.PA[x], q.PB[x], q.oo2p, i + 1, j + 1, s1, LD);
            sx[x] = s1[i * LD + j];
            double v = 4.0 * a * b * s1[(i + 1) * LD + j + 1];
            if (i > 0) v -= 2.0 * b * i * s1[(i - 1) * LD + j + 1];
            if (j > 0) v -= 2.0 * a * j * s1[(i + 1) * LD + j - 1];
            if (i > 0 && j > 0) v += (double)(i * j) * s1[(i - 1) * LD + j - 1];
            tx[x] = 0.5 * v;
        }
        const double pre_s = q.kab * pow(kPi / q.p, 1.5) * q.ca * q.cb;
        out[0] += pre_s * sx[0] * sx[1] * sx[2];
        out[1] += pre_s * (tx[0] * sx[1] * sx[2] + sx[0] * tx[1] * sx[2] + sx[0] * sx[1] * tx[2]);
        return;
    }
    const int nr = (la + lb) / 2 + 1;
    const double* C = &B.xyz[3 * cnuc];
    const double PC[3] = {q.P[0] - C[0], q.P[1] - C[1], q.P[2] - C[2]};
    const double Tn = q.p * (PC[0] * PC[0] + PC[1] * PC[1] + PC[2] * PC[2]);
    double rx[QCG_RYS_NMAX], rw[QCG_RYS_NMAX];
    onee_rys(nr, Tn, rys_tab, rx, rw);
    double acc = 0.0;
    for (int r = 0; r < nr; ++r) {
        const double u = rx[r];
        double prod = rw[r];
        for (int x = 0; x < 3; ++x) {
            const int i = ip[x], j = jp[x];
            double h[2 * kMaxL + 1];
            const double c0 = q.PA[x] - u * PC[x];
            const double bb = (1.0 - u) * q.oo2p;
            h[0] = 1.0;
            if (i + j > 0) h[1] = c0;
            for (int n = 1; n < i + j; ++n) h[n + 1] = c0 * h[n] + n * bb * h[n - 1];
            // (x-B)^j = sum_k C(j,k) (x-A)^k (A-B)^(j-k), from k = j down
            double g = 0.0, pw = 1.0, cb = 1.0;
            for (int k = j; k >= 0; --k) {
                g += cb * pw * h[i + k];
                pw *= q.AB[x];
                cb = cb * k / (j - k + 1);
            }
            prod *= g;
        }
        acc += prod;
    }
    out[2] += -(double)B.Z[cnuc] * 2.0 * kPi / q.p * q.kab * q.ca * q.cb * acc;
}

}  // namespace qcg
