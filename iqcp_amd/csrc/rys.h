// Rys quadrature nodes/weights from the piecewise fits in rys_table.inc.
//
// Same quantities as qc-core's rys_roots (crates/qc-core/src/rys/mod.rs:253): n nodes
// u_i = t_i^2 in [0,1) and weights with sum_i w_i u_i^k = F_k(T) for k < 2n.  The reference
// solves for them per call (Boys moments -> Schmidt -> Hessenberg QR, rys/mod.rs:468-583);
// here they are read from fits of the exact rule (see gen_rys_table.py), so every lane
// follows the same instruction stream.  Accuracy of the FP64 fits: ~1e-15 relative.
#pragma once
#include "qcg_common.h"
#include "rys_table.inc"

namespace qcg {

QCG_HD constexpr int rys_tri(int n) { return n * (n - 1) / 2; }

// Table entries of one interval and of the whole N-point rule.
template <int N>
constexpr int rys_stride() { return 2 * N * (qcg_rys_deg[N] + 1) + QCG_RYS_PAD; }
template <int N>
constexpr int rys_tab_size() { return qcg_rys_nint[N] * rys_stride<N>(); }

// The per-lane kernels gather the coefficients at lane-dependent intervals (from LDS up to N = 3), once
// per primitive quartet, and for the classes of low angular momentum that is what bounds them: with 14
// coefficients per polynomial on equal intervals the kernels of a (H2O)16 6-31G* FP64 build took 4.33 ms
// one after the other and the 64-alkane batch 20.8 ms, with 10 (N <= 2) or 12 on intervals that widen with
// T and strides that spread the intervals over the banks 4.01 and 19.0 ms.  (The staged tables are of 902, 1848
// and 2294 words for one to three nodes; 560, 1288 and 2268 before.)
// c[0] + c[1] s + ... + c[DEG] s^DEG in Estrin's scheme: dependency depth 5 instead of Horner's DEG
// (the FP64 FMA latency, not the issue rate, bounds a lone Horner chain per lane).
template <int DEG, typename R>
QCG_HD R rys_poly(const R* __restrict__ c, R s) {
    static_assert(DEG == 9 || DEG == 11, "degrees of the fits");
    const R s2 = s * s, s4 = s2 * s2, s8 = s4 * s4;
    const R t0 = c[0] + c[1] * s, t1 = c[2] + c[3] * s, t2 = c[4] + c[5] * s, t3 = c[6] + c[7] * s;
    R t4 = c[8] + c[9] * s;
    if constexpr (DEG == 11) t4 += (c[10] + c[11] * s) * s2;
    const R u0 = t0 + t1 * s2, u1 = t2 + t3 * s2;
    return (u0 + u1 * s4) + t4 * s8;
}

// The interval of T (below tmax) and the local variable s in [-1, 1]: exponent and leading mantissa bits
// of T + T0 name the interval, its midpoint and its width are bit patterns too.  The index is clamped, so
// a T that is no number reads within the table.
template <int N>
QCG_HD int rys_interval(double T, double& s) {
    constexpr int B = qcg_rys_bits[N], L = qcg_rys_log2t0[N];
    const unsigned hi = (unsigned)(__builtin_bit_cast(unsigned long long, T + (double)(1 << L)) >> 32);
    const unsigned mid = (hi & (~0u << (20 - B))) | (1u << (19 - B)), sc = ((unsigned)(2047 + B) << 20) - (hi & 0x7ff00000u);
    s = (T - (__builtin_bit_cast(double, (unsigned long long)mid << 32) - (double)(1 << L))) *
        __builtin_bit_cast(double, (unsigned long long)sc << 32);
    const unsigned k = (hi >> (20 - B)) - ((unsigned)(1023 + L) << B);
    return (int)(k < (unsigned)qcg_rys_nint[N] ? k : (unsigned)qcg_rys_nint[N] - 1);
}
template <int N>
QCG_HD int rys_interval(float T, float& s) {
    constexpr int B = qcg_rys_bits[N], L = qcg_rys_log2t0[N];
    const unsigned hi = __builtin_bit_cast(unsigned, T + (float)(1 << L));
    const unsigned mid = (hi & (~0u << (23 - B))) | (1u << (22 - B)), sc = ((unsigned)(255 + B) << 23) - (hi & 0x7f800000u);
    s = (T - (__builtin_bit_cast(float, mid) - (float)(1 << L))) * __builtin_bit_cast(float, sc);
    const unsigned k = (hi >> (23 - B)) - ((unsigned)(127 + L) << B);
    return (int)(k < (unsigned)qcg_rys_nint[N] ? k : (unsigned)qcg_rys_nint[N] - 1);
}

// tabN: the coefficients of the N-point rule, i.e. qcg_rys_coef + qcg_rys_off[N] (or its float
// copy), in device memory or staged in LDS.
template <typename R, int N>
QCG_HD void rys_eval_tab(R T, const R* __restrict__ tabN, R* x, R* w) {
    static_assert(N >= 1 && N <= QCG_RYS_NMAX, "Rys order out of table range");
    if (T >= (R)qcg_rys_tmax[N]) {
        const R rs = qrsqrt(T);
        const R it = rs * rs;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            x[i] = (R)qcg_rys_hx[rys_tri(N) + i] * it;
            w[i] = (R)qcg_rys_hw[rys_tri(N) + i] * rs;
        }
        return;
    }
    R s;
    const R* c = tabN + rys_interval<N>(T, s) * rys_stride<N>();
#pragma unroll
    for (int i = 0; i < 2 * N; ++i) {
        const R v = rys_poly<qcg_rys_deg[N]>(c + i * (qcg_rys_deg[N] + 1), s);
        if (i < N) x[i] = v; else w[i - N] = v;
    }
}

// Node r (runtime) of the rule: the same fits and asymptotic form.
template <typename R, int N>
QCG_HD void rys_eval_node(R T, const R* __restrict__ tabN, int r, R& x, R& w) {
    if (T >= (R)qcg_rys_tmax[N]) {
        const R rs = qrsqrt(T);
        const R it = rs * rs;
        x = (R)qcg_rys_hx[rys_tri(N) + r] * it;
        w = (R)qcg_rys_hw[rys_tri(N) + r] * rs;
        return;
    }
    constexpr int NC = qcg_rys_deg[N] + 1;
    R s;
    const R* cx = tabN + rys_interval<N>(T, s) * rys_stride<N>() + r * NC;
    x = rys_poly<qcg_rys_deg[N]>(cx, s);
    w = rys_poly<qcg_rys_deg[N]>(cx + N * NC, s);
}

// tab: qcg_rys_coef (double) or its float copy, resident in device memory.
template <typename R, int N>
QCG_HD void rys_eval(R T, const R* __restrict__ tab, R* x, R* w) {
    rys_eval_tab<R, N>(T, tab + qcg_rys_off[N], x, w);
}

// Runtime-order variant for host code and batch kernels.
template <typename R>
QCG_HD int rys_eval_n(int n, R T, const R* __restrict__ tab, R* x, R* w) {
    switch (n) {
        case 1: rys_eval<R, 1>(T, tab, x, w); return 0;
        case 2: rys_eval<R, 2>(T, tab, x, w); return 0;
        case 3: rys_eval<R, 3>(T, tab, x, w); return 0;
        case 4: rys_eval<R, 4>(T, tab, x, w); return 0;
        case 5: rys_eval<R, 5>(T, tab, x, w); return 0;
        case 6: rys_eval<R, 6>(T, tab, x, w); return 0;
        case 7: rys_eval<R, 7>(T, tab, x, w); return 0;
        default: return QCG_INVALID_ARG;
    }
}

}  // namespace qcg
