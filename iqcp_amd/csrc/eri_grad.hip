// Two-electron part of the analytic nuclear gradient (the adjoint of the Fock build) for all
// quartet classes whose bra pair class is QCG_CB (compiled once per bra class, like eri_jk.hip).
//
// Same quantity as qc-core's eri_gradient_fused (crates/qc-core/src/scf/gradient.rs:1430-1552) with
// compute_symmetry_weight (:1570-1627) and the derivative integrals of shell_eri_with_derivatives
// (integrals/eri/mod.rs:2035-2548):
//   dE/dR = sum over unique quartets, components: W_abcd d(ab|cd)/dR,
//   W_abcd = deg * 4 [ D_ab D_cd - c (D_ac D_bd + D_ad D_bc) ],  c = hf_frac / 4,
//   deg = 1/2 (a == b shell) * 1/2 (c == d shell) * 1/2 (pair P == pair Q)
// (the sum of 1/2 D_pq D_rs - c D_pr D_qs over the 8 index permutations).  Derivatives of a
// primitive with respect to its centre: d/dA_x phi_i = 2 alpha phi_(i+1) - i phi_(i-1), applied to
// the 1-D Rys factors for centres A, B, C; centre D by translational invariance, -(A + B + C).
//
// Per axis, with c(h) = sum over the components with 1-D index h of W times the other two axes' factors,
// the nine derivatives need only sum_h c(h) I(h), c(h) I(i+1), c(h) i I(i-1), ... : three products per
// component instead of nine, and the (j+1) factors follow from I(i, j+1) = I(i+1, j) + AB I(i, j).
//
// Per-lane form (one ket quartet per lane or lane group, everything in registers) for the classes whose
// components, or parts of them by component of the first shell, are at most kGradLaneMaxNQ; above that
// wave-cooperative (eri_wave.h): one wavefront per work item, one contracted quartet at a time.  Phase A
// writes the 1-D transfer tables with powers up to (la+1, lb+1, lc+1, ld) for (L+1)/2 + 1 Rys nodes (the
// derivative integrals have total angular momentum L+1) and the three primitive exponents of every
// primitive quartet to LDS; phase B has the lanes over Cartesian components: W_k times the nine
// derivative products, summed over the entries.  No derivative integral is stored.
#include "eri_launch.h"
#include "eri_wave.h"

#ifndef QCG_CB
#error "compile with -DQCG_CB=<bra pair class>"
#endif

namespace qcg {

template <int LA, int LB, int LC, int LD>
struct GradWave {
    using S = EriShape<LA, LB, LC, LD>;
    static constexpr int N = (LA + LB + LC + LD + 1) / 2 + 1;
    using T = WaveTable<LA + 1, LB + 1, LC + 1, LD, N, double>;
    static constexpr int DB = S::NAB + S::NCD + S::NA * S::NC + S::NB * S::ND + S::NA * S::ND + S::NB * S::NC;
    static constexpr int WAVE_D = T::DOUBLES + 3 * T::PQ_CAP + S::NQ + DB;
    // waves per block: four while their LDS fits in 64 KB, else two
    static constexpr int WPB = 4 * WAVE_D * 8 <= 65536 ? 4 : 2;
};

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void grad_wave_kernel(const int4* __restrict__ items, const int2* __restrict__ segs, int nitems,
                                                        const PairRec* __restrict__ bra, const PairRec* __restrict__ ket,
                                                        int diag, const PrimPair<double>* __restrict__ pp,
                                                        const double* __restrict__ rys_tab,
                                                        const double* __restrict__ D, int nbf_, double xfac,
                                                        double* __restrict__ grad) {
    using S = EriShape<LA, LB, LC, LD>;
    using G = GradWave<LA, LB, LC, LD>;
    using TB = typename G::T;
    constexpr int N = G::N, HT = TB::HT, ES = TB::ES;
    constexpr int NA = S::NA, NB = S::NB, NC = S::NC, ND = S::ND, NCD = S::NCD;
    constexpr int TB1 = LB + 2, TC1 = LC + 2, TD1 = LD + 1;
    constexpr int sI = TB1 * TC1 * TD1, sJ = TC1 * TD1, sK = TD1;
    __shared__ double smem[G::WPB * G::WAVE_D];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int item = blockIdx.x * G::WPB + wid;
    if (item >= nitems) return;  // waves are independent: no block-wide barrier below
    double* tbl = smem + wid * G::WAVE_D;
    double* alph = tbl + TB::DOUBLES;
    double* Wl = alph + 3 * TB::PQ_CAP;
    double* Dab = Wl + S::NQ;
    double* Dcd = Dab + S::NAB;
    double* Dac = Dcd + NCD;
    double* Dbd = Dac + NA * NC;
    double* Dad = Dbd + NB * ND;
    double* Dbc = Dad + NA * ND;
    const size_t nbf = (size_t)nbf_;

    const int4 it = items[item];
    const PairRec P = item_bra(bra, it);
    const int pidx = P.pos;
    KetCursor cur{segs, it.y, it.z};
    for (int o = lane; o < S::NAB; o += 64) Dab[o] = D[(P.bfa + o / NB) * nbf + P.bfb + o % NB];
    const double deg_p = (P.sa == P.sb) ? 0.5 : 1.0;
    double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};

    for (int j = 0; j < item_kets(it); ++j, ++cur.r) {
        const int q = cur.at();
        const PairRec Q = ket[q];
        const double deg = deg_p * ((Q.sa == Q.sb) ? 0.5 : 1.0) * ((diag && q == pidx) ? 0.5 : 1.0);
        wave_sync();  // previous quartet's readers of the weights and density blocks are done
        for (int o = lane; o < NCD; o += 64) Dcd[o] = D[(Q.bfa + o / ND) * nbf + Q.bfb + o % ND];
        for (int o = lane; o < NA * NC; o += 64) Dac[o] = D[(P.bfa + o / NC) * nbf + Q.bfa + o % NC];
        for (int o = lane; o < NB * ND; o += 64) Dbd[o] = D[(P.bfb + o / ND) * nbf + Q.bfb + o % ND];
        for (int o = lane; o < NA * ND; o += 64) Dad[o] = D[(P.bfa + o / ND) * nbf + Q.bfb + o % ND];
        for (int o = lane; o < NB * NC; o += 64) Dbc[o] = D[(P.bfb + o / NC) * nbf + Q.bfa + o % NC];
        wave_sync();
        for (int k = lane; k < S::NQ; k += 64) {
            const int d = k % ND, c = (k / ND) % NC, b = (k / NCD) % NB, a = k / (NCD * NB);
            Wl[k] = 4.0 * deg *
                    (Dab[a * NB + b] * Dcd[c * ND + d] - xfac * (Dac[a * NC + c] * Dbd[b * ND + d] + Dad[a * ND + d] * Dbc[b * NC + c])) *
                    cnorm(LA, a) * cnorm(LB, b) * cnorm(LC, c) * cnorm(LD, d);
        }
        double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};  // A xyz, B xyz, C xyz
        const int npq = P.npp * Q.npp;
        for (int pq0 = 0; pq0 < npq; pq0 += TB::PQ_CAP) {
            const int npc = min(TB::PQ_CAP, npq - pq0);
            wave_sync();
            wave_tables<LA + 1, LB + 1, LC + 1, LD, N, ES, double>(P, Q, pp, rys_tab, pq0, npc, tbl, lane);
            for (int u = lane; u < npc; u += 64) {
                const int pq = pq0 + u, i = pq / Q.npp, j = pq - i * Q.npp;
                const PrimPair<double>& a = pp[P.pp_off + i];
                alph[3 * u] = a.ea;
                alph[3 * u + 1] = a.p - a.ea;
                alph[3 * u + 2] = pp[Q.pp_off + j].ea;
            }
            wave_sync();
            const int ne = npc * N;
#pragma unroll 1
            for (int k = lane; k < S::NQ; k += 64) {
                const int d = k % ND, c = (k / ND) % NC, b = (k / NCD) % NB, a = k / (NCD * NB);
                const double w = Wl[k];
                // per axis: row pointers of I(i,j,k,l), I(i+1..), I(i-1..), I(.,j+1,..), ... and the powers
                const double* r0[3];
                const double *rAp[3], *rAm[3], *rBp[3], *rBm[3], *rCp[3], *rCm[3];
                double fi[3], fj[3], fk[3];
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    const int ia = x == 0 ? cart_x(LA, a) : x == 1 ? cart_y(LA, a) : cart_z(LA, a);
                    const int ib = x == 0 ? cart_x(LB, b) : x == 1 ? cart_y(LB, b) : cart_z(LB, b);
                    const int ic = x == 0 ? cart_x(LC, c) : x == 1 ? cart_y(LC, c) : cart_z(LC, c);
                    const int id = x == 0 ? cart_x(LD, d) : x == 1 ? cart_y(LD, d) : cart_z(LD, d);
                    const int h0 = ((ia * TB1 + ib) * TC1 + ic) * TD1 + id;
                    const double* base = tbl + x * HT * ES;
                    r0[x] = base + h0 * ES;
                    rAp[x] = base + (h0 + sI) * ES;
                    rAm[x] = base + (ia ? h0 - sI : h0) * ES;
                    rBp[x] = base + (h0 + sJ) * ES;
                    rBm[x] = base + (ib ? h0 - sJ : h0) * ES;
                    rCp[x] = base + (h0 + sK) * ES;
                    rCm[x] = base + (ic ? h0 - sK : h0) * ES;
                    fi[x] = ia;
                    fj[x] = ib;
                    fk[x] = ic;
                }
                double s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
                for (int e = 0; e < ne; ++e) {
                    const int pql = e / N;
                    const double two_a = 2.0 * alph[3 * pql], two_b = 2.0 * alph[3 * pql + 1],
                                 two_c = 2.0 * alph[3 * pql + 2];
                    const double i0x = r0[0][e], i0y = r0[1][e], i0z = r0[2][e];
                    const double iyz = i0y * i0z, ixz = i0x * i0z, ixy = i0x * i0y;
                    const double pr[3] = {iyz, ixz, ixy};
#pragma unroll
                    for (int x = 0; x < 3; ++x) {
                        s[x] += (two_a * rAp[x][e] - fi[x] * rAm[x][e]) * pr[x];
                        s[3 + x] += (two_b * rBp[x][e] - fj[x] * rBm[x][e]) * pr[x];
                        s[6 + x] += (two_c * rCp[x][e] - fk[x] * rCm[x][e]) * pr[x];
                    }
                }
#pragma unroll
                for (int t = 0; t < 9; ++t) acc[t] += w * s[t];
            }
        }
        // ket atoms: C directly, D = -(A + B + C) of this quartet (translational invariance)
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            gA[x] += acc[x];
            gB[x] += acc[3 + x];
            const double cx = wave_sum(acc[6 + x]);
            const double sx = wave_sum(acc[x] + acc[3 + x] + acc[6 + x]);
            if (lane == 0) {
                if (cx != 0.0) atomicAdd(&grad[3 * Q.atom_a + x], cx);
                if (sx != 0.0) atomicAdd(&grad[3 * Q.atom_b + x], -sx);
            }
        }
    }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const double ax = wave_sum(gA[x]), bx = wave_sum(gB[x]);
        if (lane == 0) {
            if (ax != 0.0) atomicAdd(&grad[3 * P.atom_a + x], ax);
            if (bx != 0.0) atomicAdd(&grad[3 * P.atom_b + x], bx);
        }
    }
}

// ------------------------------------------------------------------ per-lane form
// The wave-cooperative kernel reads 21 table entries from LDS per component, node and primitive quartet
// and is bound by them (VALU 10-15 % busy), so all classes but (dd|dd) and (dd|dp) run here, the large ones
// in parts: alone, octane/6-31+G*, (pp|pp) 2.11 -> 0.18 ms in three parts of 27 components, (dp|pp) 2.02 ->
// 0.21 in three of 54, (dp|ds) 1.84 -> 0.15 in two of 54, (dd|ps) 1.17 -> 0.10.  Lanes per ket and the
// three-product form on top: (ss|ss) 0.73 -> 0.23 ms, (pp|ps) 0.88 -> 0.28, (dp|ps) 0.61 -> 0.20.  Parts of
// up to 81 components spilled ((pp|pp) 0.20 ms as one, (dp|pp) 0.40 as two).
constexpr int kGradLaneBlock = 128;

// What the per-lane kernels take by value (see GradLaunch).
struct GradArgs {
    const int2* segs;
    const PairRec* bra;
    KetPairs kpairs;
    KetPrims<double> kprims;
    const double* kea;
    const PrimPair<double>* pp;
    const double *rys, *D;
    double* grad;
    double xfac;
    int nbf, natom, diag;
};

__device__ __forceinline__ PairRec grad_ket(const KetPairs& k, int kq, const int4 km) {
    PairRec Q;
    Q.bfa = km.x & kKetBfMask;
    Q.bfb = (km.x >> kKetBfBits) & kKetBfMask;
    Q.npp = km.y;
    const double2 c0 = k.cen[kq], c1 = k.cen[k.np + kq], c2 = k.cen[2 * k.np + kq];
    Q.ax = c0.x, Q.ay = c0.y, Q.az = c1.x, Q.abx = c1.y, Q.aby = c2.x, Q.abz = c2.y;
    return Q;
}

// Components [A0, A0 + NAS) of shell a only: the gradient is linear in the components.
template <int LA, int LB, int LC, int LD, int A0, int NAS>
struct GradPart {
    using S = EriShape<LA, LB, LC, LD>;
    static constexpr int NQ = NAS * S::NB * S::NCD;
    static constexpr int N = (LA + LB + LC + LD + 1) / 2 + 1;
    // 1-D tables with the first and third power raised by one: index ((i (LB+1) + j) (LC+2) + k) (LD+1) + l
    static constexpr int sK = LD + 1, sJ = (LC + 2) * sK, sI = (LB + 1) * sJ;
    static constexpr int HE = (LA + 2) * sI;
    static constexpr int kTab = N <= 3 ? rys_tab_size<N>() : 1;  // Rys coefficients staged in LDS
};

// Per axis x: the part's components ordered by their 1-D index on that axis (first entry o[x][m]), with the
// extended-table indices ey, ez of the other two axes, and whether a component is the last of its index.
template <int LA, int LB, int LC, int LD, int A0, int NAS>
struct GradOrder {
    using S = EriShape<LA, LB, LC, LD>;
    using G = GradPart<LA, LB, LC, LD, A0, NAS>;
    int n[3][G::NQ], e[3][G::NQ], ey[3][G::NQ], ez[3][G::NQ], ia[3][G::NQ], ib[3][G::NQ], ic[3][G::NQ];
    bool last[3][G::NQ];
    constexpr GradOrder() : n(), e(), ey(), ez(), ia(), ib(), ic(), last() {
        int idx[3][G::NQ] = {}, p[3][3][G::NQ] = {};
        for (int k = 0; k < G::NQ; ++k) {
            const int d = k % S::ND, c = k / S::ND % S::NC, b = k / S::NCD % S::NB, a = A0 + k / (S::NCD * S::NB);
            const int pa[3] = {cart_x(LA, a), cart_y(LA, a), cart_z(LA, a)}, pb[3] = {cart_x(LB, b), cart_y(LB, b), cart_z(LB, b)};
            const int pc[3] = {cart_x(LC, c), cart_y(LC, c), cart_z(LC, c)}, pd[3] = {cart_x(LD, d), cart_y(LD, d), cart_z(LD, d)};
            for (int y = 0; y < 3; ++y) {
                p[y][0][k] = pa[y], p[y][1][k] = pb[y], p[y][2][k] = pc[y];
                idx[y][k] = pa[y] * G::sI + pb[y] * G::sJ + pc[y] * G::sK + pd[y];
            }
        }
        for (int x = 0; x < 3; ++x) {
            int m = 0;
            for (int h = 0; h < G::HE; ++h) {
                const int m0 = m;
                for (int k = 0; k < G::NQ; ++k)
                    if (idx[x][k] == h) {
                        n[x][m] = k, e[x][m] = h, ey[x][m] = idx[(x + 1) % 3][k], ez[x][m] = idx[(x + 2) % 3][k];
                        ia[x][m] = p[x][0][k], ib[x][m] = p[x][1][k], ic[x][m] = p[x][2][k], last[x][m] = false;
                        ++m;
                    }
                if (m > m0) last[x][m - 1] = true;
            }
        }
    }
};
template <int LA, int LB, int LC, int LD, int A0, int NAS>
inline constexpr GradOrder<LA, LB, LC, LD, A0, NAS> kGradOrder{};

// gq += the nine derivative sums (A, B, C x xyz) of the quartet (P|Q) with density weights W, over the
// ket primitives sub, sub + lanes, ...
template <int LA, int LB, int LC, int LD, int A0, int NAS>
__device__ __forceinline__ void grad_quartet_lane(const PairRec& P, const PairRec& Q, const GradArgs& ga, int kp0,
                                                  int kstride, int sub, int lanes, const double* __restrict__ rys_n,
                                                  const double* W, double* gq) {
    using S = EriShape<LA, LB, LC, LD>;
    using G = GradPart<LA, LB, LC, LD, A0, NAS>;
    constexpr int N = G::N, sI = G::sI, sJ = G::sJ, sK = G::sK;
    const double two_pi_52 = 2.0 * kPi * kPi * 1.7724538509055160273;
    const double AB[3] = {P.abx, P.aby, P.abz}, CD[3] = {Q.abx, Q.aby, Q.abz};
    const PrimPair<double>* ppb = ga.pp + P.pp_off;
    for (int j = sub; j < Q.npp; j += lanes) {
        const PrimPair<double> c = ga.kprims.at(kp0 + j * kstride);
        const double q = c.p, hq = c.hp, two_c = 2.0 * ga.kea[kp0 + j * kstride];
        const double QC[3] = {c.px - Q.ax, c.py - Q.ay, c.pz - Q.az};
        for (int i = 0; i < P.npp; ++i) {
            const PrimPair<double> a = ppb[i];
            const double keep = a.kab * c.kab < kPrimScreen ? 0.0 : 1.0;  // the primitive screen as a factor
            const double p = a.p, hp = a.hp, two_a = 2.0 * a.ea, two_b = 2.0 * (a.p - a.ea);
            const double rs = qrsqrt(p + q), ipq = rs * rs;
            const double PQ[3] = {a.px - c.px, a.py - c.py, a.pz - c.pz};
            const double T = p * q * ipq * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
            const double pref = two_pi_52 * rs * a.ckp * c.ckp * keep;
            const double PA[3] = {a.px - P.ax, a.py - P.ay, a.pz - P.az};
            const double qf = q * ipq, pf = p * ipq;
            // one node at a time (its fit evaluated in the loop): the body is long enough, and N copies
            // of it only fill the instruction cache
#pragma unroll 1
            for (int r = 0; r < N; ++r) {
                double u, w;
                rys_eval_node<double, N>(T, rys_n, r, u, w);
                const double b00 = 0.5 * u * ipq, b10 = hp * (1.0 - u * qf), b01 = hq * (1.0 - u * pf);
                double I[3][G::HE];
#pragma unroll
                for (int x = 0; x < 3; ++x) {
                    double g[(LA + LB + 2) * (LC + LD + 2)];
                    vrr2d<LA + LB + 1, LC + LD + 1, double>(g, PA[x] - u * qf * PQ[x], QC[x] + u * pf * PQ[x], b00, b10, b01);
                    hrr1d<LA + 1, LB, LC + 1, LD, double>(g, AB[x], CD[x], I[x]);
                }
                const double wp = w * pref;
                static_for<3>([&](auto xc) {
                    constexpr int x = decltype(xc)::value, y = (x + 1) % 3, z = (x + 2) % 3;
                    double s0 = 0.0, sAp = 0.0, sAm = 0.0, sBm = 0.0, sCp = 0.0, sCm = 0.0, cs = 0.0;
                    static_for<G::NQ>([&](auto mc) {
                        constexpr int m = decltype(mc)::value;
                        constexpr const auto& o = kGradOrder<LA, LB, LC, LD, A0, NAS>;
                        constexpr int kn = o.n[x][m], ey = o.ey[x][m], ez = o.ez[x][m];
                        cs += W[kn] * (I[y][ey] * I[z][ez]);
                        if constexpr (o.last[x][m]) {
                            constexpr int e = o.e[x][m], ia = o.ia[x][m], ib = o.ib[x][m], ic = o.ic[x][m];
                            s0 += cs * I[x][e];
                            sAp += cs * I[x][e + sI];
                            sCp += cs * I[x][e + sK];
                            if constexpr (ia > 0) sAm += (double)ia * cs * I[x][e - sI];
                            if constexpr (ib > 0) sBm += (double)ib * cs * I[x][e - sJ];
                            if constexpr (ic > 0) sCm += (double)ic * cs * I[x][e - sK];
                            cs = 0.0;
                        }
                    });
                    gq[x] += wp * (two_a * sAp - sAm);
                    gq[3 + x] += wp * (two_b * (sAp + AB[x] * s0) - sBm);
                    gq[6 + x] += wp * (two_c * sCp - sCm);
                });
            }
        }
    }
}

template <int LA, int LB, int LC, int LD, int A0, int NAS>
__global__ __launch_bounds__(kGradLaneBlock) void grad_lane_kernel(const int4* __restrict__ items, const GradArgs ga) {
    using S = EriShape<LA, LB, LC, LD>;
    using G = GradPart<LA, LB, LC, LD, A0, NAS>;
    __shared__ double rys_s[G::kTab];
    extern __shared__ double gl[];  // natom x 3: the block's sums
    const int tid = threadIdx.x, natom = ga.natom;
    const double* rys_n = ga.rys + qcg_rys_off[G::N];
    if constexpr (G::N <= 3) {
        for (int i = tid; i < G::kTab; i += blockDim.x) rys_s[i] = rys_n[i];
        rys_n = rys_s;
    }
    for (int i = tid; i < 3 * natom; i += blockDim.x) gl[i] = 0.0;
    __syncthreads();
    const size_t nbf = (size_t)ga.nbf;
    const double* __restrict__ D = ga.D;
    const int4 it = items[blockIdx.x];
    const PairRec P = item_bra(ga.bra, it);
    const int lg = item_lg(it), lanes = 1 << lg, sub = tid & (lanes - 1), step = blockDim.x >> lg;
    double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};
    KetCursor cur{ga.segs, it.y, it.z + (tid >> lg)};
    for (int j = tid >> lg; j < item_kets(it); j += step, cur.r += step) {
        const int q = cur.at();
        const int4 km = ga.kpairs.meta[q];
        const PairRec Q = grad_ket(ga.kpairs, q, km);
        const double deg = ((P.sa == P.sb) ? 0.5 : 1.0) * ((km.x & kKetSame) ? 0.5 : 1.0) * ((ga.diag && q == P.pos) ? 0.5 : 1.0);
        double W[G::NQ];
        static_for<G::NQ>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            constexpr int d = k % S::ND, c = (k / S::ND) % S::NC, b = (k / S::NCD) % S::NB, a = A0 + k / (S::NCD * S::NB);
            const size_t i_ = P.bfa + a, j_ = P.bfb + b, k_ = Q.bfa + c, l_ = Q.bfb + d;
            W[k] = 4.0 * deg *
                   (D[i_ * nbf + j_] * D[k_ * nbf + l_] - ga.xfac * (D[i_ * nbf + k_] * D[j_ * nbf + l_] + D[i_ * nbf + l_] * D[j_ * nbf + k_])) *
                   (cnorm(LA, a) * cnorm(LB, b) * cnorm(LC, c) * cnorm(LD, d));
        });
        double gq[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
        grad_quartet_lane<LA, LB, LC, LD, A0, NAS>(P, Q, ga, km.z, km.w, sub, lanes, rys_n, W, gq);
        const int2 at = ga.kpairs.atoms[q];
#pragma unroll
        for (int x = 0; x < 3; ++x) {
            gA[x] += gq[x];
            gB[x] += gq[3 + x];
            atomicAdd(&gl[3 * at.x + x], gq[6 + x]);
            atomicAdd(&gl[3 * at.y + x], -(gq[x] + gq[3 + x] + gq[6 + x]));  // centre D
        }
    }
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        const double ax = wave_sum(gA[x]), bx = wave_sum(gB[x]);
        if ((tid & 63) == 0) {
            atomicAdd(&gl[3 * P.atom_a + x], ax);
            atomicAdd(&gl[3 * P.atom_b + x], bx);
        }
    }
    __syncthreads();
    for (int i = tid; i < 3 * natom; i += blockDim.x)
        if (gl[i] != 0.0) atomicAdd(&ga.grad[i], gl[i]);
}

#define QCG_LA(c) ((c) == 0 ? 0 : (c) <= 2 ? 1 : 2)
#define QCG_LB(c) ((c) == 0 || (c) == 1 || (c) == 3 ? 0 : ((c) == 2 || (c) == 4) ? 1 : 2)

// One launch per part of the first shell's components.
template <int LA, int LB, int LC, int LD, int NAS, int A0 = 0>
static hipError_t launch_grad_parts(const GradLaunch& a, const GradArgs& ga, hipStream_t st) {
    hipLaunchKernelGGL((grad_lane_kernel<LA, LB, LC, LD, A0, NAS>), dim3(a.nitems), dim3(kGradLaneBlock),
                       3 * (size_t)a.natom * sizeof(double), st, a.items, ga);
    const hipError_t e = hipGetLastError();
    if constexpr (A0 + NAS < ncart(LA))
        return e != hipSuccess ? e : launch_grad_parts<LA, LB, LC, LD, NAS, A0 + NAS>(a, ga, st);
    else
        return e;
}

template <int CB, int CK>
static hipError_t launch_grad_t(const GradLaunch& a, hipStream_t st) {
    constexpr int LA = QCG_LA(CB), LB = QCG_LB(CB), LC = QCG_LA(CK), LD = QCG_LB(CK);
    using G = GradWave<LA, LB, LC, LD>;
    if (a.nitems <= 0) return hipSuccess;
    constexpr int NAS = grad_part(CB, CK);
    if constexpr (NAS > 0) {
        const GradArgs ga{a.segs, a.bra, a.kpairs, a.kprims, a.kea, a.pp, a.rys, a.D, a.grad, a.xfac, a.nbf, a.natom, a.diag};
        return launch_grad_parts<LA, LB, LC, LD, NAS>(a, ga, st);
    } else {
        hipLaunchKernelGGL((grad_wave_kernel<LA, LB, LC, LD>), dim3((a.nitems + G::WPB - 1) / G::WPB),
                           dim3(64 * G::WPB), 0, st, a.items, a.segs, a.nitems, a.bra, a.ket, a.diag, a.pp, a.rys, a.D, a.nbf,
                           a.xfac, a.grad);
    }
    return hipGetLastError();
}

#define QCG_CAT2(a, b) a##b
#define QCG_CAT(a, b) QCG_CAT2(a, b)

hipError_t QCG_CAT(launch_grad_cb, QCG_CB)(int ck, const GradLaunch& a, hipStream_t st) {
    switch (ck) {
#define QCG_K(CK) \
    case CK: if constexpr (CK <= QCG_CB) return launch_grad_t<QCG_CB, CK>(a, st); break;
        QCG_K(0) QCG_K(1) QCG_K(2) QCG_K(3) QCG_K(4) QCG_K(5)
#undef QCG_K
    }
    return hipErrorInvalidValue;
}

}  // namespace qcg
