// Direct J/K build and compressed-tensor kernels for all quartet classes whose bra pair class
// is QCG_CB (this file is compiled once per bra class, -DQCG_CB=0..5, so the six units build
// in parallel).  Pair class c <-> (la, lb): 0 (s,s) 1 (p,s) 2 (p,p) 3 (d,s) 4 (d,p) 5 (d,d).
//
// Work decomposition of the J/K build (one launch per quartet class, bra class >= ket class):
//   * pairs of a class are ordered by contraction bucket (number of primitive pairs), then by
//     Schwarz bound (descending); for a bra pair P the surviving kets of a bucket are the prefix
//     with Q_P*Q_Q >= threshold (monotone product), found by binary search on exactly the product
//     the reference tests (q_ij * q_kl < SCHWARZ_THRESHOLD, integrals/eri/mod.rs:1008-1023); for
//     bra class == ket class only kets at or before P (each unordered pair-pair once = 8-fold
//     symmetry); in mixed precision each prefix splits into an FP64 range (Q_P*Q_Q >= cutoff) and
//     an FP32 range;
//   * the host cuts every range into work items (bra pair, ket sub-range) of a per-class size;
//     one block per item, one thread per ket (several for cheap classes), so every class
//     launch has many more blocks than the GPU has CUs;
//   * digestion: J_P in registers + wave reduction; J_Q by fixed-point atomics on arrays ordered by
//     ket pair, so a wavefront's adds are consecutive; the four K terms all land in the rows of the
//     bra functions, so they are summed in LDS rows (one block = one bra pair) and flushed with one
//     global atomic per touched element at the end of the block (device atomics are performed
//     memory-side on this GPU, so every global atomic is HBM write traffic).  J is gathered from the
//     pair-ordered sums, K = Kacc + Kacc^T after.
//   * symmetry factors: 1/2 for a == b shells, 1/2 for c == d shells, 1/2 for P == Q, folded
//     together with the component normalisation into the density sub-blocks.
// With the symmetric density this reproduces build_fock's G = J - K/2 (scf/mod.rs:825-881) and
// build_jk (dft/ks_scf.rs:1369-1394).
#include "eri_device.h"
#include "eri_launch.h"
#include "eri_wave.h"

#ifndef QCG_CB
#error "compile with -DQCG_CB=<bra pair class>"
#endif
namespace qcg {

// What every J/K kernel of a class takes by value (see JkLaunch).
struct JkArgs {
    const int2* segs;
    const PairRec* bra;
    const PairRec* ket;
    KetPairs kpairs;
    const double *D, *Dp, *fix;
    fix_t *Jacc, *Jmat, *Kacc;
    const int* ket_off;
    const int64_t* mat_off;
    const int* mol_nbf;
    int diag, do_j, do_k, jb_bra, jb_ket, np_bra, np_ket;
};

// The Rys coefficients of order N for a block: staged in LDS (lds, at least rys_tab_size<N>()
// elements) when N <= 3, where the per-lane kernels gather them at lane-dependent intervals once
// per primitive quartet, else read from device memory.  The caller's __syncthreads() follows.
template <typename R, int N>
__device__ __forceinline__ const R* rys_stage(const R* __restrict__ rys_tab, R* lds) {
    if constexpr (N <= 3) {
        for (int i = threadIdx.x; i < rys_tab_size<N>(); i += blockDim.x) lds[i] = rys_tab[qcg_rys_off[N] + i];
        return lds;
    } else {
        return rys_tab + qcg_rys_off[N];
    }
}
template <int N>
constexpr int rys_lds_doubles() { return N <= 3 ? rys_tab_size<N>() : 1; }

// Ket kq of a class (km = its meta word): the fields that the class needs.
template <int LC, int LD>
__device__ __forceinline__ PairRec ket_pair(const KetPairs& k, int kq, const int4 km) {
    PairRec Q;
    Q.bfa = km.x & kKetBfMask;
    Q.bfb = (km.x >> kKetBfBits) & kKetBfMask;
    Q.npp = km.y;
    if constexpr (LC > 0) {
        const double2 c0 = k.cen[kq], c1 = k.cen[k.np + kq];
        Q.ax = c0.x, Q.ay = c0.y, Q.az = c1.x, Q.abx = c1.y;
        if constexpr (LD > 0) {
            const double2 c2 = k.cen[2 * k.np + kq];
            Q.aby = c2.x, Q.abz = c2.y;
        }
    }
    return Q;
}

// One work item = (bra pair, run of its surviving kets over the ket segments, KetCursor); the
// host builds the items with the exact screening predicate, so no quartet is tested twice or
// skipped.  rys_n: the coefficients of this class's Rys order (rys_stage); rows: with KROWS, LDS room
// for the K rows of the bra functions a and b ((NA + NB) x nbf fixed-point words, fixacc.h), in which
// the four K terms of the item, all in the rows of a and b, are summed and then flushed once per
// block.  J and K go to the fixed-point accumulators Jacc (by shell pair) and Kacc with the scales
// fix[4 mol], fix[4 mol + 1], so the result does not depend on the order in which blocks and lanes
// arrive.  The bra's primitive pairs are uniform over the block and come through the scalar cache;
// the D rows of K through the vector caches.  A0, NA: the components of the first shell taken (jk_part);
// J_Q, and the K terms in the rows of b, are sums over the parts, which the accumulators make of them.
template <int LA, int LB, int LC, int LD, typename R, bool KROWS, int A0, int NA>
__device__ __forceinline__ void jk_item(const int4 it, const JkArgs& g, const KetPrims<R>& kprims,
                                        const PrimPair<R>* __restrict__ pp, const R* __restrict__ rys_n, double* rows) {
    using S = EriShape<LA, LB, LC, LD>;
    constexpr int NAB = NA * S::NB, NQ = NAB * S::NCD, NR = NA + S::NB;
    PairRec P = item_bra(g.bra, it);
    P.bfa += A0;  // the part's components are functions bfa .. bfa + NA - 1 from here on
    const int pidx = P.pos, ket0 = g.ket_off[P.mol];
    const double* __restrict__ D = g.D + g.mat_off[P.mol];
    fix_t* __restrict__ Jacc = g.Jacc;
    fix_t* __restrict__ Kacc = g.Kacc + g.mat_off[P.mol];
    const int nbf = g.mol_nbf[P.mol], do_j = g.do_j, do_k = g.do_k;
    const double sJ = g.fix[4 * P.mol], sK = g.fix[4 * P.mol + 1];  // fixed-point scales of J and K
    const int tid = threadIdx.x;
    const PrimPair<R>* ppb = pp + P.pp_off;
    const int nrow = NR * nbf;
    fix_t* kl = reinterpret_cast<fix_t*>(rows);
    if constexpr (KROWS)
        for (int i = tid; i < nrow; i += blockDim.x) kl[i] = 0;
    __syncthreads();
    // D element (row function a + r of the bra's shell a, or b + r of shell b; column col)
    auto drow = [&](bool row_b, int r, int col) -> double { return D[(size_t)((row_b ? P.bfb : P.bfa) + r) * nbf + col]; };
    auto kadd = [&](bool row_b, int r, int col, double v) {
        if constexpr (KROWS) fix_add_lds(kl, (row_b ? NA + r : r) * nbf + col, v, sK);
        else fix_add_global(Kacc, (size_t)((row_b ? P.bfb : P.bfa) + r) * nbf + col, v, sK);
    };

    // bra density block scaled by the bra component norms
    double Dps[NAB], jp[NAB];
    for_n<NAB>([&](int ab) {
        const int a = ab / S::NB, b = ab % S::NB;
        Dps[ab] = drow(false, a, P.bfb + b) * cnorm(LA, A0 + a) * cnorm(LB, b);
        jp[ab] = 0.0;
    });
    const double deg_p = (P.sa == P.sb) ? 0.5 : 1.0;

    // 2^lg lanes share a ket (uniform over the block): lane `sub` of them takes every 2^lg-th ket
    // primitive and a fixed butterfly sums the partial quartets, so a heavily contracted quartet is
    // no longer one lane's serial chain (alone, water (ss|ss) 335 -> 21 us, (pp|pp) 231 -> 50 us)
    const int lg = item_lg(it), lanes = 1 << lg, sub = tid & (lanes - 1), step = blockDim.x >> lg;
    KetCursor cur{g.segs, it.y, it.z + (tid >> lg)};
    for (int j = tid >> lg; j < item_kets(it); j += step, cur.r += step) {
        const int q = cur.at(), kq = ket0 + q;
        const int4 km = g.kpairs.meta[kq];
        const PairRec Q = ket_pair<LC, LD>(g.kpairs, kq, km);
        const int kstride = km.w;
        R eri[NQ];
        for_n<NQ>([&](int i) { eri[i] = R(0); });
        contract_quartet_pp<LA, LB, LC, LD, R, true, A0 * S::NB * S::NCD, NQ>(
            P, Q, ppb, [&](int i) { return kprims.at(km.z + i * kstride); }, rys_n, eri, sub, lanes);
        if (lg) {
            for (int off = 1; off < lanes; off <<= 1)
                for_n<NQ>([&](int i) { eri[i] += __shfl_xor(eri[i], off, 64); });
            if (sub) continue;  // the group's first lane digests
        }
        const double deg = deg_p * ((km.x & kKetSame) ? 0.5 : 1.0) * ((g.diag && q == pidx) ? 0.5 : 1.0);
        if (do_j) {
            double Dqs[S::NCD];
            for_n<S::NCD>([&](int cd) { Dqs[cd] = g.Dp[g.jb_ket + cd * g.np_ket + kq]; });
            const double fj = 2.0 * deg;
            for_n<NAB>([&](int ab) {
                double s = 0.0;
                for_n<S::NCD>([&](int cd) { s += Dqs[cd] * (double)eri[ab * S::NCD + cd]; });
                const int a = ab / S::NB, b = ab % S::NB;
                jp[ab] += fj * cnorm(LA, A0 + a) * cnorm(LB, b) * s;
            });
            for_n<S::NCD>([&](int cd) {
                double s = 0.0;
                for_n<NAB>([&](int ab) { s += Dps[ab] * (double)eri[ab * S::NCD + cd]; });
                const int c = cd / S::ND, d = cd % S::ND;
                fix_add_global(Jacc, g.jb_ket + cd * g.np_ket + kq, fj * cnorm(LC, c) * cnorm(LD, d) * s, sJ);
            });
        }
        if (do_k) {
            // Kacc_ik += D_jl v, Kacc_jk += D_il v, Kacc_il += D_jk v, Kacc_jl += D_ik v
            // (i in a, j in b, k in c, l in d); every D sub-block pre-scaled by the norms it sums over.
            double Dbd[S::NB * S::ND], Dad[NA * S::ND], Dbc[S::NB * S::NC], Dac[NA * S::NC];
            for_n<S::NB * S::ND>([&](int i) {
                const int b = i / S::ND, d = i % S::ND;
                Dbd[i] = drow(true, b, Q.bfb + d) * cnorm(LB, b) * cnorm(LD, d);
            });
            for_n<NA * S::ND>([&](int i) {
                const int a = i / S::ND, d = i % S::ND;
                Dad[i] = drow(false, a, Q.bfb + d) * cnorm(LA, A0 + a) * cnorm(LD, d);
            });
            for_n<S::NB * S::NC>([&](int i) {
                const int b = i / S::NC, c = i % S::NC;
                Dbc[i] = drow(true, b, Q.bfa + c) * cnorm(LB, b) * cnorm(LC, c);
            });
            for_n<NA * S::NC>([&](int i) {
                const int a = i / S::NC, c = i % S::NC;
                Dac[i] = drow(false, a, Q.bfa + c) * cnorm(LA, A0 + a) * cnorm(LC, c);
            });
#define VIDX(a, b, c, d) ((((a) * S::NB + (b)) * S::NC + (c)) * S::ND + (d))
            for_n<NA * S::NC>([&](int ac) {
                const int a = ac / S::NC, c = ac % S::NC;
                double s = 0.0;
                for_n<S::NB * S::ND>([&](int bd) {
                    const int b = bd / S::ND, d = bd % S::ND;
                    s += Dbd[bd] * (double)eri[VIDX(a, b, c, d)];
                });
                kadd(false, a, Q.bfa + c, deg * cnorm(LA, A0 + a) * cnorm(LC, c) * s);
            });
            for_n<S::NB * S::NC>([&](int bc) {
                const int b = bc / S::NC, c = bc % S::NC;
                double s = 0.0;
                for_n<NA * S::ND>([&](int ad) {
                    const int a = ad / S::ND, d = ad % S::ND;
                    s += Dad[ad] * (double)eri[VIDX(a, b, c, d)];
                });
                kadd(true, b, Q.bfa + c, deg * cnorm(LB, b) * cnorm(LC, c) * s);
            });
            for_n<NA * S::ND>([&](int ad) {
                const int a = ad / S::ND, d = ad % S::ND;
                double s = 0.0;
                for_n<S::NB * S::NC>([&](int bc) {
                    const int b = bc / S::NC, c = bc % S::NC;
                    s += Dbc[bc] * (double)eri[VIDX(a, b, c, d)];
                });
                kadd(false, a, Q.bfb + d, deg * cnorm(LA, A0 + a) * cnorm(LD, d) * s);
            });
            for_n<S::NB * S::ND>([&](int bd) {
                const int b = bd / S::ND, d = bd % S::ND;
                double s = 0.0;
                for_n<NA * S::NC>([&](int ac) {
                    const int a = ac / S::NC, c = ac % S::NC;
                    s += Dac[ac] * (double)eri[VIDX(a, b, c, d)];
                });
                kadd(true, b, Q.bfb + d, deg * cnorm(LB, b) * cnorm(LD, d) * s);
            });
#undef VIDX
        }
    }
    // J_P: wave reduction (a fixed shuffle tree), one fixed-point add per component per wave
    if (do_j) {
        for_n<NAB>([&](int ab) {
            double s = jp[ab];
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
            if ((tid & 63) == 0 && s != 0.0) fix_add_global(Jacc, g.jb_bra + (A0 * S::NB + ab) * g.np_bra + it.x, s, sJ);
        });
    }
    if constexpr (KROWS) {
        __syncthreads();
        for (int i = tid; i < nrow; i += blockDim.x) {
            const int r = i / nbf, col = i - r * nbf;
            const int row = r < NA ? P.bfa + r : P.bfb + (r - NA);
            fix_add_word_global(Kacc, (size_t)row * nbf + col, kl[i]);
        }
    }
}

template <int LA, int LB, int LC, int LD, typename R, bool KROWS, int A0, int NAS>
__global__ __launch_bounds__(256) void jk_kernel(const int4* __restrict__ items, const JkArgs g, const KetPrims<R> kprims,
                                                 const PrimPair<R>* __restrict__ pp, const R* __restrict__ rys_tab) {
    constexpr int NR = EriShape<LA, LB, LC, LD>::NROOTS;
    extern __shared__ double rows[];
    __shared__ double rys_raw[rys_lds_doubles<NR>()];
    const R* rys_n = rys_stage<R, NR>(rys_tab, reinterpret_cast<R*>(rys_raw));
    jk_item<LA, LB, LC, LD, R, KROWS, A0, NAS>(items[blockIdx.x], g, kprims, pp, rys_n, rows);
}

// Mixed precision in one launch: items [0, n64) are FP64 quartets, the rest FP32 (one branch per
// block); saves the second launch per class and its tail.
template <int LA, int LB, int LC, int LD, bool KROWS, int A0, int NAS>
__global__ __launch_bounds__(256) void jk_kernel_mp(const int4* __restrict__ items, int n64, const JkArgs g,
                                                    const KetPrims<double> kprims, const KetPrims<float> kprimsf,
                                                    const PrimPair<double>* __restrict__ pp,
                                                    const PrimPair<float>* __restrict__ ppf,
                                                    const double* __restrict__ rys_tab,
                                                    const float* __restrict__ rys_tabf) {
    constexpr int NR = EriShape<LA, LB, LC, LD>::NROOTS;
    extern __shared__ double rows[];
    __shared__ double rys_raw[rys_lds_doubles<NR>()];
    if ((int)blockIdx.x < n64) {
        const double* rys_n = rys_stage<double, NR>(rys_tab, rys_raw);
        jk_item<LA, LB, LC, LD, double, KROWS, A0, NAS>(items[blockIdx.x], g, kprims, pp, rys_n, rows);
    } else {
        const float* rys_n = rys_stage<float, NR>(rys_tabf, reinterpret_cast<float*>(rys_raw));
        jk_item<LA, LB, LC, LD, float, KROWS, A0, NAS>(items[blockIdx.x], g, kprimsf, ppf, rys_n, rows);
    }
}

// Wave-cooperative J/K for the classes with many components (eri_wave.h): four wavefronts per
// block, each takes one work item (bra pair, ket range) and walks its kets one quartet at a time.
// Digestion of a contracted quartet (phase C): the quartet v (norms and symmetry factor applied)
// goes to LDS, lanes over output elements form
//   J_ab += 2 sum_cd D_cd v   (kept in a register of lane ab until the item ends),
//   J_cd += 2 sum_ab D_ab v,  K_ac += sum_bd D_bd v,  K_bc += sum_ad D_ad v,
//   K_ad += sum_bc D_bc v,    K_bd += sum_ac D_ac v   (FP64 atomics per quartet).
template <int LA, int LB, int LC, int LD, typename R>
struct JkWave {
    using S = EriShape<LA, LB, LC, LD>;
    using T = WaveTable<LA, LB, LC, LD, S::NROOTS, R>;
    static constexpr int VD = T::DOUBLES > S::NQ ? T::DOUBLES : S::NQ;  // table, then the quartet
    static constexpr int DB = S::NAB + S::NCD + S::NB * S::ND + S::NA * S::ND + S::NB * S::NC + S::NA * S::NC;
    static constexpr int WAVE_D = VD + DB;
    static constexpr int KPL = (S::NQ + 63) / 64;
    static constexpr bool kEnabled = S::NQ >= 27;
};

// One work item on one wavefront; V: the wave's LDS region (JkWave<..., R>::WAVE_D doubles).
template <int LA, int LB, int LC, int LD, typename R>
__device__ __forceinline__ void jk_wave_item(
    const int4 it, int lane, double* V, const JkArgs& g, const PrimPair<R>* __restrict__ pp, const R* __restrict__ rys_tab) {
    using S = EriShape<LA, LB, LC, LD>;
    using W = JkWave<LA, LB, LC, LD, R>;
    constexpr int KPL = W::KPL;
    constexpr int NA = S::NA, NB = S::NB, NC = S::NC, ND = S::ND, NCD = S::NCD;
    double* Dab = V + W::VD;
    double* Dcd = Dab + S::NAB;
    double* Dbd = Dcd + NCD;
    double* Dad = Dbd + NB * ND;
    double* Dbc = Dad + NA * ND;
    double* Dac = Dbc + NB * NC;

    const PairRec P = item_bra(g.bra, it);
    const int pidx = P.pos;
    const PairRec* __restrict__ ket = g.ket + g.ket_off[P.mol];
    const double* __restrict__ D = g.D + g.mat_off[P.mol];
    fix_t* __restrict__ Jmat = g.Jmat + g.mat_off[P.mol];
    fix_t* __restrict__ Kacc = g.Kacc + g.mat_off[P.mol];
    const size_t nbf = (size_t)g.mol_nbf[P.mol];
    const int do_j = g.do_j, do_k = g.do_k;
    const double sJ = g.fix[4 * P.mol], sK = g.fix[4 * P.mol + 1];  // fixed-point scales of J and K

    for (int o = lane; o < S::NAB; o += 64) Dab[o] = D[(P.bfa + o / NB) * nbf + P.bfb + o % NB];
    double jp = 0.0;  // J_ab of lane ab over the item's kets
    const double deg_p = (P.sa == P.sb) ? 0.5 : 1.0;

    KetCursor cur{g.segs, it.y, it.z};
    for (int j = 0; j < item_kets(it); ++j, ++cur.r) {
        const int q = cur.at();
        const PairRec Q = ket[q];
        R acc[KPL];
        wave_quartet<LA, LB, LC, LD, R>(P, Q, pp, rys_tab, V, lane, acc);
        wave_sync();
        const double deg = deg_p * ((Q.sa == Q.sb) ? 0.5 : 1.0) * ((g.diag && q == pidx) ? 0.5 : 1.0);
#pragma unroll
        for (int j = 0; j < KPL; ++j) {
            const int k = lane + 64 * j;
            if (k < S::NQ) {
                const int d = k % ND, c = (k / ND) % NC, b = (k / NCD) % NB, a = k / (NCD * NB);
                V[k] = (double)acc[j] * (cnorm(LA, a) * cnorm(LB, b) * cnorm(LC, c) * cnorm(LD, d) * deg);
            }
        }
        if (do_j)
            for (int o = lane; o < NCD; o += 64) Dcd[o] = D[(Q.bfa + o / ND) * nbf + Q.bfb + o % ND];
        if (do_k) {
            for (int o = lane; o < NB * ND; o += 64) Dbd[o] = D[(P.bfb + o / ND) * nbf + Q.bfb + o % ND];
            for (int o = lane; o < NA * ND; o += 64) Dad[o] = D[(P.bfa + o / ND) * nbf + Q.bfb + o % ND];
            for (int o = lane; o < NB * NC; o += 64) Dbc[o] = D[(P.bfb + o / NC) * nbf + Q.bfa + o % NC];
            for (int o = lane; o < NA * NC; o += 64) Dac[o] = D[(P.bfa + o / NC) * nbf + Q.bfa + o % NC];
        }
        wave_sync();
#define VAT(a, b, c, d) V[(((a) * NB + (b)) * NC + (c)) * ND + (d)]
        if (do_j) {
            if (lane < S::NAB) {
                double s = 0.0;
                for (int cd = 0; cd < NCD; ++cd) s += Dcd[cd] * V[lane * NCD + cd];
                jp += 2.0 * s;
            }
            for (int o = lane; o < NCD; o += 64) {
                double s = 0.0;
                for (int ab = 0; ab < S::NAB; ++ab) s += Dab[ab] * V[ab * NCD + o];
                fix_add_global(Jmat, (Q.bfa + o / ND) * nbf + Q.bfb + o % ND, 2.0 * s, sJ);
            }
        }
        if (do_k) {
            for (int o = lane; o < NA * NC; o += 64) {
                const int a = o / NC, c = o % NC;
                double s = 0.0;
                for (int b = 0; b < NB; ++b)
                    for (int d = 0; d < ND; ++d) s += Dbd[b * ND + d] * VAT(a, b, c, d);
                fix_add_global(Kacc, (P.bfa + a) * nbf + Q.bfa + c, s, sK);
            }
            for (int o = lane; o < NB * NC; o += 64) {
                const int b = o / NC, c = o % NC;
                double s = 0.0;
                for (int a = 0; a < NA; ++a)
                    for (int d = 0; d < ND; ++d) s += Dad[a * ND + d] * VAT(a, b, c, d);
                fix_add_global(Kacc, (P.bfb + b) * nbf + Q.bfa + c, s, sK);
            }
            for (int o = lane; o < NA * ND; o += 64) {
                const int a = o / ND, d = o % ND;
                double s = 0.0;
                for (int b = 0; b < NB; ++b)
                    for (int c = 0; c < NC; ++c) s += Dbc[b * NC + c] * VAT(a, b, c, d);
                fix_add_global(Kacc, (P.bfa + a) * nbf + Q.bfb + d, s, sK);
            }
            for (int o = lane; o < NB * ND; o += 64) {
                const int b = o / ND, d = o % ND;
                double s = 0.0;
                for (int a = 0; a < NA; ++a)
                    for (int c = 0; c < NC; ++c) s += Dac[a * NC + c] * VAT(a, b, c, d);
                fix_add_global(Kacc, (P.bfb + b) * nbf + Q.bfb + d, s, sK);
            }
        }
#undef VAT
    }
    if (do_j && lane < S::NAB && jp != 0.0) fix_add_global(Jmat, (P.bfa + lane / NB) * nbf + P.bfb + lane % NB, jp, sJ);
}

template <int LA, int LB, int LC, int LD, typename R>
__global__ __launch_bounds__(256) void jk_wave_kernel(const int4* __restrict__ items, int nitems, const JkArgs g,
                                                      const PrimPair<R>* __restrict__ pp, const R* __restrict__ rys_tab) {
    constexpr int WD = JkWave<LA, LB, LC, LD, R>::WAVE_D;
    __shared__ double smem[4 * WD];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + wid;
    if (item >= nitems) return;  // no block-wide barriers in the item: waves are independent
    jk_wave_item<LA, LB, LC, LD, R>(items[item], lane, smem + wid * WD, g, pp, rys_tab);
}

// Mixed precision in one launch: items [0, n64) FP64, the rest FP32 (one branch per wavefront).
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void jk_wave_kernel_mp(const int4* __restrict__ items, int nitems, int n64,
                                                         const JkArgs g, const PrimPair<double>* __restrict__ pp,
                                                         const PrimPair<float>* __restrict__ ppf,
                                                         const double* __restrict__ rys_tab,
                                                         const float* __restrict__ rys_tabf) {
    constexpr int WD64 = JkWave<LA, LB, LC, LD, double>::WAVE_D, WD32 = JkWave<LA, LB, LC, LD, float>::WAVE_D;
    constexpr int WD = WD64 > WD32 ? WD64 : WD32;
    __shared__ double smem[4 * WD];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + wid;
    if (item >= nitems) return;
    if (item < n64) jk_wave_item<LA, LB, LC, LD, double>(items[item], lane, smem + wid * WD, g, pp, rys_tab);
    else jk_wave_item<LA, LB, LC, LD, float>(items[item], lane, smem + wid * WD, g, ppf, rys_tabf);
}

__device__ __forceinline__ int64_t pair_index64(int64_t i, int64_t j) {
    return i >= j ? i * (i + 1) / 2 + j : j * (j + 1) / 2 + i;
}

// One element of the 8-fold compressed tensor (eri_compressed, integrals/eri/mod.rs:992-1070; index
// pair_index/eri_index :946-960): component (a, b, c, d) of the quartet (P|Q), v with the norms.  Every
// element of a surviving quartet is written once.
__device__ __forceinline__ void tensor_put(double* __restrict__ out, int bfa, int bfb, bool same_p, int bfc, int bfd,
                                           bool same_q, bool same_pq, int a, int b, int c, int d, double v) {
    const int i = bfa + a, j = bfb + b, k = bfc + c, l = bfd + d;
    if ((same_p && i < j) || (same_q && k < l)) return;
    const int64_t ij = pair_index64(i, j), kl = pair_index64(k, l);
    if (same_pq && ij < kl) return;
    const int64_t hi = ij > kl ? ij : kl, lo = ij > kl ? kl : ij;
    out[hi * (hi + 1) / 2 + lo] = v;
}

// The tensor by work items like those of J/K (lanes per ket, ket arrays), one block per item, for the
// classes up to kTensorLaneMaxNQ components, whose quartet fits a lane's registers; one wavefront per
// quartet above (eri_tensor_wave_kernel).  With one lane per quartet whatever its class the d classes'
// quartets lived in scratch: propane/6-31G* (61 functions) took 16.9 ms per call, now 1.34 ms, of which
// the kernels (35 us each, four streams) are a quarter and the 14 MB copy to the host most of the rest.
template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(128) void eri_tensor_kernel(const int4* __restrict__ items, const JkArgs g,
                                                         const KetPrims<double> kprims,
                                                         const PrimPair<double>* __restrict__ pp,
                                                         const double* __restrict__ rys_tab, double* __restrict__ out) {
    using S = EriShape<LA, LB, LC, LD>;
    __shared__ double rys_raw[rys_lds_doubles<S::NROOTS>()];
    const double* rys_n = rys_stage<double, S::NROOTS>(rys_tab, rys_raw);
    __syncthreads();
    const int4 it = items[blockIdx.x];
    const PairRec P = item_bra(g.bra, it);
    const int tid = threadIdx.x, lg = item_lg(it), lanes = 1 << lg, sub = tid & (lanes - 1), step = blockDim.x >> lg;
    KetCursor cur{g.segs, it.y, it.z + (tid >> lg)};
    for (int j = tid >> lg; j < item_kets(it); j += step, cur.r += step) {
        const int q = cur.at();
        const int4 km = g.kpairs.meta[q];
        const PairRec Q = ket_pair<LC, LD>(g.kpairs, q, km);
        const int kstride = km.w;
        double eri[S::NQ];
        for_n<S::NQ>([&](int i) { eri[i] = 0.0; });
        contract_quartet_pp<LA, LB, LC, LD, double, true>(
            P, Q, pp + P.pp_off, [&](int i) { return kprims.at(km.z + i * kstride); }, rys_n, eri, sub, lanes);
        if (lg) {
            for (int off = 1; off < lanes; off <<= 1)
                for_n<S::NQ>([&](int i) { eri[i] += __shfl_xor(eri[i], off, 64); });
            if (sub) continue;
        }
        const bool same_q = km.x & kKetSame, same_pq = g.diag && q == P.pos;
        static_for<S::NQ>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            constexpr int d = k % S::ND, c = (k / S::ND) % S::NC, b = (k / S::NCD) % S::NB, a = k / (S::NCD * S::NB);
            tensor_put(out, P.bfa, P.bfb, P.sa == P.sb, Q.bfa, Q.bfb, same_q, same_pq, a, b, c, d,
                       eri[k] * (cnorm(LA, a) * cnorm(LB, b) * cnorm(LC, c) * cnorm(LD, d)));
        });
    }
}

template <int LA, int LB, int LC, int LD>
__global__ __launch_bounds__(256) void eri_tensor_wave_kernel(const int4* __restrict__ items, int nitems, const JkArgs g,
                                                              const PrimPair<double>* __restrict__ pp,
                                                              const double* __restrict__ rys_tab,
                                                              double* __restrict__ out) {
    using W = JkWave<LA, LB, LC, LD, double>;
    using S = EriShape<LA, LB, LC, LD>;
    __shared__ double smem[4 * W::T::DOUBLES];
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + wid;
    if (item >= nitems) return;
    const int4 it = items[item];
    const PairRec P = item_bra(g.bra, it);
    KetCursor cur{g.segs, it.y, it.z};
    for (int j = 0; j < item_kets(it); ++j, ++cur.r) {
        const int q = cur.at();
        const PairRec Q = g.ket[q];
        double acc[W::KPL];
        wave_quartet<LA, LB, LC, LD, double>(P, Q, pp, rys_tab, smem + wid * W::T::DOUBLES, lane, acc);
#pragma unroll
        for (int m = 0; m < W::KPL; ++m) {
            const int k = lane + 64 * m;
            if (k < S::NQ) {
                const int d = k % S::ND, c = (k / S::ND) % S::NC, b = (k / S::NCD) % S::NB, a = k / (S::NCD * S::NB);
                tensor_put(out, P.bfa, P.bfb, P.sa == P.sb, Q.bfa, Q.bfb, Q.sa == Q.sb, g.diag && q == P.pos, a, b, c, d,
                           acc[m] * (cnorm(LA, a) * cnorm(LB, b) * cnorm(LC, c) * cnorm(LD, d)));
            }
        }
    }
}

#define QCG_LA(c) ((c) == 0 ? 0 : (c) <= 2 ? 1 : 2)
#define QCG_LB(c) ((c) == 0 || (c) == 1 || (c) == 3 ? 0 : ((c) == 2 || (c) == 4) ? 1 : 2)

static JkArgs jk_args(const JkLaunch& a) {
    return {a.segs, a.bra, a.ket, a.kpairs, a.D, a.Dp, a.fix, a.Jacc, a.Jmat, a.Kacc, a.ket_off, a.mat_off, a.mol_nbf,
            a.diag, a.do_j, a.do_k, a.jb_bra, a.jb_ket, a.np_bra, a.np_ket};
}

// One launch per part of the first shell's components (jk_part).
template <int LA, int LB, int LC, int LD, typename R, int NAS, int A0 = 0>
static hipError_t launch_jk_parts(const JkLaunch& a, const JkArgs& g, hipStream_t st) {
    // K rows of the bra functions in LDS when they fit (a.nbf is the largest molecule's nbf)
    const size_t rows = a.do_k ? jk_row_bytes(NAS + ncart(LB), jk_table_bytes(EriShape<LA, LB, LC, LD>::NROOTS), a.nbf) : 0;
    const KetPrims<R>* kp;
    if constexpr (sizeof(R) == 8) kp = &a.kprims;
    else kp = &a.kprimsf;
    const dim3 block(a.block > 0 ? a.block : 64);
    if (rows)
        hipLaunchKernelGGL((jk_kernel<LA, LB, LC, LD, R, true, A0, NAS>), dim3(a.nitems), block, rows, st, a.items, g, *kp,
                           (const PrimPair<R>*)a.pp, (const R*)a.rys);
    else
        hipLaunchKernelGGL((jk_kernel<LA, LB, LC, LD, R, false, A0, NAS>), dim3(a.nitems), block, 0, st, a.items, g, *kp,
                           (const PrimPair<R>*)a.pp, (const R*)a.rys);
    const hipError_t e = hipGetLastError();
    if constexpr (A0 + NAS < ncart(LA)) return e != hipSuccess ? e : launch_jk_parts<LA, LB, LC, LD, R, NAS, A0 + NAS>(a, g, st);
    else return e;
}
template <int LA, int LB, int LC, int LD, int NAS, int A0 = 0>
static hipError_t launch_jk_mp_parts(const JkLaunch& a, const JkArgs& g, hipStream_t st) {
    const size_t rows = a.do_k ? jk_row_bytes(NAS + ncart(LB), jk_table_bytes(EriShape<LA, LB, LC, LD>::NROOTS), a.nbf) : 0;
    auto go = [&](auto rows_c) {
        hipLaunchKernelGGL((jk_kernel_mp<LA, LB, LC, LD, decltype(rows_c)::value, A0, NAS>), dim3(a.nitems),
                           dim3(a.block > 0 ? a.block : 64), rows, st, a.items, a.n64, g, a.kprims, a.kprimsf,
                           (const PrimPair<double>*)a.pp, (const PrimPair<float>*)a.ppf, (const double*)a.rys,
                           (const float*)a.rysf);
    };
    if (rows) go(std::true_type{});
    else go(std::false_type{});
    const hipError_t e = hipGetLastError();
    if constexpr (A0 + NAS < ncart(LA)) return e != hipSuccess ? e : launch_jk_mp_parts<LA, LB, LC, LD, NAS, A0 + NAS>(a, g, st);
    else return e;
}

template <int CB, int CK, typename R>
static hipError_t launch_jk_t(const JkLaunch& a, hipStream_t st) {
    constexpr int LA = QCG_LA(CB), LB = QCG_LB(CB), LC = QCG_LA(CK), LD = QCG_LB(CK), NAS = jk_part(CB, CK);
    if (a.nitems <= 0) return hipSuccess;
    // wave-cooperative mode (four items per block); classes without a per-lane form always take it
    if (a.block == 0 || NAS == 0) {
        if constexpr (JkWave<LA, LB, LC, LD, R>::kEnabled) {
            hipLaunchKernelGGL((jk_wave_kernel<LA, LB, LC, LD, R>), dim3((a.nitems + 3) / 4), dim3(256), 0, st, a.items,
                               a.nitems, jk_args(a), (const PrimPair<R>*)a.pp, (const R*)a.rys);
            return hipGetLastError();
        }
    }
    if constexpr (NAS > 0) return launch_jk_parts<LA, LB, LC, LD, R, NAS>(a, jk_args(a), st);
    else return hipErrorInvalidValue;  // not reached: these classes take the wave-cooperative form above
}

// Mixed precision, both parts in one launch: a.items holds a.n64 FP64 items then the FP32 items,
// all cut for the same tile (a.block); a.pp/a.rys are the FP64 data, a.ppf/a.rysf the FP32 copies.
template <int CB, int CK>
static hipError_t launch_jk_mp_t(const JkLaunch& a, hipStream_t st) {
    constexpr int LA = QCG_LA(CB), LB = QCG_LB(CB), LC = QCG_LA(CK), LD = QCG_LB(CK), NAS = jk_part(CB, CK);
    if (a.nitems <= 0) return hipSuccess;
    if (a.block == 0 || NAS == 0) {
        if constexpr (JkWave<LA, LB, LC, LD, double>::kEnabled) {
            hipLaunchKernelGGL((jk_wave_kernel_mp<LA, LB, LC, LD>), dim3((a.nitems + 3) / 4), dim3(256), 0, st, a.items,
                               a.nitems, a.n64, jk_args(a), (const PrimPair<double>*)a.pp, (const PrimPair<float>*)a.ppf,
                               (const double*)a.rys, (const float*)a.rysf);
            return hipGetLastError();
        }
    }
    if constexpr (NAS > 0) return launch_jk_mp_parts<LA, LB, LC, LD, NAS>(a, jk_args(a), st);
    else return hipErrorInvalidValue;  // not reached: these classes take the wave-cooperative form above
}

template <int CB, int CK>
static hipError_t launch_tensor_t(const JkLaunch& a, double* out, hipStream_t st) {
    constexpr int LA = QCG_LA(CB), LB = QCG_LB(CB), LC = QCG_LA(CK), LD = QCG_LB(CK);
    using S = EriShape<LA, LB, LC, LD>;
    if (a.nitems <= 0) return hipSuccess;
    if constexpr (S::NQ <= kTensorLaneMaxNQ)
        hipLaunchKernelGGL((eri_tensor_kernel<LA, LB, LC, LD>), dim3(a.nitems), dim3(a.block), 0, st, a.items, jk_args(a),
                           a.kprims, (const PrimPair<double>*)a.pp, (const double*)a.rys, out);
    else
        hipLaunchKernelGGL((eri_tensor_wave_kernel<LA, LB, LC, LD>), dim3((a.nitems + 3) / 4), dim3(256), 0, st, a.items,
                           a.nitems, jk_args(a), (const PrimPair<double>*)a.pp, (const double*)a.rys, out);
    return hipGetLastError();
}

#define QCG_CAT2(a, b) a##b
#define QCG_CAT(a, b) QCG_CAT2(a, b)

hipError_t QCG_CAT(launch_jk_cb, QCG_CB)(int ck, bool fp32, const JkLaunch& a, hipStream_t st) {
    switch (ck) {
#define QCG_K(CK) \
    case CK: if constexpr (CK <= QCG_CB) return a.n64 >= 0 ? launch_jk_mp_t<QCG_CB, CK>(a, st) : fp32 ? launch_jk_t<QCG_CB, CK, float>(a, st) : launch_jk_t<QCG_CB, CK, double>(a, st); break;
        QCG_K(0) QCG_K(1) QCG_K(2) QCG_K(3) QCG_K(4) QCG_K(5)
#undef QCG_K
    }
    return hipErrorInvalidValue;
}

hipError_t QCG_CAT(launch_tensor_cb, QCG_CB)(int ck, const JkLaunch& a, double* out, hipStream_t st) {
    switch (ck) {
#define QCG_K(CK) \
    case CK: if constexpr (CK <= QCG_CB) return launch_tensor_t<QCG_CB, CK>(a, out, st); break;
        QCG_K(0) QCG_K(1) QCG_K(2) QCG_K(3) QCG_K(4) QCG_K(5)
#undef QCG_K
    }
    return hipErrorInvalidValue;
}

}  // namespace qcg
