// Host-side launch interface of the two-electron kernels.
#pragma once
#include <algorithm>
#include <vector>

#include "fixacc.h"
#include "qcg_types.h"
#include "rys.h"

namespace qcg {

// Work items over ket segments.  The surviving kets of one bra pair are one contiguous range per
// contraction bucket; the host lists those ranges as segments (first ket, count) and cuts their
// concatenation into items (bra index, first segment, offset into it, w), so a block's lanes stay
// busy across bucket boundaries instead of idling at the end of every bucket.
//
// w packs the ket count (bits 0-12), the lanes per ket of the per-lane J/K kernels as a power of two
// (bits 13-15) and an optional range of the bra's primitive pairs: first (bits 16-23)
// and count (bits 24-31, 0 = all).  A bra pair with many primitive pairs is cut into such ranges so
// that no lane runs the whole npp_bra x npp_ket primitive loop of a heavy quartet alone; the integral
// is linear in the bra primitives, so the partial quartets are digested (J and K) like whole ones.
constexpr int kItemMaxKets = 0x1fff;
constexpr int kItemMaxPrim = 0xff;
constexpr int kItemMaxLg = 6;  // at most a whole wavefront per ket

// items of at most ch kets over segments [g0, g1) of bra `bra`, 2^lg lanes per ket, primitive
// range (pbeg, pcnt) (pcnt = 0: all of them)
inline void cut_items(std::vector<int4>& items, const std::vector<int2>& segs, int g0, int g1, int bra, int ch,
                      int lg = 0, int pbeg = 0, int pcnt = 0) {
    int total = 0;
    for (int g = g0; g < g1; ++g) total += segs[g].y;
    const int wbits = (lg << 13) | (pbeg << 16) | (pcnt << 24);
    int g = g0, r = 0;
    for (int off = 0; off < total; off += ch) {
        const int n = std::min(ch, total - off);
        items.push_back(make_int4(bra, g, r, n | wbits));
        r += n;
        while (g < g1 && r >= segs[g].y) r -= segs[g++].y;
    }
}

// cut_items for every primitive range of a bra pair with npp primitive pairs: ranges of at most
// split pairs (split <= 0 or npp <= split: one range, the whole pair), sizes balanced; npp is at most
// kItemMaxPrim (the planners refuse longer contractions)
inline void cut_items_split(std::vector<int4>& items, const std::vector<int2>& segs, int g0, int g1, int bra, int ch,
                            int npp, int split, int lg = 0) {
    if (split <= 0 || npp <= split) {
        cut_items(items, segs, g0, g1, bra, ch, lg);
        return;
    }
    const int nr = (npp + split - 1) / split;
    for (int k = 0; k < nr; ++k) {
        const int b = k * npp / nr, e = (k + 1) * npp / nr;
        cut_items(items, segs, g0, g1, bra, ch, lg, b, e - b);
    }
}

QCG_HD int item_kets(const int4& it) { return it.w & kItemMaxKets; }
QCG_HD int item_lg(const int4& it) { return (it.w >> 13) & 7; }

// Most bra primitive pairs one J/K item may have: the planner cuts heavier bras into primitive ranges
// of at most this many.
constexpr int kBraPPMax = 64;

// Largest class (Cartesian components) whose per-lane J/K kernel holds a whole quartet in registers;
// classes from 27 components on may also run the wave-cooperative kernel (tile block 0).
constexpr int kJkLaneMaxNQ = 81;

// Components of the first shell that one launch of the per-lane J/K kernel of a class takes: all of them up
// to kJkLaneMaxNQ components, else as many as keep a part at kJkPartMaxNQ (0: no per-lane form).  Every
// part evaluates the quartet's roots and 2D integrals anew, yet against the wave-cooperative kernel, whose
// lanes share one quartet's components and leave half of the fused multiply-adds to index arithmetic, a
// class with at most two or three parts is the faster one once a launch has lanes enough (default_tiles):
// (H2O)16 6-31G* FP64 (dp|ds) 0.50 -> 0.18 ms, (dd|ps) 0.29 -> 0.20, (dp|pp) 0.25 -> 0.22, the build 3.40 ->
// 2.73 ms.  At a total angular momentum of 6 the classes alone are slower ((dp|dp) 0.12 -> 0.28 ms), but run
// beside others on the four streams they fill the chip better: build 2.80 ms without them, 2.73 with.  The same
// with and without them over sizes, FP64 / mixed: (H2O)12 -2 / -1 %, (H2O)16 -4 / -2 %, (H2O)24 -4 / -3 %, dodecane
// -2 / -1 %, decane 0 / 0, (H2O)8 6-31+G* +1 / +1 %; smaller molecules have too few quartets for parts.
// Above, (dd|dp) and (dd|dd) would need six or more parts.
constexpr int kJkPartMaxNQ = 54;
constexpr int kJkPartMaxL = 6;
constexpr int jk_part(int cb, int ck) {
    const int na = cb == 0 ? 1 : cb <= 2 ? 3 : 6;
    const int nc[6] = {1, 3, 9, 6, 18, 36};
    const int rest = nc[cb] / na * nc[ck];
    if (na * rest <= kJkLaneMaxNQ) return na;
    const int l[6] = {0, 1, 2, 2, 3, 4};
    if (l[cb] + l[ck] > kJkPartMaxL) return 0;
    for (int n = na; n >= 1; --n)
        if (na % n == 0 && n * rest <= kJkPartMaxNQ) return n;
    return 0;
}

// LDS of a per-lane J/K block: the Rys coefficients of nr nodes when they are staged (else one word), and the K rows of the
// bra's functions (nrow of them in a part) for nbf functions (the largest molecule's) when they fit the
// budget that the coefficients leave; 0 rows: K goes to memory directly.
constexpr size_t kJkLdsBudget = 65536;
inline size_t jk_table_bytes(int nr) { return nr <= 3 ? (size_t)(qcg_rys_off[nr + 1] - qcg_rys_off[nr]) * sizeof(double) : sizeof(double); }
inline size_t jk_row_bytes(int nrow, size_t table, int nbf) {
    const size_t kb = (size_t)nrow * nbf * sizeof(fix_t);
    return table + kb <= kJkLdsBudget ? kb : 0;
}

// The same limit for the compressed tensor's kernels.
constexpr int kTensorLaneMaxNQ = 54;

// the bra pair of an item, restricted to the item's primitive range
QCG_HD PairRec item_bra(const PairRec* __restrict__ bra, const int4& it) {
    PairRec P = bra[it.x];
    const int pcnt = (it.w >> 24) & kItemMaxPrim;
    if (pcnt) {
        P.pp_off += (it.w >> 16) & kItemMaxPrim;
        P.npp = pcnt;
    }
    return P;
}

// Device cursor over an item's kets: position r counts kets from the start of segment g; at()
// returns the ket index and may be called only for the item's own kets (j < item count), which
// keeps the walk inside the bra's segments.
struct KetCursor {
    const int2* __restrict__ seg;
    int g, r;
    __device__ __forceinline__ int at() {
        int2 s = seg[g];
        while (r >= s.y) {
            r -= s.y;
            s = seg[++g];
        }
        return s.x + r;
    }
};

struct JkLaunch {
    const PairRec* bra;
    const PairRec* ket;
    int diag;           // bra class == ket class: only ket positions <= bra position
    const void* pp;     // PrimPair<double> or PrimPair<float>
    const void* rys;    // Rys table (double or float)
    const double* D;    // density, nbf x nbf, symmetric
    int nbf;
    // J side by shell pair instead of by matrix element: component ab of pair i (index in its class)
    // is word base + ab * (pairs of the class) + i of Dp (the density with the component norms) and
    // Jacc (its accumulator), so the lanes of a wavefront, on consecutive kets, touch consecutive words
    const double* Dp;
    int jb_bra, jb_ket, np_bra, np_ket;  // bases and pair counts of the two classes
    fix_t* Jacc;        // fixed-point accumulators (fixacc.h): J by shell pair
    fix_t* Jmat;        // the wave-cooperative kernels' J, nbf x nbf: their few lanes per ket would all
                        // add to the same lines of Jacc ((dd|ps) of benzene 52 -> 109 us)
    fix_t* Kacc;        // nbf x nbf
    KetPairs kpairs;    // the kets of the class as arrays (per-lane kernels); primitives in kprims / kprimsf
    KetPrims<double> kprims;
    KetPrims<float> kprimsf;
    const double* fix;  // per molecule: scale of J, scale of K, and their inverses (fix_scale_kernel)
    int do_j, do_k;
    // batch of molecules (nmol = 1 for a single molecule): kets of bra pair P are
    // those of the items from ket[ket_off[P.mol]] on; matrices of molecule m start at mat_off[m],
    // dimension mol_nbf[m]; nbf above is the largest mol_nbf.
    const int* ket_off;
    const int64_t* mat_off;
    const int* mol_nbf;
    // J/K work items (index in the bra class list, first segment, offset into it, ket count) over
    // the ket segments segs[g] = (first ket, count), ket indices relative to the molecule's list
    // (see KetCursor); one block of `block` threads per item
    const int4* items;
    const int2* segs;
    int nitems;
    int block;
    // mixed precision in one launch (n64 >= 0): the first n64 items are FP64, the rest FP32 with
    // the FP32 primitive pairs ppf and Rys table rysf; n64 < 0: one precision, given by the caller
    int n64 = -1;
    const void* ppf = nullptr;
    const void* rysf = nullptr;
};

hipError_t launch_jk_cb0(int ck, bool fp32, const JkLaunch& a, hipStream_t st);
hipError_t launch_jk_cb1(int ck, bool fp32, const JkLaunch& a, hipStream_t st);
hipError_t launch_jk_cb2(int ck, bool fp32, const JkLaunch& a, hipStream_t st);
hipError_t launch_jk_cb3(int ck, bool fp32, const JkLaunch& a, hipStream_t st);
hipError_t launch_jk_cb4(int ck, bool fp32, const JkLaunch& a, hipStream_t st);
hipError_t launch_jk_cb5(int ck, bool fp32, const JkLaunch& a, hipStream_t st);
hipError_t launch_tensor_cb0(int ck, const JkLaunch& a, double* out, hipStream_t st);
hipError_t launch_tensor_cb1(int ck, const JkLaunch& a, double* out, hipStream_t st);
hipError_t launch_tensor_cb2(int ck, const JkLaunch& a, double* out, hipStream_t st);
hipError_t launch_tensor_cb3(int ck, const JkLaunch& a, double* out, hipStream_t st);
hipError_t launch_tensor_cb4(int ck, const JkLaunch& a, double* out, hipStream_t st);
hipError_t launch_tensor_cb5(int ck, const JkLaunch& a, double* out, hipStream_t st);

inline hipError_t launch_jk(int cb, int ck, bool fp32, const JkLaunch& a, hipStream_t st) {
    switch (cb) {
        case 0: return launch_jk_cb0(ck, fp32, a, st);
        case 1: return launch_jk_cb1(ck, fp32, a, st);
        case 2: return launch_jk_cb2(ck, fp32, a, st);
        case 3: return launch_jk_cb3(ck, fp32, a, st);
        case 4: return launch_jk_cb4(ck, fp32, a, st);
        case 5: return launch_jk_cb5(ck, fp32, a, st);
    }
    return hipErrorInvalidValue;
}

inline hipError_t launch_eri_tensor(int cb, int ck, const JkLaunch& a, double* out, hipStream_t st) {
    switch (cb) {
        case 0: return launch_tensor_cb0(ck, a, out, st);
        case 1: return launch_tensor_cb1(ck, a, out, st);
        case 2: return launch_tensor_cb2(ck, a, out, st);
        case 3: return launch_tensor_cb3(ck, a, out, st);
        case 4: return launch_tensor_cb4(ck, a, out, st);
        case 5: return launch_tensor_cb5(ck, a, out, st);
    }
    return hipErrorInvalidValue;
}

struct GradLaunch {
    const PairRec* bra;
    const PairRec* ket;
    int diag;
    const PrimPair<double>* pp;  // ea and p - ea are the two primitive exponents
    KetPairs kpairs;             // the kets as arrays (per-lane kernels), kea their first exponents
    KetPrims<double> kprims;
    const double* kea;
    const double* rys;
    const double* D;
    int nbf;
    double xfac;  // exchange weight c = hf_frac / 4 (eri_gradient_fused, scf/gradient.rs:1438)
    int natom;
    double* grad;  // 3 * natom, accumulated
    // work items (index in the bra class list, first segment, offset into it, ket count) over the
    // ket segments segs (see KetCursor): one wavefront, or one block of lanes, each
    const int4* items;
    const int2* segs;
    int nitems;
};

// Components of the first shell that one launch of the per-lane gradient kernel of a class takes (0: the
// class runs wave-cooperatively): as many as keep the weights and 1-D tables of a lane in registers
// (measured at the kernel).
constexpr int kGradLaneMaxNQ = 54;
constexpr int grad_part(int cb, int ck) {
    const int na = cb == 0 ? 1 : cb <= 2 ? 3 : 6;
    const int nc[6] = {1, 3, 9, 6, 18, 36};
    const int rest = nc[cb] / na * nc[ck];
    for (int n = na; n >= 1; --n)
        if (na % n == 0 && n * rest <= kGradLaneMaxNQ) return n;
    return 0;
}

// Work-item length (kets per item) of a class with n quartets in the gradient: one block of 128 threads
// per item for the per-lane kernel, up to eight kets per lane once that leaves 4096 blocks, and one to
// eight kets per wavefront otherwise.
inline int grad_item_kets(int cb, int ck, int64_t n) {
    if (grad_part(cb, ck) > 0) return 128 * (int)std::max<int64_t>(1, std::min<int64_t>(8, n / (128 * 4096)));
    return (int)std::max<int64_t>(1, std::min<int64_t>(8, n / 2048));
}

hipError_t launch_grad_cb0(int ck, const GradLaunch& a, hipStream_t st);
hipError_t launch_grad_cb1(int ck, const GradLaunch& a, hipStream_t st);
hipError_t launch_grad_cb2(int ck, const GradLaunch& a, hipStream_t st);
hipError_t launch_grad_cb3(int ck, const GradLaunch& a, hipStream_t st);
hipError_t launch_grad_cb4(int ck, const GradLaunch& a, hipStream_t st);
hipError_t launch_grad_cb5(int ck, const GradLaunch& a, hipStream_t st);

inline hipError_t launch_grad(int cb, int ck, const GradLaunch& a, hipStream_t st) {
    switch (cb) {
        case 0: return launch_grad_cb0(ck, a, st);
        case 1: return launch_grad_cb1(ck, a, st);
        case 2: return launch_grad_cb2(ck, a, st);
        case 3: return launch_grad_cb3(ck, a, st);
        case 4: return launch_grad_cb4(ck, a, st);
        case 5: return launch_grad_cb5(ck, a, st);
    }
    return hipErrorInvalidValue;
}

hipError_t launch_schwarz(int c, const PairRec* pairs, int n, const PrimPair<double>* pp, const double* rys,
                          double* Q, hipStream_t st);
hipError_t launch_fill(double* x, size_t n, double v, hipStream_t st);
// The kets of all classes as arrays (KetPairs, KetPrims) from the pair records and their primitive pairs: meta is
// given, the others are written.  jmap: of every matrix element the word of the pair-ordered J arrays, pair i of
// class k and component ab at jbase[k] + ab * (pairs of the class) + i, -1 where only the transposed element has one.
struct KetArrays {
    int np, npr;  // pairs, primitive pairs
    int off[kNumPairClasses + 1], jbase[kNumPairClasses], nb[kNumPairClasses], nab[kNumPairClasses];
    const PairRec* pairs;
    const PrimPair<double>* pp;
    const PrimPair<float>* ppf;
    const int4* meta;
    const int64_t* mat_off;
    const int* mol_nbf;
    double2 *cen, *prim;
    double *hp, *ea;
    int2* atoms;
    float4* primf;
    int* jmap;
};
hipError_t launch_ket_arrays(const KetArrays& a, size_t mat_total, hipStream_t st);
// What the fixed-point scale kernels read (device pointers, packed per molecule): the Schwarz bounds
// of the shell pairs as nshell x nshell matrices (qsh, offsets qsh_off), their maximum (qmax), the
// shell of every function (bf_shell, offsets bf_off into the functions of all molecules), the first
// function of every shell plus a sentinel (shell_first, offsets shell_first_off), the molecule of
// every function (row_mol, nrows functions in all) and 2 doubles of scratch per function (rowsum).
struct FixData {
    const int64_t* mat_off;
    const int* mol_nbf;
    const double* qsh;
    const int64_t* qsh_off;
    const int* mol_ns;
    const int* bf_shell;
    const int* bf_off;
    const int* row_mol;
    int nrows;
    double* rowsum;
    const double* qmax;
    const int* shell_first;
    const int* shell_first_off;
    // word of the pair-ordered J arrays (JkLaunch) that matrix element e belongs to, -1 for the
    // elements of the pair's transposed block, and the component norm of every function
    const int* jmap;
    const double* bf_norm;
};
// Per molecule m the fixed-point scales fix[4m] (J) and fix[4m + 1] (K) and their inverses from a
// bound on the accumulated magnitudes at density D: B_J = 2 Qmax sum_ls Q_ls |D_ls|,
// B_K = 2 Qmax max_s sum_t Q_st sum_(n in t) sum_l |D_nl|.  Also zeroes the accumulators Jacc and
// Kacc (either may be null).
// With Jacc also fills the pair-ordered density Dp.
hipError_t launch_fix_scale(const double* D, const FixData& f, double* fix, int nmol, fix_t* Jacc, fix_t* Jmat,
                            fix_t* Kacc, double* Dp, hipStream_t st);
hipError_t launch_symmetrize(const fix_t* Jacc, const fix_t* Jmat, const fix_t* Kacc, const int* jmap, const double* fix,
                             double* J, double* K, int nbf, hipStream_t st);
// batched J = Jacc + Jacc^T, K = Kacc + Kacc^T over block-diagonal packed matrices
hipError_t launch_symmetrize_batch(const fix_t* Jacc, const fix_t* Jmat, const fix_t* Kacc, const int* jmap,
                                   const double* fix, double* J, double* K, int nmol, const int64_t* mat_off, const int* mol_nbf, int max_nbf, hipStream_t st);
hipError_t launch_fock_combine(const double* H, const fix_t* Jacc, const fix_t* Jmat, const fix_t* Kacc, const int* jmap,
                               const double* fix, double* F, int nbf, double kfac, hipStream_t st);
hipError_t launch_boys_batch(int m, int n, const double* T, double* F, int* status, hipStream_t st);
hipError_t launch_rys_batch(int nroots, int n, const double* T, const double* tab, double* x, double* w,
                            hipStream_t st);
hipError_t launch_rys_batch_f32(int nroots, int n, const float* T, const float* tab, float* x, float* w,
                                hipStream_t st);

}  // namespace qcg
