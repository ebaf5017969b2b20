// Small kernels around the J/K build: Schwarz bounds, Boys/Rys batches, fills, J/K symmetrisation.
#include "boys.h"
#include "eri_device.h"
#include "eri_launch.h"
#include "eri_wave.h"

namespace qcg {

// Schwarz bound per pair: sqrt(max |(ab|ab)|) (compute_schwarz_bounds, integrals/eri/mod.rs:1263-1290).
// One wavefront per pair: up to 81 components its lanes split the ket's primitives and sum the partial
// quartets (a fixed butterfly), above it works as eri_wave.h.  One lane per pair had run every primitive
// quartet in series, the (dp|dp) and (dd|dd) ones in scratch: 6.0 ms for any molecule with d shells.
template <int LA, int LB>
__global__ __launch_bounds__(256) void schwarz_kernel(const PairRec* __restrict__ pairs, int n,
                                                      const PrimPair<double>* __restrict__ pp,
                                                      const double* __restrict__ rys_tab, double* __restrict__ Q) {
    using S = EriShape<LA, LB, LA, LB>;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;  // the whole wavefront; no block-wide barrier below
    const PairRec P = pairs[i];
    double mx = 0.0;
    auto norm = [](int k) {
        const int d = k % S::NB, c = (k / S::NB) % S::NA, b = (k / S::NAB) % S::NB, a = k / (S::NAB * S::NB);
        return cnorm(LA, a) * cnorm(LB, b) * cnorm(LA, c) * cnorm(LB, d);
    };
    if constexpr (S::NQ <= 81) {
        double eri[S::NQ];
        for_n<S::NQ>([&](int k) { eri[k] = 0.0; });
        const PrimPair<double>* ppk = pp + P.pp_off;
        contract_quartet_pp<LA, LB, LA, LB, double>(P, P, ppk, [ppk](int j) { return ppk[j]; }, rys_tab, eri, lane, 64);
        for (int off = 1; off < 64; off <<= 1) for_n<S::NQ>([&](int k) { eri[k] += __shfl_xor(eri[k], off, 64); });
        for_n<S::NQ>([&](int k) { mx = fmax(mx, fabs(eri[k] * norm(k))); });
    } else {
        using TB = WaveTable<LA, LB, LA, LB, S::NROOTS, double>;
        constexpr int KPL = (S::NQ + 63) / 64;
        __shared__ double smem[4 * TB::DOUBLES];
        double acc[KPL];
        wave_quartet<LA, LB, LA, LB, double>(P, P, pp, rys_tab, smem + (threadIdx.x >> 6) * TB::DOUBLES, lane, acc);
#pragma unroll
        for (int j = 0; j < KPL; ++j)
            if (lane + 64 * j < S::NQ) mx = fmax(mx, fabs(acc[j] * norm(lane + 64 * j)));
        for (int off = 1; off < 64; off <<= 1) mx = fmax(mx, __shfl_xor(mx, off, 64));
    }
    if (lane == 0) Q[i] = sqrt(mx);
}

hipError_t launch_schwarz(int c, const PairRec* pairs, int n, const PrimPair<double>* pp, const double* rys,
                          double* Q, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    const dim3 g((n + 3) / 4), b(256);
    switch (c) {
        case 0: hipLaunchKernelGGL((schwarz_kernel<0, 0>), g, b, 0, st, pairs, n, pp, rys, Q); break;
        case 1: hipLaunchKernelGGL((schwarz_kernel<1, 0>), g, b, 0, st, pairs, n, pp, rys, Q); break;
        case 2: hipLaunchKernelGGL((schwarz_kernel<1, 1>), g, b, 0, st, pairs, n, pp, rys, Q); break;
        case 3: hipLaunchKernelGGL((schwarz_kernel<2, 0>), g, b, 0, st, pairs, n, pp, rys, Q); break;
        case 4: hipLaunchKernelGGL((schwarz_kernel<2, 1>), g, b, 0, st, pairs, n, pp, rys, Q); break;
        case 5: hipLaunchKernelGGL((schwarz_kernel<2, 2>), g, b, 0, st, pairs, n, pp, rys, Q); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

__global__ void fill_kernel(double* __restrict__ x, size_t n, double v) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) x[i] = v;
}

hipError_t launch_fill(double* x, size_t n, double v, hipStream_t st) {
    if (n == 0) return hipSuccess;
    size_t blocks = (n + 255) / 256;
    if (blocks > 8192) blocks = 8192;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, st, x, n, v);
    return hipGetLastError();
}

__global__ void jmap_clear_kernel(int* __restrict__ jmap, size_t n) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) jmap[i] = -1;
}

// One lane per pair.  As host loops with copies of the arrays this was a quarter of qcg_set_basis_batch: 64 alkanes
// 6-31G 85 -> 64 ms (60 ms before there were such arrays), (H2O)16 6-31G* 3.7 -> 3.5 ms.
__global__ __launch_bounds__(256) void ket_arrays_kernel(const KetArrays a) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= a.np) return;
    const PairRec r = a.pairs[g];
    const int4 km = a.meta[g];
    const size_t np = a.np, npr = a.npr;
    a.atoms[g] = make_int2(r.atom_a, r.atom_b);
    a.cen[g] = make_double2(r.ax, r.ay);
    a.cen[np + g] = make_double2(r.az, r.abx);
    a.cen[2 * np + g] = make_double2(r.aby, r.abz);
    for (int j = 0; j < km.y; ++j) {
        const size_t e = (size_t)km.z + (size_t)j * km.w;
        const PrimPair<double> q = a.pp[r.pp_off + j];
        const PrimPair<float> f = a.ppf[r.pp_off + j];
        a.prim[e] = make_double2(q.px, q.py);
        a.prim[npr + e] = make_double2(q.pz, q.p);
        a.prim[2 * npr + e] = make_double2(q.ckp, q.kab);
        a.hp[e] = q.hp;
        a.ea[e] = q.ea;
        a.primf[e] = make_float4(f.px, f.py, f.pz, f.p);
        a.primf[npr + e] = make_float4(f.ckp, f.hp, f.kab, f.ea);
    }
    int k = 0;
    while (g >= a.off[k + 1]) ++k;
    const int n = a.off[k + 1] - a.off[k];
    const size_t nbf = a.mol_nbf[r.mol];
    int* m = a.jmap + a.mat_off[r.mol] + (size_t)r.bfa * nbf + r.bfb;
    for (int ab = 0; ab < a.nab[k]; ++ab)
        m[(size_t)(ab / a.nb[k]) * nbf + ab % a.nb[k]] = a.jbase[k] + ab * n + (g - a.off[k]);
}

hipError_t launch_ket_arrays(const KetArrays& a, size_t mat_total, hipStream_t st) {
    hipLaunchKernelGGL(jmap_clear_kernel, dim3((unsigned)((mat_total + 255) / 256)), dim3(256), 0, st, a.jmap, mat_total);
    if (a.np > 0) hipLaunchKernelGGL(ket_arrays_kernel, dim3((a.np + 255) / 256), dim3(256), 0, st, a);
    return hipGetLastError();
}

// Fixed-point scales of one build (fixacc.h).  Every J contribution to element (m, n) is a product
// (mn|ls) D_ls with |(mn|ls)| <= Q_mn Q_ls (Schwarz, per component), so
// |Jacc_mn| <= Qmax sum_ls Q_ls |D_ls| (counted twice for the symmetry images: B_J); a K contribution
// to (m, l) is (mn|ls) D_ns, so |Kacc_ml| <= Qmax sum_t Q_sh(m),t rho_t with rho_t = sum over the
// functions n of shell t of sum_s |D_ns| (twice: B_K).  Two kernels: one wavefront per row of D for
// the row sums, then one block per molecule for the shell sums and the scales.  Every reduction runs
// in a fixed order, so the scales, like the sums they serve, are the same on every build of the same
// density.
__global__ __launch_bounds__(256) void fix_rows_kernel(
    const double* __restrict__ D, const int64_t* __restrict__ mat_off, const int* __restrict__ mol_nbf,
    const double* __restrict__ qsh, const int64_t* __restrict__ qsh_off, const int* __restrict__ mol_ns,
    const int* __restrict__ bf_shell, const int* __restrict__ bf_off, const int* __restrict__ row_mol, int nrows,
    double* __restrict__ rowsum, fix_t* __restrict__ Jacc, fix_t* __restrict__ Jmat, fix_t* __restrict__ Kacc,
    const int* __restrict__ jmap,
    const double* __restrict__ bf_norm, double* __restrict__ Dp) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= nrows) return;
    const int m = row_mol[row], n = row - bf_off[m], nbf = mol_nbf[m], ns = mol_ns[m];
    const int* bs = bf_shell + bf_off[m];
    const size_t ro = mat_off[m] + (size_t)n * nbf;
    const double* Drow = D + ro;
    const double* Qrow = qsh + qsh_off[m] + (size_t)bs[n] * ns;
    double r = 0.0, j = 0.0;
    for (int l = lane; l < nbf; l += 64) {
        const double a = fabs(Drow[l]);
        r += a;
        j += Qrow[bs[l]] * a;
        // the accumulators start at zero (null: that matrix is not built); J's are in pair order
        // next to the density with the component norms
        if (Kacc) Kacc[ro + l] = 0;
        if (Jacc) {
            Jmat[ro + l] = 0;
            const int e = jmap[ro + l];
            if (e >= 0) {
                Jacc[e] = 0;
                Dp[e] = Drow[l] * bf_norm[row] * bf_norm[bf_off[m] + l];
            }
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
        r += __shfl_xor(r, off, 64);
        j += __shfl_xor(j, off, 64);
    }
    if (lane == 0) {
        rowsum[2 * row] = r;
        rowsum[2 * row + 1] = j;
    }
}

constexpr int kFixMaxShells = 4096;  // shells per molecule the scale kernel handles (rho in LDS)

__global__ __launch_bounds__(1024) void fix_scale_kernel(FixData f, double* __restrict__ fix) {
    __shared__ double red[1024];
    __shared__ double rho[kFixMaxShells];
    const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nbf = f.mol_nbf[m], ns = f.mol_ns[m];
    const double* Q = f.qsh + f.qsh_off[m];
    const int* first = f.shell_first + f.shell_first_off[m];
    const double* rs = f.rowsum + 2 * (size_t)f.bf_off[m];
    // shell row sums rho_t over the shell's consecutive functions, and sum_n jrow_n
    double aj = 0.0;
    for (int n = tid; n < nbf; n += blockDim.x) aj += rs[2 * n + 1];
    for (int t = tid; t < ns; t += blockDim.x) {
        double v = 0.0;
        for (int n = first[t]; n < first[t + 1]; ++n) v += rs[2 * n];
        rho[t] = v;
    }
    red[tid] = aj;
    __syncthreads();
    for (int h = 512; h > 0; h >>= 1) {
        if (tid < h) red[tid] += red[tid + h];
        __syncthreads();
    }
    const double sumJ = red[0];
    __syncthreads();
    // max over shells s of sum_t Q_st rho_t: one wavefront per shell s, lanes over t
    double km = 0.0;
    for (int sh = wave; sh < ns; sh += 16) {
        double t = 0.0;
        for (int u = lane; u < ns; u += 64) t += Q[(size_t)sh * ns + u] * rho[u];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) t += __shfl_xor(t, off, 64);
        km = fmax(km, t);
    }
    red[tid] = km;
    __syncthreads();
    for (int h = 512; h > 0; h >>= 1) {
        if (tid < h) red[tid] = fmax(red[tid], red[tid + h]);
        __syncthreads();
    }
    if (tid == 0) {
        const double qmax = f.qmax[m];
        const double sj = fix_scale_for(2.0 * qmax * sumJ), sk = fix_scale_for(2.0 * qmax * red[0]);
        fix[4 * m] = sj;
        fix[4 * m + 1] = sk;
        fix[4 * m + 2] = 1.0 / sj;
        fix[4 * m + 3] = 1.0 / sk;
    }
}

hipError_t launch_fix_scale(const double* D, const FixData& f, double* fix, int nmol, fix_t* Jacc, fix_t* Jmat,
                            fix_t* Kacc, double* Dp, hipStream_t st) {
    hipLaunchKernelGGL(fix_rows_kernel, dim3((f.nrows + 3) / 4), dim3(256), 0, st, D, f.mat_off, f.mol_nbf, f.qsh,
                       f.qsh_off, f.mol_ns, f.bf_shell, f.bf_off, f.row_mol, f.nrows, f.rowsum, Jacc, Jmat, Kacc,
                       f.jmap, f.bf_norm, Dp);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(fix_scale_kernel, dim3(nmol), dim3(1024), 0, st, f, fix);
    return hipGetLastError();
}

// Element (i, j) of A + A^T for a fixed-point accumulator: the integer words are summed before
// the conversion, so the result is exactly symmetric.
__device__ __forceinline__ double fix_sym(const fix_t* __restrict__ a, size_t ij, size_t ji, double inv) {
    return fix_value(a[ij] + a[ji], inv);
}

// The same for J, whose words are in shell-pair order: jmap holds the word of element e, or -1 where
// only the transposed element has one (both do inside a pair of equal shells); mat: Jmat.
__device__ __forceinline__ double fix_sym_pairs(const fix_t* __restrict__ a, const fix_t* __restrict__ mat,
                                                const int* __restrict__ jmap, size_t ij, size_t ji, double inv) {
    const int e = jmap[ij], f = jmap[ji];
    return fix_value((e >= 0 ? a[e] : 0) + (f >= 0 ? a[f] : 0) + mat[ij] + mat[ji], inv);
}

// J = Jacc + Jacc^T, K = Kacc + Kacc^T
__global__ void symmetrize_kernel(const fix_t* __restrict__ Jacc, const fix_t* __restrict__ Jmat,
                                  const fix_t* __restrict__ Kacc,
                                  const int* __restrict__ jmap, const double* __restrict__ fix, double* __restrict__ J,
                                  double* __restrict__ K, int nbf) {
    const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nbf) return;
    const size_t ij = (size_t)i * nbf + j, ji = (size_t)j * nbf + i;
    if (J) J[ij] = fix_sym_pairs(Jacc, Jmat, jmap, ij, ji, fix[2]);
    if (K) K[ij] = fix_sym(Kacc, ij, ji, fix[3]);
}

__global__ void symmetrize_batch_kernel(const fix_t* __restrict__ Jacc, const fix_t* __restrict__ Jmat,
                                        const fix_t* __restrict__ Kacc,
                                        const int* __restrict__ jmap, const double* __restrict__ fix,
                                        double* __restrict__ J, double* __restrict__ K,
                                        const int64_t* __restrict__ mat_off, const int* __restrict__ mol_nbf) {
    const int m = blockIdx.z, n = mol_nbf[m];
    const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n || j >= n) return;
    const size_t o = (size_t)mat_off[m];
    const size_t ij = o + (size_t)i * n + j, ji = o + (size_t)j * n + i;
    if (J) J[ij] = fix_sym_pairs(Jacc, Jmat, jmap, ij, ji, fix[4 * m + 2]);
    if (K) K[ij] = fix_sym(Kacc, ij, ji, fix[4 * m + 3]);
}

hipError_t launch_symmetrize_batch(const fix_t* Jacc, const fix_t* Jmat, const fix_t* Kacc, const int* jmap,
                                   const double* fix, double* J, double* K, int nmol, const int64_t* mat_off, const int* mol_nbf, int max_nbf,
                                   hipStream_t st) {
    hipLaunchKernelGGL(symmetrize_batch_kernel, dim3((max_nbf + 127) / 128, max_nbf, nmol), dim3(128), 0, st, Jacc,
                       Jmat, Kacc, jmap, fix, J, K, mat_off, mol_nbf);
    return hipGetLastError();
}

hipError_t launch_symmetrize(const fix_t* Jacc, const fix_t* Jmat, const fix_t* Kacc, const int* jmap, const double* fix,
                             double* J, double* K, int nbf, hipStream_t st) {
    hipLaunchKernelGGL(symmetrize_kernel, dim3((nbf + 127) / 128, nbf), dim3(128), 0, st, Jacc, Jmat, Kacc, jmap, fix, J, K,
                       nbf);
    return hipGetLastError();
}

// F = H + J - kfac K  (build_fock, scf/mod.rs:825-881 with kfac = 1/2; hybrid form dft/ks_scf.rs:1960)
__global__ void fock_combine_kernel(const double* __restrict__ H, const fix_t* __restrict__ Jacc,
                                    const fix_t* __restrict__ Jmat,
                                    const fix_t* __restrict__ Kacc, const int* __restrict__ jmap,
                                    const double* __restrict__ fix, double* __restrict__ F, int nbf, double kfac) {
    const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nbf) return;
    const size_t ij = (size_t)i * nbf + j, ji = (size_t)j * nbf + i;
    F[ij] = H[ij] + fix_sym_pairs(Jacc, Jmat, jmap, ij, ji, fix[2]) - kfac * fix_sym(Kacc, ij, ji, fix[3]);
}

hipError_t launch_fock_combine(const double* H, const fix_t* Jacc, const fix_t* Jmat, const fix_t* Kacc, const int* jmap,
                               const double* fix, double* F, int nbf, double kfac, hipStream_t st) {
    hipLaunchKernelGGL(fock_combine_kernel, dim3((nbf + 127) / 128, nbf), dim3(128), 0, st, H, Jacc, Jmat, Kacc, jmap, fix, F,
                       nbf, kfac);
    return hipGetLastError();
}

// Batched Boys F_0..F_m (boys_eval_all, boys/mod.rs:327): one T per lane.
__global__ void boys_batch_kernel(int m, int n, const double* __restrict__ T, double* __restrict__ F,
                                  int* __restrict__ status) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double f[51];
    const int rc = boys_all(m, T[i], f);
    if (rc) {
        atomicOr(status, 1);
        for (int k = 0; k <= m; ++k) F[(size_t)i * (m + 1) + k] = 0.0;
        return;
    }
    for (int k = 0; k <= m; ++k) F[(size_t)i * (m + 1) + k] = f[k];
}

hipError_t launch_boys_batch(int m, int n, const double* T, double* F, int* status, hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL(boys_batch_kernel, dim3((n + 255) / 256), dim3(256), 0, st, m, n, T, F, status);
    return hipGetLastError();
}

// Batched Rys nodes/weights (rys_roots, rys/mod.rs:253): one T per lane.
template <typename R>
__global__ void rys_batch_kernel(int nroots, int n, const R* __restrict__ T, const R* __restrict__ tab,
                                 R* __restrict__ x, R* __restrict__ w) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    R xr[QCG_RYS_NMAX], wr[QCG_RYS_NMAX];
    rys_eval_n<R>(nroots, T[i], tab, xr, wr);
    for (int k = 0; k < nroots; ++k) {
        x[(size_t)i * nroots + k] = xr[k];
        w[(size_t)i * nroots + k] = wr[k];
    }
}

hipError_t launch_rys_batch(int nroots, int n, const double* T, const double* tab, double* x, double* w,
                            hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL((rys_batch_kernel<double>), dim3((n + 255) / 256), dim3(256), 0, st, nroots, n, T, tab, x, w);
    return hipGetLastError();
}

hipError_t launch_rys_batch_f32(int nroots, int n, const float* T, const float* tab, float* x, float* w,
                                hipStream_t st) {
    if (n <= 0) return hipSuccess;
    hipLaunchKernelGGL((rys_batch_kernel<float>), dim3((n + 255) / 256), dim3(256), 0, st, nroots, n, T, tab, x, w);
    return hipGetLastError();
}

}  // namespace qcg
