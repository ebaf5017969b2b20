// One-electron integrals and gradient terms on the device.
//
// Gradient: one thread per (unordered shell pair, primitive pair) and term (blockIdx.y = 0: overlap and
// kinetic; blockIdx.y = 1 + c: attraction to nucleus c), per-atom sums in LDS.  The pairs of a block have
// the same angular momenta (the work list pads each class to whole blocks with si = -1), so the nuclear
// terms, all but 1 / (natom + 1) of the work, run in registers; the block's nucleus is summed over the
// wavefront before it goes to LDS.  Octane 6-31+G*: 1.17 ms for ordered pairs with the
// tables in scratch, 0.11 ms now.
#include "onee_pair.h"
#include "onee_launch.h"

namespace qcg {

__global__ __launch_bounds__(kOneeBlock) void onee_grad_kernel(BasisView B, const int4* __restrict__ work, int nwork,
                                                               const double* __restrict__ D, const double* __restrict__ W,
                                                               const double* __restrict__ rys_tab,
                                                               double* __restrict__ grad) {
    extern __shared__ double gl[];  // natom x 3
    const int n3 = 3 * B.natom;
    for (int i = threadIdx.x; i < n3; i += blockDim.x) gl[i] = 0.0;
    __syncthreads();
    const int4 w0 = work[blockIdx.x * kOneeBlock];  // a block's first entry is never padding
    const int4 w = work[blockIdx.x * kOneeBlock + threadIdx.x];
    auto add = [&](int atom, int x, double v) {
        if (v != 0.0) __hip_atomic_fetch_add(&gl[3 * atom + x], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    const int cnuc = (int)blockIdx.y - 1;
    double gA[3] = {0, 0, 0}, gB[3] = {0, 0, 0};
    if (w.x >= 0) {
        const bool mirror = w.x != w.y;
        switch (pair_class(B.l[w0.x], B.l[w0.y])) {
#define QCG_ONEE(k, la, lb)                                                                                  \
    case k:                                                                                                  \
        if (cnuc < 0) onee_grad_overlap_kinetic<la, lb>(B, w.x, w.y, w.z, w.w, mirror, D, W, gA, gB);        \
        else onee_grad_nuclear<la, lb>(B, w.x, w.y, w.z, w.w, cnuc, mirror, D, rys_tab, gA, gB);             \
        break;
            QCG_ONEE(0, 0, 0) QCG_ONEE(1, 1, 0) QCG_ONEE(2, 1, 1) QCG_ONEE(3, 2, 0) QCG_ONEE(4, 2, 1) QCG_ONEE(5, 2, 2)
#undef QCG_ONEE
        }
    }
    const int atA = w.x >= 0 ? B.shell_atom[w.x] : 0, atB = w.x >= 0 ? B.shell_atom[w.y] : 0;
#pragma unroll
    for (int x = 0; x < 3; ++x) {
        add(atA, x, gA[x]);
        add(atB, x, gB[x]);
        if (cnuc >= 0) {
            double c = -(gA[x] + gB[x]);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) c += __shfl_xor(c, off, 64);
            if ((threadIdx.x & 63) == 0) add(cnuc, x, c);
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < n3; i += blockDim.x)
        if (gl[i] != 0.0) atomicAdd(&grad[i], gl[i]);
}

// S, T, V: one wavefront per Cartesian component pair of the shell pairs si <= sj (work = {si, sj,
// ia, jb}); its lanes take the (primitive pair, term) combinations, term = overlap+kinetic or one
// nucleus, and a fixed-order wavefront reduction sums them.  The wavefront writes its element
// and, off the diagonal blocks, the mirrored one.
__global__ __launch_bounds__(256) void onee_matrix_kernel(BasisView B, const int4* __restrict__ work, int nwork,
                                                         const double* __restrict__ rys_tab, double* __restrict__ S,
                                                         double* __restrict__ T, double* __restrict__ V) {
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (u >= nwork) return;  // the whole wavefront leaves together
    const int4 w = work[u];
    const int nb = B.nprim[w.y], nterm = B.natom + 1;
    const int ncomb = B.nprim[w.x] * nb * nterm;
    double out[3] = {0.0, 0.0, 0.0};
    for (int t = lane; t < ncomb; t += 64) {
        const int pp = t / nterm, c = t - pp * nterm;
        onee_element_term(B, w.x, w.y, w.z, w.w, pp / nb, pp % nb, c == B.natom ? -1 : c, rys_tab, out);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) out[k] += __shfl_xor(out[k], off, 64);
    if (lane != 0) return;
    const double nrm = onee_norm_comp(B.l[w.x], w.z) * onee_norm_comp(B.l[w.y], w.w);
    const int nbf = B.nbf;
    const size_t i = (size_t)B.bf_off[w.x] + w.z, j = (size_t)B.bf_off[w.y] + w.w;
    S[i * nbf + j] = nrm * out[0];
    T[i * nbf + j] = nrm * out[1];
    V[i * nbf + j] = nrm * out[2];
    if (w.x != w.y) {
        S[j * nbf + i] = nrm * out[0];
        T[j * nbf + i] = nrm * out[1];
        V[j * nbf + i] = nrm * out[2];
    }
}

hipError_t launch_onee_matrices(const BasisView& B, const int4* work, int nwork, const double* rys_tab, double* S,
                                double* T, double* V, hipStream_t st) {
    if (nwork <= 0) return hipSuccess;
    hipLaunchKernelGGL(onee_matrix_kernel, dim3((nwork + 3) / 4), dim3(256), 0, st, B, work, nwork, rys_tab, S, T, V);
    return hipGetLastError();
}

hipError_t launch_onee_grad(const BasisView& B, const int4* work, int nwork, const double* D, const double* W,
                            const double* rys_tab, double* grad, hipStream_t st) {
    if (nwork <= 0) return hipSuccess;
    const size_t lds = 3 * (size_t)B.natom * sizeof(double);
    if (lds > 65536) return hipErrorInvalidValue;
    if (B.natom + 1 > 65535) return hipErrorInvalidValue;
    hipLaunchKernelGGL(onee_grad_kernel, dim3(nwork / kOneeBlock, B.natom + 1), dim3(kOneeBlock), lds, st, B, work, nwork, D,
                       W, rys_tab, grad);
    return hipGetLastError();
}

}  // namespace qcg
