// The FP64 grid data of the XC build in packed form: the grid points sorted along a space-filling curve,
// cut into blocks of S consecutive points, and each block keeping only the functions that reach any of
// its points (the others' Phi and grad Phi are exactly zero there, basis_kernel's cut-off).  (H2O)16 on
// 1.05e6 points: a block of 1024 points keeps about 45 % of the 304 functions, so the two grid products
// take a fifth to a quarter of the dense ones' flops and the arrays 45 % of the bytes; benzene keeps 80 %.
#pragma once
#include "qcg_common.h"

namespace qcg {

struct GridShell {
    double cx, cy, cz, amin;  // centre, smallest exponent (screening)
    int l, nprim, poff, bf;
    int atom, pad;
};

// GAUSSIAN_SCREENING_THRESHOLD (orbital/grid.rs:174): a shell is zero where amin r^2 is above it
constexpr double kGridCut = 34.5388;

// Block b holds functions fl[floff[b] .. + nfn[b]) (ascending; padded to ld[b], a multiple of 16, with
// function 0, whose packed columns are zero) and, in every packed array, S rows of ld[b] elements from off[b]
// (rows past the last point are zero).  Its partial V is ld[b] x ld[b] from voff[b].
struct PackedGrid {
    int G, S, nblk, nbf, max_ld;
    const int* ld;
    const int* nfn;
    const int64_t* off;
    const int64_t* voff;
    const int* floff;
    const int* fl;
    const short* pos;  // nblk x nbf: column of a function in the block, -1 if it has none
    const double *pts, *w;
    const double *phi, *dpx, *dpy, *dpz;
};

// Widest block (functions, padded) of the packed kernels: the density kernel holds the whole row of X in
// the accumulators of two wavefronts (2 x 11 MFMA tiles of 16 columns).
constexpr int kPackedMaxLd = 352;

// active[b * nshell + s] = 1 if shell s reaches a point of block b
hipError_t launch_packed_active(int G, int S, int nblk, int nshell, const GridShell* shells, const double* pts,
                                unsigned char* active, hipStream_t st);
// Phi and grad Phi of every block; shcol[b * nshell + s]: the shell's first column or -1
hipError_t launch_packed_basis(const PackedGrid& g, int nshell, const GridShell* shells, const double* exps,
                               const double* cn, const short* shcol, double* phi, double* dpx, double* dpy, double* dpz,
                               hipStream_t st);
// The XC build at density D: aow rows (packed), E_xc added to exc_sum, V_xc symmetrised in V.
// tiles: the V kernel's output tiles (block, first row, first column) sorted by width, ntile[w - 3] of
// width class w = 3, 4, 5 (32 w columns); Vparts: partial matrices; Vsum: kPackedVGroups x nbf^2.
constexpr int kPackedVGroups = 32;
hipError_t launch_xc_packed(const PackedGrid& g, const double* D, double* aow, const int4* tiles, const int ntile[3],
                            double* Vparts, double* Vsum, double* V, double* exc_sum, hipStream_t st);
// The XC nuclear gradient at density D, added into grad (natom x 3): X, M (packed work arrays), t (3 per
// row), A rows in aow.  shcol as for launch_packed_basis.
hipError_t launch_xc_grad_packed(const PackedGrid& g, int nshell, int natom, const GridShell* shells, const double* exps,
                                 const double* cn, const short* shcol, const double* D, double* X, double* aow, double* M,
                                 double* t, double* grad, hipStream_t st);
// Output tile width of a block of ld functions, in MFMA tiles per wavefront and dimension (3, 4 or 5)
int packed_v_width(int ld);

}  // namespace qcg
