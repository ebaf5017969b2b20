// The FP64 grid data of the XC build in packed form: the grid points sorted along a space-filling curve,
// cut into blocks of S consecutive points, and each block keeping only the functions that reach any of
// its points (the others' Phi and grad Phi are exactly zero there, basis_kernel's cut-off).  (H2O)16 on
// 1.05e6 points: a block of 1024 points keeps about 45 % of the 304 functions, so the two grid products
// take a quarter of the dense ones' flops and the arrays a sixth of the bytes; benzene keeps 80 %.
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

// What a kernel needs of a function to make Phi and grad Phi from its shell's radial parts: the centre and
// the axes whose coordinates make its angular part (2 bits each, 3: none).
struct GridFn {
    double cx, cy, cz;
    int axes, pad;
};

// Block b holds functions fl[floff[b] .. + nfn[b]) (shell by shell, sorted by angular momentum: the s
// functions end at nl[2 b], the p functions at nl[2 b + 1]; padded to ld[b], a multiple of 16, with
// function 0, whose packed columns are zero) and, in every packed array, S rows of ld[b] elements from off[b]
// (rows past the last point are zero).  Its partial V is ld[b] x ld[b] from voff[b].
// grad Phi is not kept: rad holds, per point and shell of the block, the radial parts R0 = sum c e and
// R1 = -2 sum c alpha e (e = exp(-alpha r^2)), in rows of ldr[b] (one zero entry after the last shell, which
// the padding columns use) from roff[b]; Phi = ang R0, grad Phi = (grad ang) R0 + (r - A) ang R1.  Two words
// per shell instead of three per function: 20 instead of 57 for a 6-31G* water.
struct PackedGrid {
    int G, S, nblk, nbf, max_ld;
    const int* ld;
    const int* nfn;
    const int64_t* off;
    const int64_t* voff;
    const int* floff;
    const int* fl;
    const int* fs;     // the block's shell of each entry of fl
    const int* ldr;
    const int* nl;
    const int64_t* roff;
    const GridFn* fn;  // by function
    const short* pos;  // nblk x nbf: column of a function in the block, -1 if it has none
    const double *pts, *w;
    const double* phi;
    const double2* rad;
};

// Widest block (functions, padded) of the packed kernels: the density kernel holds the whole row of X in
// the accumulators of two wavefronts (2 x 11 MFMA tiles of 16 columns).
constexpr int kPackedMaxLd = 352;

// out: 3 n coordinates, then n weights, of the points order[0 .. G), zero from G to n
hipError_t launch_packed_points(int G, size_t n, const int* order, const double* pts, const double* w, double* out,
                                hipStream_t st);
// active[b * nshell + s] = 1 if shell s reaches a point of block b
hipError_t launch_packed_active(int G, int S, int nblk, int nshell, const GridShell* shells, const double* pts,
                                unsigned char* active, hipStream_t st);
// Phi and the radial parts of every block; shcol[b * nshell + s]: the shell's first column or -1,
// shrad: its place among the block's shells
hipError_t launch_packed_basis(const PackedGrid& g, int nshell, const GridShell* shells, const double* exps,
                               const double* cn, const short* shcol, const short* shrad, double* phi, double2* rad,
                               hipStream_t st);
// The XC build at density D: aow rows (packed), E_xc added to exc_sum, V_xc symmetrised in V.
// tiles: the V kernel's ntile output tiles (block, first row, first column, width class w = 3, 4 or 5: 32 w
// columns), the widest first; Vparts: partial matrices; Vsum: kPackedVGroups x nbf^2.
constexpr int kPackedVGroups = 32;
hipError_t launch_xc_packed(const PackedGrid& g, const double* D, double* aow, const int4* tiles, int ntile,
                            double* Vparts, double* Vsum, double* V, double* exc_sum, hipStream_t st);
// The XC nuclear gradient at density D, added into grad (natom x 3): X, M (packed work arrays), t (3 per
// row), A rows in aow.  shcol as for launch_packed_basis.
hipError_t launch_xc_grad_packed(const PackedGrid& g, int nshell, int natom, const GridShell* shells, const double* exps,
                                 const double* cn, const short* shcol, const double* D, double* X, double* aow, double* M,
                                 double* t, double* grad, hipStream_t st);
// Output tile width of a block of ld functions, in MFMA tiles per wavefront and dimension (3, 4 or 5)
int packed_v_width(int ld);

}  // namespace qcg
