// Grid contractions of the XC build on the matrix cores (MFMA), element type T = float (mixed
// precision) or double:
//   xc_rho_kernel : X = Phi D one 64-point block at a time on MFMA, reduced on the fly into rho and
//                   grad rho (X never goes to HBM), then B3LYP per point (FP64), the aow rows and
//                   E_xc -- the work of compute_density_and_gradient_matmul and the point part of
//                   build_vxc_gga_matmul (dft/ks_scf.rs:1028-1093, :1150-1296) in one kernel;
//   xc_rho_all_kernel : the same for nbf <= 352 with X for all columns held per wavefront, so Phi is read
//                   once per K step instead of once per column pass;
//   xc_rho_packed_kernel, xc_v_packed_kernel : the FP64 build on the packed grid (xc_packed.h);
//   xc_v_kernel   : V = Phi^T aow as 128x128 output tiles over grid chunks (split K), one partial
//                   matrix per chunk, summed and symmetrised afterwards (sum_parts, sym_half).
// rho, grad rho, E_xc and the functional are accumulated in FP64 whatever T is; with T = float the
// GEMM products are FP32 MFMA with FP32 accumulation.
#include "xc_functional.h"
#include "xc_launch.h"

namespace qcg {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef double f64x4_t __attribute__((ext_vector_type(4)));

// v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64: D (16x16) += A (16x4) B (4x16).  Lane l supplies
// A[l % 16][l / 16] and B[l / 16][l % 16] and holds D[row(l / 16, r)][l % 16] in element r, with
// row = 4 (l / 16) + r for FP32 and (l / 16) + 4 r for FP64 (both checked on the device).
template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
    using acc = f32x4_t;
    static __device__ __forceinline__ acc mma(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};
template <>
struct Mfma<double> {
    using acc = f64x4_t;
    static __device__ __forceinline__ acc mma(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};

constexpr int kRhoMT = 1;                 // MFMA row tiles (16 points each) per wavefront
constexpr int kRhoBM = 4 * 16 * kRhoMT;   // grid points per block
constexpr int kRhoPW = 16 * kRhoMT;       // grid points per wavefront
constexpr int kRhoBK = 16;                // basis functions per K step
constexpr int kPad = 16;                  // LDS row padding: the lanes of a fragment row hit distinct banks
// V: VW MFMA tiles per wavefront and dimension (xc_v_width, 3 to 5), so the block's output tile
// (2 x 2 wavefronts) is 32 VW square
constexpr int kVBK = 16;                  // grid points per K step

// NT: MFMA column tiles (16 columns each) of X per pass over the columns; a pass covers 16 NT
// columns, all passes together the nbf columns of X.  Each wavefront owns kRhoPW points (kRhoMT
// row tiles), so every D fragment read from LDS feeds kRhoMT MFMAs.
// Phi, dPhi/dx, dPhi/dy, dPhi/dz at (point g, function mu) = element idx = g nbf + mu: FP32 from
// one interleaved float4 array (one 16-byte load), FP64 from the four separate arrays.
template <typename T>
struct GridVals {
    const T *phi, *dpx, *dpy, *dpz;
    const float4* g4;
    __device__ __forceinline__ void get(size_t idx, double& f, double& x, double& y, double& z) const {
        if constexpr (sizeof(T) == 4) {
            const float4 v = g4[idx];
            f = v.x; x = v.y; y = v.z; z = v.w;
        } else {
            f = phi[idx]; x = dpx[idx]; y = dpy[idx]; z = dpz[idx];
        }
    }
};

// LDS row padding that makes a fragment read conflict-free: the four rows l / 16 of one read start
// 16 elements apart modulo the bank width (32 doubles or 64 floats), so with 16 consecutive
// elements per row the 64 lanes cover the banks evenly.
template <typename T>
constexpr int lds_pad(int n) {
    return sizeof(T) == 8 ? (16 - n % 32 + 32) % 32 : (16 - n % 64 + 64) % 64;
}

// The density kernels of 512 threads are compiled for four waves per SIMD (two blocks per CU, at most
// 128 VGPRs).
#define QCG_XC_RHO_ATTR __attribute__((amdgpu_waves_per_eu(4)))

// Most MFMA column tiles the all-columns kernel holds (nbf <= 352): D rows of one K step, all
// columns, stay within the 64 KB of static LDS per block.
constexpr int kRhoAllMaxNT = 22;
// From more column tiles than this on it leaves out the zero ones (octane 6-31G, 7 tiles: 313 us without, 317
// with; (H2O)16, 19 tiles: see the kernel).
constexpr int kRhoMaskNT = 12;

// The functional (B3LYP, FP64) at the block's 64 points, whose rho and grad rho sums are in red[row tile]
// [point]: coef = w vrho, 4 w vsigma grad rho; returns the point's E_xc (wavefronts 0 to 3).
// tgrad: instead w vrho and 2 w vsigma grad rho, the latter also in tgrad (three per point).
__device__ __forceinline__ double xc_point_coef(int G, int wv, int l, int g0, const double* __restrict__ w,
                                                double (*red)[kRhoPW][4], double (*coef)[kRhoPW][4], bool half,
                                                double* __restrict__ tgrad) {
    const int rt = wv & 3, gw = g0 + kRhoPW * rt;
    double contrib = 0.0;
    if (wv < 4 && l < kRhoPW) {
        const int g = gw + l;
        double c0 = 0.0, c1 = 0.0, c2 = 0.0, c3 = 0.0;
        if (g < G) {
            const double rho = fmax(red[rt][l][0], 0.0);
            const double grx = 2.0 * red[rt][l][1], gry = 2.0 * red[rt][l][2], grz = 2.0 * red[rt][l][3];
            double exc, vrho, vsig;
            xc_b3lyp(rho, grx * grx + gry * gry + grz * grz, exc, vrho, vsig);
            const double wg = w[g], f4 = (half ? 2.0 : 4.0) * wg * vsig;
            c0 = wg * vrho;
            c1 = f4 * grx;
            c2 = f4 * gry;
            c3 = f4 * grz;
            contrib = wg * exc * rho;
        }
        coef[rt][l][0] = c0;
        coef[rt][l][1] = c1;
        coef[rt][l][2] = c2;
        coef[rt][l][3] = c3;
        if (tgrad) {
            tgrad[3 * (size_t)g] = c1;
            tgrad[3 * (size_t)g + 1] = c2;
            tgrad[3 * (size_t)g + 2] = c3;
        }
    }
    return contrib;
}
// E_xc of the block: part is four doubles of LDS.
__device__ __forceinline__ void xc_point_exc(double contrib, int wv, int l, double* __restrict__ exc_sum, double* part) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) contrib += __shfl_xor(contrib, off, 64);
    if (l == 0 && wv < 4) part[wv] = contrib;
    __syncthreads();
    if (wv == 0 && l == 0) {
        const double s = part[0] + part[1] + part[2] + part[3];
        if (s != 0.0) atomicAdd(exc_sum, s);
    }
}

// The point part shared by both rho kernels, once the rho and grad rho sums of the block's 64 points
// are in red[row tile][point]: B3LYP per point (FP64), the aow rows, E_xc.  NW wavefronts per block
// (4 or 8); wavefront wv works on row tile wv % 4, and with 8 wavefronts each takes half its rows
// in the aow pass.
template <typename T, int NW, int MAXC = 0>
__device__ __forceinline__ void xc_point_tail(int G, int nbf, int wv, int l, int g0, const double* __restrict__ w,
                                              const GridVals<T>& gv, T* __restrict__ aow, double* __restrict__ exc_sum,
                                              double (*red)[kRhoPW][4], double (*coef)[kRhoPW][4], double* part,
                                              unsigned tiles = ~0u) {
    static_assert(NW == 4 || NW == 8, "four or eight wavefronts per block");
    const int rt = wv & 3, gw = g0 + kRhoPW * rt;
    const double contrib = xc_point_coef(G, wv, l, g0, w, red, coef, false, nullptr);
    __syncthreads();
    // aow = w vrho Phi + 4 w vsigma (grad rho . grad Phi), row by row of the wavefront's points
    constexpr int kRows = kRhoPW / (NW / 4);
    const int p0 = (wv >> 2) * kRows;
    for (int p = p0; p < p0 + kRows; ++p) {
        const int g = gw + p;
        if (g >= G) break;  // uniform over the wavefront
        const double c0 = coef[rt][p][0], c1 = coef[rt][p][1], c2 = coef[rt][p][2], c3 = coef[rt][p][3];
        const size_t row = (size_t)g * nbf;
        if constexpr (MAXC > 0) {
            // nbf <= 64 MAXC: the row's loads all in flight before the first use (unconditional, at
            // columns clamped into the basis, so none waits inside a branch of its own); the lanes of
            // column tiles that are zero at these points (not in `tiles`) read the row's first element
            double f[MAXC], dx[MAXC], dy[MAXC], dz[MAXC];
#pragma unroll
            for (int i = 0; i < MAXC; ++i) {
                const int col = min(l + 64 * i, nbf - 1);
                gv.get(row + ((tiles >> (col >> 4)) & 1 ? col : 0), f[i], dx[i], dy[i], dz[i]);
            }
#pragma unroll
            for (int i = 0; i < MAXC; ++i)
                if (l + 64 * i < nbf)
                    aow[row + l + 64 * i] = (tiles >> ((l + 64 * i) >> 4)) & 1
                                                ? (T)(c0 * f[i] + c1 * dx[i] + c2 * dy[i] + c3 * dz[i]) : T(0);
        } else {
            for (int col = l; col < nbf; col += 64) {
                double f, dx, dy, dz;
                gv.get(row + col, f, dx, dy, dz);
                aow[row + col] = (T)(c0 * f + c1 * dx + c2 * dy + c3 * dz);
            }
        }
    }
    xc_point_exc(contrib, wv, l, exc_sum, part);
}

template <typename T, int NT>
__global__ __launch_bounds__(256) void xc_rho_kernel(int G, int nbf, const double* __restrict__ w,
                                                     const T* __restrict__ phi, const GridVals<T> gv,
                                                     const T* __restrict__ Dm, T* __restrict__ aow,
                                                     double* __restrict__ exc_sum) {
    using M = Mfma<T>;
    using acc_t = typename M::acc;
    constexpr int BN = 16 * NT;
    constexpr int NA = kRhoBM * kRhoBK / 256, NB = kRhoBK * BN / 256;  // staged elements per thread
    static_assert(kRhoBM * kRhoBK % 256 == 0 && kRhoBK * BN % 256 == 0, "tile sizes");
    __shared__ T As[kRhoBK][kRhoBM + kPad];  // Phi block, transposed: As[k][point]
    __shared__ T Bs[kRhoBK][BN + kPad];      // rows k0.. of D, this pass's columns
    __shared__ double red[4][kRhoPW][4];     // per wavefront and point: rho, d rho / dx, dy, dz sums
    __shared__ double coef[4][kRhoPW][4];    // per wavefront and point: w vrho, 4 w vsigma grad rho
    __shared__ double part[4];
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
    const int g0 = blockIdx.x * kRhoBM, gw = g0 + kRhoPW * wv;
    double rs[kRhoMT][4], xs[kRhoMT][4], ys[kRhoMT][4], zs[kRhoMT][4];
#pragma unroll
    for (int m = 0; m < kRhoMT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) rs[m][r] = xs[m][r] = ys[m][r] = zs[m][r] = 0.0;
    T ra[NA], rb[NB];  // next K step's tiles, loaded while the current one is multiplied
    auto load = [&](int n0, int k0) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int e = tid + 256 * i, r = e / kRhoBK, c = e % kRhoBK, g = g0 + r, k = k0 + c;
            ra[i] = (g < G && k < nbf) ? phi[(size_t)g * nbf + k] : T(0);
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int e = tid + 256 * i, r = e / BN, c = e % BN, k = k0 + r, n = n0 + c;
            rb[i] = (k < nbf && n < nbf) ? Dm[(size_t)k * nbf + n] : T(0);
        }
    };
    for (int n0 = 0; n0 < nbf; n0 += BN) {
        acc_t acc[kRhoMT][NT];
#pragma unroll
        for (int m = 0; m < kRhoMT; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[m][t] = acc_t{T(0), T(0), T(0), T(0)};
        load(n0, 0);
        for (int k0 = 0; k0 < nbf; k0 += kRhoBK) {
            __syncthreads();  // the previous step's fragment reads are done
#pragma unroll
            for (int i = 0; i < NA; ++i) {
                const int e = tid + 256 * i;
                As[e % kRhoBK][e / kRhoBK] = ra[i];
            }
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int e = tid + 256 * i;
                Bs[e / BN][e % BN] = rb[i];
            }
            __syncthreads();
            if (k0 + kRhoBK < nbf) load(n0, k0 + kRhoBK);
#pragma unroll
            for (int ks = 0; ks < kRhoBK; ks += 4) {
                T a[kRhoMT];
#pragma unroll
                for (int m = 0; m < kRhoMT; ++m) a[m] = As[ks + lk][kRhoPW * wv + 16 * m + li];
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const T b = Bs[ks + lk][16 * t + li];
#pragma unroll
                    for (int m = 0; m < kRhoMT; ++m) acc[m][t] = M::mma(a[m], b, acc[m][t]);
                }
            }
        }
        // rho = sum_mu X Phi, grad rho / 2 = sum_mu X grad Phi over this pass's columns
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int col = n0 + 16 * t + li;
            if (col < nbf) {
#pragma unroll
                for (int m = 0; m < kRhoMT; ++m)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int g = gw + 16 * m + M::row(lk, r);
                        if (g < G) {
                            double f, dx, dy, dz;
                            gv.get((size_t)g * nbf + col, f, dx, dy, dz);
                            const double x = (double)acc[m][t][r];
                            rs[m][r] += x * f;
                            xs[m][r] += x * dx;
                            ys[m][r] += x * dy;
                            zs[m][r] += x * dz;
                        }
                    }
            }
            // one tile's loads in flight at a time: hoisting all of them costs hundreds of VGPRs
            asm volatile("" ::: "memory");
        }
    }
    // sums over the 16 lanes that share a point row (same l / 16)
#pragma unroll
    for (int m = 0; m < kRhoMT; ++m)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
            for (int off = 1; off < 16; off <<= 1) {
                rs[m][r] += __shfl_xor(rs[m][r], off, 64);
                xs[m][r] += __shfl_xor(xs[m][r], off, 64);
                ys[m][r] += __shfl_xor(ys[m][r], off, 64);
                zs[m][r] += __shfl_xor(zs[m][r], off, 64);
            }
        }
    if (li == 0) {
#pragma unroll
        for (int m = 0; m < kRhoMT; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = 16 * m + M::row(lk, r);
                red[wv][p][0] = rs[m][r];
                red[wv][p][1] = xs[m][r];
                red[wv][p][2] = ys[m][r];
                red[wv][p][3] = zs[m][r];
            }
    }
    __syncthreads();
    xc_point_tail<T, 4>(G, nbf, wv, l, g0, w, gv, aow, exc_sum, red, coef, part);
}

// All-columns form of xc_rho_kernel for nbf <= 16 kRhoAllMaxNT, eight wavefronts per block of 64
// points: wavefront wv keeps the X tile of the 16 points of row tile wv % 4 for column half wv / 4
// (NH = ceil(NT / 2) MFMA column tiles, one accumulator each), so Phi is read from HBM once per K
// step instead of once per column pass; D rows k0..k0+15 (all columns) are staged in LDS per K step
// (D stays L2-resident: every block reads all of it).
// FP64 products run here in a build that is captured on a grid made for the mixed option (xc_build); they
// stage D without the look-ahead, whose registers would cost the second block per CU ((H2O)16, 1.05e6 points:
// 11.2 -> 9.3 ms), and take no mask.
// mask (FP32, more than kRhoMaskNT tiles): per 16 points the tiles of 16 functions that reach one of them
// (tile_mask_kernel).  K steps that are zero at all 64 points are not staged, and a wavefront multiplies only
// the K steps and column tiles that its 16 points see: what is left out are exact zeros, so every sum keeps
// its bits.  (H2O)16, 1.05e6 points, FP32: 2.97 -> 2.50 ms.  (The
// same in xc_v_kernel: 1.88 -> 3.44 ms, the scan for the next step and the registers cost more.)
template <typename T, int NT>
__global__ __launch_bounds__(512) QCG_XC_RHO_ATTR void xc_rho_all_kernel(int G, int nbf, const double* __restrict__ w,
                                                         const T* __restrict__ phi, const GridVals<T> gv,
                                                         const T* __restrict__ Dm, T* __restrict__ aow,
                                                         double* __restrict__ exc_sum, const unsigned* __restrict__ mask) {
    using M = Mfma<T>;
    using acc_t = typename M::acc;
    static_assert(NT < 32, "one mask word");
    constexpr int NH = (NT + 1) / 2, BN = 16 * NT, SA = kRhoBM + lds_pad<T>(kRhoBM);
    // Bs row stride: padded for conflict-free fragment reads, and Bs large enough to hold red2 after
    // the K loop (2 x 4 x 16 x 4 doubles)
    constexpr int SB0 = BN + lds_pad<T>(BN), SBM = 4096 / (kRhoBK * (int)sizeof(T));
    constexpr int SB = SB0 >= SBM ? SB0 : SBM;
    constexpr int NA = kRhoBM * kRhoBK / 512;  // Phi elements staged per thread and K step
    static_assert(kRhoMT == 1 && kRhoBM == 64 && NA * 512 == kRhoBM * kRhoBK, "one 16-point row tile per wavefront");
    __shared__ T As[kRhoBK][SA];  // Phi block, transposed: As[k][point]
    __shared__ T Bs[kRhoBK][SB];  // D rows k0 .. k0 + 15, all columns
    __shared__ double red[4][kRhoPW][4];
    __shared__ double coef[4][kRhoPW][4];
    __shared__ double part[4];
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
    const int rt = wv & 3, half = wv >> 2, t0 = half * NH;
    const int g0 = blockIdx.x * kRhoBM, gw = g0 + kRhoPW * rt;
    acc_t acc[NH];
#pragma unroll
    for (int t = 0; t < NH; ++t) acc[t] = acc_t{T(0), T(0), T(0), T(0)};
    // next K step's Phi (FP32: and D) elements, loaded while the current step is multiplied
    constexpr bool kAheadD = sizeof(T) == 4, kMask = sizeof(T) == 4 && NT > kRhoMaskNT;
    constexpr int NBD = (kRhoBK * BN + 511) / 512;
    T ra[NA], rb[kAheadD ? NBD : 1];
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int e = tid + 512 * i, r = e / kRhoBK, c = e % kRhoBK, g = g0 + r, k = k0 + c;
            ra[i] = (g < G && k < nbf) ? phi[(size_t)g * nbf + k] : T(0);
        }
        if constexpr (kAheadD) {
#pragma unroll
            for (int i = 0; i < NBD; ++i) {
                const int e = tid + 512 * i, r = e / BN, c = e - r * BN, k = k0 + r;
                rb[i] = (e < kRhoBK * BN && k < nbf && c < nbf) ? Dm[(size_t)k * nbf + c] : T(0);
            }
        }
    };
    static_assert(kRhoBK == 16, "a K step is a tile of the mask");
    unsigned wm = (1u << NT) - 1, left = wm;  // the wavefront's tiles; the block's K steps still to do
    if constexpr (kMask) {
        const unsigned* mk = mask + 4 * (size_t)blockIdx.x;
        wm = __builtin_amdgcn_readfirstlane(mk[rt]);
        left = __builtin_amdgcn_readfirstlane(mk[0] | mk[1] | mk[2] | mk[3]);
    }
    const auto on = [wm](int t) { return !kMask || ((wm >> t) & 1); };
    if (left) load(kRhoBK * __builtin_ctz(left));
    for (; left; left &= left - 1) {
        const int kt = __builtin_ctz(left);
        __syncthreads();  // the previous step's fragment reads are done
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int e = tid + 512 * i;
            As[e % kRhoBK][e / kRhoBK] = ra[i];
        }
        if constexpr (kAheadD) {
#pragma unroll
            for (int i = 0; i < NBD; ++i) {
                const int e = tid + 512 * i, r = e / BN, c = e - r * BN;
                if (e < kRhoBK * BN) Bs[r][c] = rb[i];
            }
        } else {
            for (int e = tid; e < kRhoBK * BN; e += 512) {
                const int r = e / BN, c = e - r * BN, k = kRhoBK * kt + r;
                Bs[r][c] = (k < nbf && c < nbf) ? Dm[(size_t)k * nbf + c] : T(0);
            }
        }
        __syncthreads();
        if (left & (left - 1)) load(kRhoBK * __builtin_ctz(left & (left - 1)));
        if (!on(kt)) continue;
        // two k sub-steps per unrolled body: all four hoist 4 NH fragment reads (spills at NH = 8)
#pragma unroll 2
        for (int ks = 0; ks < kRhoBK; ks += 4) {
            const T a = As[ks + lk][kRhoPW * rt + li];
#pragma unroll
            for (int t = 0; t < NH; ++t)
                if (t0 + t < NT && on(t0 + t)) acc[t] = M::mma(a, Bs[ks + lk][16 * (t0 + t) + li], acc[t]);
        }
    }
    // rho = sum_mu X Phi, grad rho / 2 = sum_mu X grad Phi over this half's columns
    double rs[4] = {}, xs[4] = {}, ys[4] = {}, zs[4] = {};
#pragma unroll
    for (int t = 0; t < NH; ++t) {
        if (!on(t0 + t)) continue;
        // the tile's loads are unconditional, at addresses clamped into the grid and the basis (X is
        // zero outside them, and the product is masked too), so the four rows' loads issue back to
        // back instead of each waiting inside its own branch: (H2O)16 XC, mixed 5.78 -> 5.41 ms,
        // FP64 products 14.25 -> 12.49 ms
        const int col = 16 * (t0 + t) + li;
        const bool cin = col < nbf;
        const int cc = cin ? col : nbf - 1;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int g = gw + M::row(lk, r);
            double f, dx, dy, dz;
            gv.get((size_t)(g < G ? g : G - 1) * nbf + cc, f, dx, dy, dz);
            const double x = (cin && g < G) ? (double)acc[t][r] : 0.0;
            rs[r] += x * f;
            xs[r] += x * dx;
            ys[r] += x * dy;
            zs[r] += x * dz;
        }
        // one tile's loads in flight at a time: hoisting all of them costs hundreds of VGPRs
        asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) {
            rs[r] += __shfl_xor(rs[r], off, 64);
            xs[r] += __shfl_xor(xs[r], off, 64);
            ys[r] += __shfl_xor(ys[r], off, 64);
            zs[r] += __shfl_xor(zs[r], off, 64);
        }
    }
    // per column half, row tile and point: rho, grad rho sums, in the D staging area (free now)
    static_assert(sizeof(Bs) >= 2 * 4 * kRhoPW * 4 * sizeof(double), "red2 fits in Bs");
    auto red2 = reinterpret_cast<double (*)[4][kRhoPW][4]>(&Bs[0][0]);
    __syncthreads();  // every wavefront's last fragment reads are done
    if (li == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int p = M::row(lk, r);
            red2[half][rt][p][0] = rs[r];
            red2[half][rt][p][1] = xs[r];
            red2[half][rt][p][2] = ys[r];
            red2[half][rt][p][3] = zs[r];
        }
    }
    __syncthreads();
    // the two column halves, in a fixed order
    if (tid < 4 * kRhoPW * 4) {
        const int q = tid & 3, p = (tid >> 2) % kRhoPW, r4 = tid / (4 * kRhoPW);
        red[r4][p][q] = red2[0][r4][p][q] + red2[1][r4][p][q];
    }
    __syncthreads();
    xc_point_tail<T, 8, (16 * NT + 63) / 64>(G, nbf, wv, l, g0, w, gv, aow, exc_sum, red, coef, part, kMask ? wm : ~0u);
}

// One wavefront per 16 points, four lanes to a point: the tiles of 16 functions of the shells that reach one of the points
// (basis_kernel's cut-off, with room for another rounding of it).  From the points and shells instead of the 16 nbf
// bytes per point of the arrays: the first mixed build on a grid of (H2O)16, 286081 points, 3.20 -> 2.97 ms
// (3.04 ms before there was a mask), the same bits of V.
__global__ __launch_bounds__(256) void tile_mask_kernel(int G, int nshell, int n, const GridShell* __restrict__ shells,
                                                        const double* __restrict__ pts, unsigned* __restrict__ mask) {
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (i >= n) return;
    const size_t p = 16 * (size_t)i + (lane & 15);
    unsigned m = 0;
    if (p < (size_t)G) {
        const double x = pts[3 * p], y = pts[3 * p + 1], z = pts[3 * p + 2];
        for (int s = lane >> 4; s < nshell; s += 4) {
            const double dx = x - shells[s].cx, dy = y - shells[s].cy, dz = z - shells[s].cz;
            const int f = shells[s].bf;
            if (!(shells[s].amin * (dx * dx + dy * dy + dz * dz) > kGridCut * (1.0 + 1e-12)))
                m |= 1u << (f >> 4) | 1u << ((f + ncart(shells[s].l) - 1) >> 4);
        }
    }
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) m |= __shfl_xor(m, off, 64);
    if (lane == 0) mask[i] = m;
}

size_t xc_tile_mask_words(int G, int nbf) {
    const int tiles = (nbf + 15) / 16;
    return tiles > kRhoMaskNT && tiles <= kRhoAllMaxNT ? 4 * ((size_t)(G + 63) / 64) + 4 : 0;
}

hipError_t launch_tile_mask(int G, int nbf, int nshell, const GridShell* shells, const double* pts, unsigned* mask,
                            hipStream_t st) {
    const int n = (int)xc_tile_mask_words(G, nbf);
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(tile_mask_kernel, dim3((n + 3) / 4), dim3(256), 0, st, G, nshell, n, shells, pts, mask);
    return hipGetLastError();
}

// Vparts[chunk] = Phi[chunk rows]^T aow[chunk rows] by 32 VW square output tiles (each wavefront a
// 16 VW square quarter: every fragment read feeds VW MFMAs); block -> (chunk, tile) so that the
// tiles of one chunk share an XCD (blocks are dealt round-robin over the 8 XCDs) and reuse its Phi
// and aow rows from that XCD's L2.
template <typename T, int VW>
__global__ __launch_bounds__(256) void xc_v_kernel(int G, int nbf, int ntile, int nchunk, int chunk,
                                                   const T* __restrict__ phi, const T* __restrict__ aow,
                                                   double* __restrict__ Vparts) {
    using M = Mfma<T>;
    using acc_t = typename M::acc;
    constexpr int kVW = VW, kVBM = 32 * VW;
    static_assert(kVBK * kVBM % 256 == 0, "whole elements per thread in the staging");
    __shared__ T As[kVBK][kVBM + kPad];  // Phi[g][m0 + i]
    __shared__ T Bs[kVBK][kVBM + kPad];  // aow[g][n0 + j]
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
    const int wr = wv >> 1, wc = wv & 1;  // this wavefront's quarter of the tile
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, nt2 = ntile * ntile;
    const int ch = (slot / nt2) * 8 + xcd, tile = slot % nt2;
    if (ch >= nchunk) return;  // the whole block: before any barrier
    const int m0 = (tile / ntile) * kVBM, n0 = (tile % ntile) * kVBM;
    const int gb = ch * chunk, ge = min(G, gb + chunk);
    acc_t acc[kVW][kVW];
#pragma unroll
    for (int i = 0; i < kVW; ++i)
#pragma unroll
        for (int j = 0; j < kVW; ++j) acc[i][j] = acc_t{T(0), T(0), T(0), T(0)};
    constexpr int NE = kVBK * kVBM / 256;  // staged elements per thread and operand
    T ra[NE], rb[NE];                       // next K step's rows, loaded during the current MFMAs
    auto load = [&](int k0) {
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int e = tid + 256 * i, r = e / kVBM, c = e % kVBM, g = k0 + r;
            const bool in = g < ge;
            ra[i] = (in && m0 + c < nbf) ? phi[(size_t)g * nbf + m0 + c] : T(0);
            rb[i] = (in && n0 + c < nbf) ? aow[(size_t)g * nbf + n0 + c] : T(0);
        }
    };
    load(gb);
    for (int k0 = gb; k0 < ge; k0 += kVBK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NE; ++i) {
            const int e = tid + 256 * i;
            As[e / kVBM][e % kVBM] = ra[i];
            Bs[e / kVBM][e % kVBM] = rb[i];
        }
        __syncthreads();
        if (k0 + kVBK < ge) load(k0 + kVBK);
#pragma unroll
        for (int ks = 0; ks < kVBK; ks += 4) {
            T a[kVW], b[kVW];
#pragma unroll
            for (int i = 0; i < kVW; ++i) {
                a[i] = As[ks + lk][16 * kVW * wr + 16 * i + li];
                b[i] = Bs[ks + lk][16 * kVW * wc + 16 * i + li];
            }
            // 16 x 16 sub-tiles wholly past nbf (the edge tiles of the 128 x 128 grid) are skipped:
            // for nbf = 304 that is 37 % of the products; the condition is uniform per wavefront
#pragma unroll
            for (int i = 0; i < kVW; ++i)
#pragma unroll
                for (int j = 0; j < kVW; ++j)
                    if (m0 + 16 * kVW * wr + 16 * i < nbf && n0 + 16 * kVW * wc + 16 * j < nbf)
                        acc[i][j] = M::mma(a[i], b[j], acc[i][j]);
        }
    }
    double* out = Vparts + (size_t)ch * nbf * nbf;
#pragma unroll
    for (int i = 0; i < kVW; ++i)
#pragma unroll
        for (int j = 0; j < kVW; ++j) {
            const int col = n0 + 16 * kVW * wc + 16 * j + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + 16 * kVW * wr + 16 * i + M::row(lk, r);
                if (row < nbf && col < nbf) out[(size_t)row * nbf + col] = (double)acc[i][j][r];
            }
        }
}

// FP64 correction of E_xc for the rounding of D to FP32: dE_xc/dD = V_xc, so
// E_xc(D) = E_xc(D32) + sum V_xc (D - D32) + O(|D - D32|^2) with |D - D32| ~ 6e-8 |D|.
__global__ __launch_bounds__(256) void exc_d32_correction_kernel(const double* __restrict__ V,
                                                                 const double* __restrict__ D,
                                                                 const float* __restrict__ D32, size_t n,
                                                                 double* __restrict__ exc_sum) {
    __shared__ double part[4];
    double s = 0.0;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        s += V[i] * (D[i] - (double)D32[i]);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) s += __shfl_xor(s, off, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        const double t = part[0] + part[1] + part[2] + part[3];
        if (t != 0.0) atomicAdd(exc_sum, t);
    }
}

hipError_t launch_exc_d32_correction(const double* V, const double* D, const float* D32, size_t n, double* exc_sum,
                                     hipStream_t st) {
    if (n == 0) return hipSuccess;
    const unsigned blocks = (unsigned)std::min<size_t>(256, (n + 255) / 256);
    hipLaunchKernelGGL(exc_d32_correction_kernel, dim3(blocks), dim3(256), 0, st, V, D, D32, n, exc_sum);
    return hipGetLastError();
}

__global__ void to_f32x4_kernel(const double* __restrict__ a, const double* __restrict__ b,
                                const double* __restrict__ c, const double* __restrict__ d, float4* __restrict__ out,
                                size_t n) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) out[i] = make_float4((float)a[i], (float)b[i], (float)c[i], (float)d[i]);
}

hipError_t launch_to_f32x4(const double* a, const double* b, const double* c, const double* d, float4* out, size_t n,
                           hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(to_f32x4_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a, b, c, d, out, n);
    return hipGetLastError();
}

__global__ void to_f32_kernel(const double* __restrict__ in, float* __restrict__ out, size_t n) {
    const size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x;
    if (i < n) out[i] = (float)in[i];
}

hipError_t launch_to_f32(const double* in, float* out, size_t n, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(to_f32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, in, out, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------- packed FP64 form (xc_packed.h)
// Functions of angular momentum up to L at a point without branches: the angular part is 1, u or n u v with
// u and v the coordinates along the function's axes (meta: bits 0-1 and 2-3; L below the function's own
// never asked for; axis 3 stands for the constant 1) and n the norm of the d components x^2, y^2, z^2.
template <int L>
struct FnAt {
    double cx, cy, cz, n;
    int shell;
    double a[3], b[3], a1, b1;  // unit vectors of the axes, and 1 for the constant
    __device__ __forceinline__ FnAt(double x, double y, double z, int meta) : cx(x), cy(y), cz(z), shell(meta >> 4) {
        const int i = meta & 3, j = (meta >> 2) & 3;
        if constexpr (L >= 1) {
#pragma unroll
            for (int k = 0; k < 3; ++k) a[k] = i == k ? 1.0 : 0.0;
            a1 = i == 3 ? 1.0 : 0.0;
        }
        if constexpr (L >= 2) {
            n = i == j && i < 3 ? 0.57735026918962576451 : 1.0;
#pragma unroll
            for (int k = 0; k < 3; ++k) b[k] = j == k ? 1.0 : 0.0;
            b1 = j == 3 ? 1.0 : 0.0;
        }
    }
    __device__ __forceinline__ void angular(double x, double y, double z, double& ang, double& ax, double& ay,
                                            double& az) const {
        if constexpr (L == 0) {
            ang = 1.0;
            ax = ay = az = 0.0;
        } else {
            const double u = a1 + a[0] * x + a[1] * y + a[2] * z;
            if constexpr (L == 1) {
                ang = u;
                ax = a[0];
                ay = a[1];
                az = a[2];
            } else {
                const double v = b1 + b[0] * x + b[1] * y + b[2] * z, nu = n * u, nv = n * v;
                ang = nu * v;
                ax = nv * a[0] + nu * b[0];
                ay = nv * a[1] + nu * b[1];
                az = nv * a[2] + nu * b[2];
            }
        }
    }
    // adds f * (Phi, grad Phi) into s
    __device__ __forceinline__ void add(double x, double y, double z, const double2 R, double f, double (&s)[4]) const {
        double ang, ax, ay, az;
        angular(x, y, z, ang, ax, ay, az);
        const double v0 = f * R.x;
        if constexpr (L == 0) {
            const double v1 = f * R.y;
            s[0] += v0;
            s[1] += v1 * x;
            s[2] += v1 * y;
            s[3] += v1 * z;
        } else {
            const double v1 = f * R.y * ang;
            s[0] += v0 * ang;
            s[1] += v0 * ax + v1 * x;
            s[2] += v0 * ay + v1 * y;
            s[3] += v0 * az + v1 * z;
        }
    }
    // c0 Phi + (c1, c2, c3) . grad Phi
    __device__ __forceinline__ double dot(double x, double y, double z, const double2 R, const double* c) const {
        double ang, ax, ay, az;
        angular(x, y, z, ang, ax, ay, az);
        const double cd = c[1] * x + c[2] * y + c[3] * z;
        if constexpr (L == 0) return R.x * c[0] + R.y * cd;
        else return R.x * (c[0] * ang + c[1] * ax + c[2] * ay + c[3] * az) + R.y * ang * cd;
    }
};

// X = Phi D for 64 points of a block on MFMA, reduced into rho and grad rho, then the functional, the
// aow rows and E_xc: xc_rho_all_kernel over the block's own functions.  Eight wavefronts, wavefront wv
// holding the X tile of row tile wv % 4 and column half wv / 4 (at most NH of 16 columns); no bounds
// checks, since rows and columns are padded with zeros.  D is gathered by function number straight into
// LDS, 16 rows per K step, 32 threads per row; the next step's Phi and D elements are loaded during the
// current MFMAs while the registers allow two blocks per CU (NH <= kPackedPrefNH).
// Reading Phi and grad Phi for the reduction and again for the aow rows it was bound by memory; both are made
// from the radial parts instead (a sixth of the bytes; a block's functions are sorted by angular momentum,
// so a tile of 16 s or p columns takes the shorter code), and what bounds it now is latency at the 16
// wavefronts a CU that the accumulators leave (matrix cores 26 %, vector units 28 % busy).
// (H2O)16, 1.05e6 points: density kernel 6.98 ms dense, 2.50 ms packed, 2.02 ms from radial parts; V 3.67 ->
// 0.92 ms, summing the partial V 0.05 -> 0.17 ms; benzene, 1.3e5 points: density 0.29, 0.22, 0.18 ms (0.27 with
// every tile treated as d), V 0.18 -> 0.085 ms.
// The gradient uses it twice: kPackedGrad stores X, the gradient's rows and t as well, kPackedProduct only
// the product `out` = `in` D.
constexpr int kPackedPrefNH = 8;
enum { kPackedBuild, kPackedGrad, kPackedProduct };
template <int NH, int MODE>
__global__ __launch_bounds__(512) QCG_XC_RHO_ATTR void xc_rho_packed_kernel(
    const PackedGrid g, const double* __restrict__ in, const double* __restrict__ Dm, double* __restrict__ out,
    double* __restrict__ aow, double* __restrict__ exc_sum) {
    using M = Mfma<double>;
    using acc_t = typename M::acc;
    constexpr int BN = 32 * NH, SA = kRhoBM + 16, SB = BN + lds_pad<double>(BN);
    constexpr bool kPref = NH <= kPackedPrefNH;
    __shared__ double As[kRhoBK][SA];
    __shared__ double Bs[kRhoBK][SB < 32 ? 32 : SB];
    __shared__ double red[4][kRhoPW][4];
    __shared__ double coef[4][kRhoPW][4];
    __shared__ double part[4];
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
    const int per = g.S / kRhoBM, b = blockIdx.x / per, p0 = (blockIdx.x - b * per) * kRhoBM;
    const int ld = g.ld[b], nt = ld >> 4, nh = (nt + 1) >> 1;
    const int rt = wv & 3, half = wv >> 2, t0 = half * nh, mine = half ? nt - nh : nh;
    const size_t base = (size_t)g.off[b] + (size_t)p0 * ld;
    const int* fl = g.fl + g.floff[b];
    const double* __restrict__ phi = in + base;
    acc_t acc[NH];
#pragma unroll
    for (int t = 0; t < NH; ++t) acc[t] = acc_t{0.0, 0.0, 0.0, 0.0};
    // staging: A two functions of one point per thread, B columns (tid % 32) + 32 i of row tid / 32
    const int ar = tid >> 3, ac = 2 * (tid & 7), br = tid >> 5, bc = tid & 31;
    int fc[NH];
#pragma unroll
    for (int i = 0; i < NH; ++i) fc[i] = bc + 32 * i < ld ? fl[bc + 32 * i] : 0;
    double2 ra;
    double rb[kPref ? NH : 1];
    auto load_b = [&](int k0) {
        const double* row = Dm + (size_t)fl[k0 + br] * g.nbf;
#pragma unroll
        for (int i = 0; i < NH; ++i)
            if (32 * i < ld) rb[kPref ? i : 0] = row[fc[i]];
    };
    auto load = [&](int k0) {
        ra = *reinterpret_cast<const double2*>(phi + (size_t)ar * ld + k0 + ac);
        if constexpr (kPref) load_b(k0);
    };
    load(0);
    for (int k0 = 0; k0 < ld; k0 += kRhoBK) {
        __syncthreads();  // the previous step's fragment reads are done
        As[ac][ar] = ra.x;
        As[ac + 1][ar] = ra.y;
        if constexpr (kPref) {
#pragma unroll
            for (int i = 0; i < NH; ++i)
                if (32 * i < ld) Bs[br][bc + 32 * i] = rb[i];
        } else {
            const double* row = Dm + (size_t)fl[k0 + br] * g.nbf;
#pragma unroll
            for (int i = 0; i < NH; ++i)
                if (32 * i < ld) Bs[br][bc + 32 * i] = row[fc[i]];
        }
        __syncthreads();
        if (k0 + kRhoBK < ld) load(k0 + kRhoBK);
#pragma unroll 2
        for (int ks = 0; ks < kRhoBK; ks += 4) {
            const double a = As[ks + lk][kRhoPW * rt + li];
#pragma unroll
            for (int t = 0; t < NH; ++t)
                if (t < mine) acc[t] = M::mma(a, Bs[ks + lk][16 * (t0 + t) + li], acc[t]);
        }
    }
    if constexpr (MODE != kPackedBuild) {
#pragma unroll
        for (int t = 0; t < NH; ++t)
            if (t < mine)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    out[base + (size_t)(kRhoPW * rt + M::row(lk, r)) * ld + 16 * (t0 + t) + li] = acc[t][r];
        if constexpr (MODE == kPackedProduct) return;
    }
    // the block's functions, in the Phi staging area (free now)
    static_assert(sizeof(As) >= BN * (3 * sizeof(double) + sizeof(int)), "the functions fit in As");
    double(*fcen)[BN] = reinterpret_cast<double(*)[BN]>(&As[0][0]);
    int* fmeta = reinterpret_cast<int*>(fcen + 3);
    __syncthreads();  // every wavefront's last fragment reads are done
    if (tid < ld) {
        const GridFn f = g.fn[fl[tid]];
        fcen[0][tid] = f.cx;
        fcen[1][tid] = f.cy;
        fcen[2][tid] = f.cz;
        fmeta[tid] = f.axes | g.fs[g.floff[b] + tid] << 4;
    }
    const double2* __restrict__ rad = g.rad + g.roff[b] + (size_t)p0 * g.ldr[b];
    const double* __restrict__ pts = g.pts + 3 * ((size_t)b * g.S + p0);
    const int ldr = g.ldr[b];
    if (tid < 3 * kRhoBM) coef[tid / (3 * kRhoPW)][tid / 3 % kRhoPW][tid % 3] = pts[tid];
    __syncthreads();
    // per column half, row tile and point, in the D staging area (free now)
    static_assert(sizeof(Bs) >= 2 * 4 * kRhoPW * 4 * sizeof(double), "red2 fits in Bs");
    auto red2 = reinterpret_cast<double (*)[4][kRhoPW][4]>(&Bs[0][0]);
    // highest angular momentum among the columns c0 to c0 + n - 1 (a block's functions are sorted by it)
    const int nfn = g.nfn[b], n0 = g.nl[2 * b], n1 = g.nl[2 * b + 1];
    auto max_l = [&](int c0, int n) {
        const int e = min(c0 + n, nfn);
        return e <= n0 ? 0 : e <= n1 ? 1 : 2;
    };
    // RS of the lane's four points at a time, as many as the registers allow beside the accumulators
    constexpr int RS = NH <= 1 ? 4 : NH <= 5 ? 2 : 1;
#pragma unroll
    for (int r0 = 0; r0 < 4; r0 += RS) {
        double sum[RS][4] = {}, pt[RS][3];
        const double2* row[RS];
#pragma unroll
        for (int r = 0; r < RS; ++r) {
            const int p = M::row(lk, r0 + r);
            row[r] = rad + (kRhoPW * rt + p) * ldr;
#pragma unroll
            for (int q = 0; q < 3; ++q) pt[r][q] = coef[rt][p][q];
        }
#pragma unroll
        for (int t = 0; t < NH; ++t) {
            const int col = 16 * (t0 + t) + li;
            auto tile = [&](auto lc) {
                const FnAt<decltype(lc)::value> fn(fcen[0][col], fcen[1][col], fcen[2][col], fmeta[col]);
                double2 R[RS];
#pragma unroll
                for (int r = 0; r < RS; ++r) R[r] = row[r][fn.shell];
#pragma unroll
                for (int r = 0; r < RS; ++r)
                    fn.add(pt[r][0] - fn.cx, pt[r][1] - fn.cy, pt[r][2] - fn.cz, R[r], acc[t][r0 + r], sum[r]);
            };
            if (t < mine) {
                const int lmax = max_l(16 * (t0 + t), 16);
                if (lmax == 0) tile(std::integral_constant<int, 0>{});
                else if (lmax == 1) tile(std::integral_constant<int, 1>{});
                else tile(std::integral_constant<int, 2>{});
            }
            // one tile's loads in flight at a time: hoisting all of them costs hundreds of VGPRs
            asm volatile("" ::: "memory");
        }
#pragma unroll
        for (int r = 0; r < RS; ++r)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
#pragma unroll
                for (int off = 1; off < 16; off <<= 1) sum[r][q] += __shfl_xor(sum[r][q], off, 64);
                if (li == 0) red2[half][rt][M::row(lk, r0 + r)][q] = sum[r][q];
            }
    }
    __syncthreads();
    if (tid < 4 * kRhoPW * 4) {  // the two column halves, in a fixed order
        const int q = tid & 3, p = (tid >> 2) % kRhoPW, r4 = tid / (4 * kRhoPW);
        red[r4][p][q] = red2[0][r4][p][q] + red2[1][r4][p][q];
    }
    __syncthreads();
    const size_t pt0 = (size_t)b * g.S + p0;
    const double contrib = xc_point_coef(kRhoBM, wv, l, 0, g.w + pt0, red, coef, MODE == kPackedGrad,
                                         MODE == kPackedGrad ? exc_sum + 3 * pt0 : nullptr);
    __syncthreads();
    // aow = w vrho Phi + 4 w vsigma (grad rho . grad Phi) (the gradient's rows: 2): lanes over the columns,
    // each wavefront half the points of its row tile
    constexpr int kRows = kRhoPW / 2;
    const int q0 = kRhoPW * rt + kRows * half;
    for (int c0 = 0; c0 < ld; c0 += 64) {
        const int col = c0 + l;
        auto rows = [&](auto lc) {
            const FnAt<decltype(lc)::value> fn(fcen[0][col], fcen[1][col], fcen[2][col], fmeta[col]);
#pragma unroll 4
            for (int p = q0; p < q0 + kRows; ++p)
                aow[base + (size_t)p * ld + col] = fn.dot(pts[3 * p] - fn.cx, pts[3 * p + 1] - fn.cy, pts[3 * p + 2] - fn.cz,
                                                          rad[p * ldr + fn.shell], coef[rt][p - kRhoPW * rt]);
        };
        const int lmax = max_l(c0, 64);
        if (col < ld) {
            if (lmax == 0) rows(std::integral_constant<int, 0>{});
            else if (lmax == 1) rows(std::integral_constant<int, 1>{});
            else rows(std::integral_constant<int, 2>{});
        }
    }
    if constexpr (MODE == kPackedBuild) xc_point_exc(contrib, wv, l, exc_sum, part);
}

// in D for every block (or the whole XC build / gradient step, MODE)
template <int MODE>
static hipError_t launch_packed_rows(const PackedGrid& g, const double* in, const double* D, double* out, double* aow,
                                     double* sum, hipStream_t st) {
    const dim3 grid((unsigned)(g.nblk * (g.S / kRhoBM)));
    switch ((g.max_ld / 16 + 1) / 2) {
#define QCG_RHO_PACKED(n)                                                                                       \
    case n:                                                                                                     \
        hipLaunchKernelGGL((xc_rho_packed_kernel<n, MODE>), grid, dim3(512), 0, st, g, in, D, out, aow, sum);   \
        break;
        QCG_RHO_PACKED(1) QCG_RHO_PACKED(2) QCG_RHO_PACKED(3) QCG_RHO_PACKED(4) QCG_RHO_PACKED(5) QCG_RHO_PACKED(6)
        QCG_RHO_PACKED(7) QCG_RHO_PACKED(8) QCG_RHO_PACKED(9) QCG_RHO_PACKED(10) QCG_RHO_PACKED(11)
#undef QCG_RHO_PACKED
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_packed_grad_rows(const PackedGrid& g, const double* D, double* X, double* aow, double* M, double* t,
                                   hipStream_t st) {
    const hipError_t e = launch_packed_rows<kPackedGrad>(g, g.phi, D, X, aow, t, st);
    return e != hipSuccess ? e : launch_packed_rows<kPackedProduct>(g, aow, D, M, nullptr, nullptr, st);
}

// One output tile of the partial V of a block: Phi^T aow over its S points, 32 VW square (xc_v_kernel's
// tiling), written packed.
template <int VW>
__device__ __forceinline__ void xc_v_packed_tile(const PackedGrid& g, const int4 tl, const double* __restrict__ aow,
                                                 double* __restrict__ Vparts, double* smem) {
    using M = Mfma<double>;
    using acc_t = typename M::acc;
    constexpr int BM = 32 * VW;
    auto As = reinterpret_cast<double (*)[BM + kPad]>(smem);
    auto Bs = As + kVBK;
    const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, li = l & 15, lk = l >> 4;
    const int wr = wv >> 1, wc = wv & 1;
    const int b = tl.x, m0 = tl.y, n0 = tl.z, ld = g.ld[b];
    const double* __restrict__ A = g.phi + g.off[b] + m0;
    const double* __restrict__ B = aow + g.off[b] + n0;
    acc_t acc[VW][VW];
#pragma unroll
    for (int i = 0; i < VW; ++i)
#pragma unroll
        for (int j = 0; j < VW; ++j) acc[i][j] = acc_t{0.0, 0.0, 0.0, 0.0};
    // staging: 16 threads per row of 16 points, two columns each per pass of 32
    const int sr = tid >> 4, sc = 2 * (tid & 15);
    double2 ra[VW], rb[VW];
    auto load = [&](int k0) {
        const size_t row = (size_t)(k0 + sr) * ld + sc;
#pragma unroll
        for (int i = 0; i < VW; ++i) {
            ra[i] = m0 + 32 * i + sc < ld ? *reinterpret_cast<const double2*>(A + row + 32 * i) : make_double2(0.0, 0.0);
            rb[i] = n0 + 32 * i + sc < ld ? *reinterpret_cast<const double2*>(B + row + 32 * i) : make_double2(0.0, 0.0);
        }
    };
    load(0);
    for (int k0 = 0; k0 < g.S; k0 += kVBK) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < VW; ++i) {
            *reinterpret_cast<double2*>(&As[sr][32 * i + sc]) = ra[i];
            *reinterpret_cast<double2*>(&Bs[sr][32 * i + sc]) = rb[i];
        }
        __syncthreads();
        if (k0 + kVBK < g.S) load(k0 + kVBK);
#pragma unroll
        for (int ks = 0; ks < kVBK; ks += 4) {
            double a[VW], c[VW];
#pragma unroll
            for (int i = 0; i < VW; ++i) {
                a[i] = As[ks + lk][16 * VW * wr + 16 * i + li];
                c[i] = Bs[ks + lk][16 * VW * wc + 16 * i + li];
            }
#pragma unroll
            for (int i = 0; i < VW; ++i)
#pragma unroll
                for (int j = 0; j < VW; ++j)  // sub-tiles past the block's functions: uniform per wavefront
                    if (m0 + 16 * VW * wr + 16 * i < ld && n0 + 16 * VW * wc + 16 * j < ld) acc[i][j] = M::mma(a[i], c[j], acc[i][j]);
        }
    }
    double* out = Vparts + g.voff[b];
#pragma unroll
    for (int i = 0; i < VW; ++i)
#pragma unroll
        for (int j = 0; j < VW; ++j) {
            const int col = n0 + 16 * VW * wc + 16 * j + li;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = m0 + 16 * VW * wr + 16 * i + M::row(lk, r);
                if (row < ld && col < ld) out[(size_t)row * ld + col] = acc[i][j][r];
            }
        }
}

// The tiles of all widths in one launch, the widest first.  One launch per width left the chip half idle in
// each: (H2O)16 0.47 + 0.28 + 0.24 ms (half a wavefront per SIMD in the widest), benzene 0.08 + 0.05.
__global__ __launch_bounds__(256) void xc_v_packed_kernel(const PackedGrid g, const int4* __restrict__ tiles,
                                                          const double* __restrict__ aow, double* __restrict__ Vparts) {
    __shared__ double smem[2 * kVBK * (32 * 5 + kPad)];
    const int4 tl = tiles[blockIdx.x];
    if (tl.w == 3) xc_v_packed_tile<3>(g, tl, aow, Vparts, smem);
    else if (tl.w == 4) xc_v_packed_tile<4>(g, tl, aow, Vparts, smem);
    else xc_v_packed_tile<5>(g, tl, aow, Vparts, smem);
}

// Vsum[k] = sum of the partial matrices of the k-th run of blocks, one matrix row per thread block
__global__ __launch_bounds__(128) void packed_vsum_kernel(const PackedGrid g, int per, const double* __restrict__ Vparts,
                                                          double* __restrict__ Vsum) {
    const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.z;
    const int b1 = min(g.nblk, (k + 1) * per);
    const bool in = j < g.nbf;
    double s = 0.0;
    for (int b = k * per; b < b1; ++b) {
        const int pi = g.pos[(size_t)b * g.nbf + i];
        if (pi < 0) continue;  // uniform
        const int pj = in ? g.pos[(size_t)b * g.nbf + j] : -1;
        if (pj >= 0) s += Vparts[(size_t)g.voff[b] + (size_t)pi * g.ld[b] + pj];
    }
    if (in) Vsum[((size_t)k * g.nbf + i) * g.nbf + j] = s;
}

__global__ __launch_bounds__(128) void packed_vsym_kernel(int nbf, int ngrp, const double* __restrict__ Vsum,
                                                          double* __restrict__ V) {
    const int i = blockIdx.y, j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= nbf) return;
    const size_t n2 = (size_t)nbf * nbf, ij = (size_t)i * nbf + j, ji = (size_t)j * nbf + i;
    double s = 0.0, t = 0.0;
#pragma unroll 8
    for (int k = 0; k < ngrp; ++k) {
        s += Vsum[k * n2 + ij];
        t += Vsum[k * n2 + ji];
    }
    V[ij] = 0.5 * (s + t);
}

int packed_v_width(int ld) { return xc_v_width(ld, false); }

hipError_t launch_xc_packed(const PackedGrid& g, const double* D, double* aow, const int4* tiles, int ntile,
                            double* Vparts, double* Vsum, double* V, double* exc_sum, hipStream_t st) {
    hipError_t e = launch_packed_rows<kPackedBuild>(g, g.phi, D, nullptr, aow, exc_sum, st);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(xc_v_packed_kernel, dim3((unsigned)ntile), dim3(256), 0, st, g, tiles, aow, Vparts);
    const int ngrp = g.nblk < kPackedVGroups ? g.nblk : kPackedVGroups, per = (g.nblk + ngrp - 1) / ngrp;
    const dim3 vg((g.nbf + 127) / 128, g.nbf, ngrp);
    hipLaunchKernelGGL(packed_vsum_kernel, vg, dim3(128), 0, st, g, per, Vparts, Vsum);
    hipLaunchKernelGGL(packed_vsym_kernel, dim3((g.nbf + 127) / 128, g.nbf), dim3(128), 0, st, g.nbf, ngrp, Vsum, V);
    return hipGetLastError();
}

template <typename T>
static hipError_t launch_xc_mfma_t(int G, int nbf, int nchunk, const double* w, const T* phi, const T* dpx,
                                   const T* dpy, const T* dpz, const float4* g4, const T* Dm, T* aow, double* exc_sum,
                                   double* Vparts, const unsigned* mask, hipStream_t st) {
    const GridVals<T> gv{phi, dpx, dpy, dpz, g4};
    if (G <= 0 || nbf <= 0 || nchunk <= 0) return hipErrorInvalidValue;
    // column passes of at most 5 MFMA tiles (4 for FP64, whose accumulators take twice the
    // registers), with the tiles spread evenly over the passes.  FP32: 5 tiles keep the kernel at
    // 164 registers, three wavefronts per SIMD; 7 or 8 tiles need about 200 (two wavefronts) and
    // were 7 % slower on (H2O)16, 4 tiles 1.5 % slower.
    constexpr int kMaxNT = sizeof(T) == 8 ? 4 : 5;
    const int tiles = (nbf + 15) / 16, passes = (tiles + kMaxNT - 1) / kMaxNT, nt = (tiles + passes - 1) / passes;
    const dim3 grid((G + kRhoBM - 1) / kRhoBM);
    // up to kRhoAllMaxNT column tiles: the all-columns kernel (Phi read once per K step)
    if (sizeof(T) == 4 && !mask && xc_tile_mask_words(G, nbf)) return hipErrorInvalidValue;
    switch (tiles <= kRhoAllMaxNT ? 100 + tiles : nt) {
#define QCG_RHO_ALL(n)                                                                                  \
    case 100 + n:                                                                                       \
        hipLaunchKernelGGL((xc_rho_all_kernel<T, n>), grid, dim3(512), 0, st, G, nbf, w, phi, gv, Dm, aow,  \
                           exc_sum, mask);                                                              \
        break;
        QCG_RHO_ALL(1) QCG_RHO_ALL(2) QCG_RHO_ALL(3) QCG_RHO_ALL(4) QCG_RHO_ALL(5) QCG_RHO_ALL(6) QCG_RHO_ALL(7)
        QCG_RHO_ALL(8) QCG_RHO_ALL(9) QCG_RHO_ALL(10) QCG_RHO_ALL(11) QCG_RHO_ALL(12) QCG_RHO_ALL(13)
        QCG_RHO_ALL(14) QCG_RHO_ALL(15) QCG_RHO_ALL(16) QCG_RHO_ALL(17) QCG_RHO_ALL(18) QCG_RHO_ALL(19)
        QCG_RHO_ALL(20) QCG_RHO_ALL(21) QCG_RHO_ALL(22)
#undef QCG_RHO_ALL
#define QCG_RHO_NT(n)                                                                                   \
    case n:                                                                                             \
        hipLaunchKernelGGL((xc_rho_kernel<T, n>), grid, dim3(256), 0, st, G, nbf, w, phi, gv, Dm, aow,      \
                           exc_sum);                                                                    \
        break;
        QCG_RHO_NT(1) QCG_RHO_NT(2) QCG_RHO_NT(3) QCG_RHO_NT(4) QCG_RHO_NT(5)
#undef QCG_RHO_NT
        default: return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int chunk = (G + nchunk - 1) / nchunk;
    const int nch = (G + chunk - 1) / chunk;  // <= nchunk partial matrices written
    const int vw = xc_v_width(nbf, sizeof(T) == 4);
    const int ntile = (nbf + 32 * vw - 1) / (32 * vw);
    const int nblk = 8 * ((nch + 7) / 8) * ntile * ntile;
    switch (vw) {
        case 3:
            hipLaunchKernelGGL((xc_v_kernel<T, 3>), dim3(nblk), dim3(256), 0, st, G, nbf, ntile, nch, chunk, phi, aow,
                               Vparts);
            break;
        case 4:
            hipLaunchKernelGGL((xc_v_kernel<T, 4>), dim3(nblk), dim3(256), 0, st, G, nbf, ntile, nch, chunk, phi, aow,
                               Vparts);
            break;
        case 5:
            hipLaunchKernelGGL((xc_v_kernel<T, 5>), dim3(nblk), dim3(256), 0, st, G, nbf, ntile, nch, chunk, phi, aow,
                               Vparts);
            break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <typename T>
static int v_blocks_per_cu_t(int vw) {
    int n = 0;
    hipError_t e = hipErrorInvalidValue;
    if (vw == 3) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, xc_v_kernel<T, 3>, 256, 0);
    else if (vw == 4) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, xc_v_kernel<T, 4>, 256, 0);
    else if (vw == 5) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, xc_v_kernel<T, 5>, 256, 0);
    return e == hipSuccess && n > 0 ? n : 1;
}

int xc_v_blocks_per_cu(int nbf, bool fp32) {
    const int vw = xc_v_width(nbf, fp32);
    return fp32 ? v_blocks_per_cu_t<float>(vw) : v_blocks_per_cu_t<double>(vw);
}

hipError_t launch_xc_mfma(int G, int nbf, int nchunk, const double* w, const float* phi, const float4* g4,
                          const unsigned* mask, const float* Dm, float* aow, double* exc_sum, double* Vparts,
                          hipStream_t st) {
    return launch_xc_mfma_t<float>(G, nbf, nchunk, w, phi, nullptr, nullptr, nullptr, g4, Dm, aow, exc_sum, Vparts,
                                   mask, st);
}

hipError_t launch_xc_mfma(int G, int nbf, int nchunk, const double* w, const double* phi, const double* dpx,
                          const double* dpy, const double* dpz, const double* Dm, double* aow, double* exc_sum,
                          double* Vparts, hipStream_t st) {
    return launch_xc_mfma_t<double>(G, nbf, nchunk, w, phi, dpx, dpy, dpz, nullptr, Dm, aow, exc_sum, Vparts, nullptr, st);
}

}  // namespace qcg
