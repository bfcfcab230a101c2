// Device construction of the V-list transfer blocks (implemented in transfer.hip).
#pragma once
#include <cstdint>

#include <hip/hip_runtime_api.h>

namespace pvfmm_amd {

// Frequency grid of the V-list transforms: n points per axis, the x axis halved (nh), M
// frequencies f = kx + nh * (ky + n * kz).
struct VGrid {
  int n = 0, nh = 0, M = 0;
};
VGrid v_grid(int m);

// Spectra of the child-to-child M2L kernels (include/fmm_pts.txx:671-719): for the source-minus-
// target child offset r in [-3, 3]^3, ri = (rx + 3) + 7 (ry + 3) + 49 (rz + 3), component
// q = i * e1 + j, G[(ri * e0 e1 + q) * M + f] (complex) is the DFT over the n^3 grid of
// K_ij(w h - r), w the lattice displacement, h the lattice spacing of unit boxes, times 1 / n^3;
// zero for adjacent boxes (all |r_d| <= 1).  kind as in build_matrix_device (0 or 2).  All FP64;
// blocks until done (it owns its scratch memory).
void transfer_spectra(hipStream_t s, int kind, int m, double* G);

// The transfer block of parent offset R in real form for y = x B, x and y interleaved (re, im):
// with row position k holding component k / 16 of child (k % 16) / 2 (real part for even k) and
// the same for the output position n, B[k][n] = +-Re or +-Im of G at the children's offset.  The
// forms the Hadamard kernels read (offsets R in increasing order without 13, in pairs for the
// split forms):
//   real:   Vp[((R * M + f) * e0 + kb) * e1 + nb][lane][q], FP64 kernels, R of 27
//   fp16:   two parts of tau_f B, scalar (the second times kSplitLow) and Stokes layouts of
//           hadamard_tiled; tinv = 1 / tau_f
void transfer_real(hipStream_t s, int e0, int e1, int M, const double* G, double* Vp);
void transfer_fp16(hipStream_t s, int e0, int e1, int M, const double* G, uint16_t* Vh, float* tinv);

// out (rows x ld_out, Real) = in (rows_in x cols_in, FP64), zero outside it; transposed: out
// (rows x ld_out) = in^T.
template <typename Real>
void convert_matrix(hipStream_t s, const double* in, int rows_in, int cols_in, Real* out, int rows, int ld_out,
                    bool transposed = false);
// out (cols x rows) = in^T, in rows x cols
template <typename Real>
void transpose_matrix(hipStream_t s, const Real* in, int rows, int cols, Real* out);

}  // namespace pvfmm_amd
