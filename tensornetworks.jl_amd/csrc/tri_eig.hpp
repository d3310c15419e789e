// Whole-GPU eigensolver of Hermitian (Gram) matrices: see tri_eig.hip.
#pragma once

#include <cstdint>

struct tnh_ctx;

namespace tnh {

// Gram sides solved here; smaller ones take one workgroup (dc_eig.hpp), and the largest is what
// the column step's three vectors per plane leave room for in LDS (147 of 160 KB).
// Smallest sides: measured on graded matrices, this / one workgroup, ms, complex 10 0.09 / 0.12, 16
// 0.11 / 0.17, 24 0.16 / 0.22, 64 0.30 / 0.51; real 16 0.10 / 0.15, 64 0.27 / 0.46, 96 0.39 / 0.74.
// By time alone both lines would be near 10 (a whole complex split of side 16 0.22 / 0.28 ms:
// that much the line at 24 leaves to be had). Real sides up to 96 (bond dimensions up to 48) are the
// splits of short DMRG runs from random states, which amplify rounding (four passes after a
// start changed by 1e-15: observables moved by 5.5e-11 in the median of 100 seeds and by 2.5e-9
// at most): they stay with the solver whose rounding those runs have always had.
constexpr int kTriMinReal = 97, kTriMinCplx = 24;
constexpr int kTriMaxReal = 6144, kTriMaxCplx = 3072;

// Reduce the p x p Hermitian G (planar, device, overwritten) and solve the tridiagonal
// problem: dout[0..p) = eigenvalues, ascending, dout[p] = 1 on success, 0 otherwise. The
// reflectors and tridiagonal eigenvectors stay in workspaces until the next call.
void tri_eig_solve(tnh_ctx *ctx, double *G, int p, bool cplx, double *dout);
// Eigenvectors perm[0..k) (device indices into the ascending order) of the last solved matrix
// into basis (p x k, planar).
void tri_eig_vectors(tnh_ctx *ctx, int p, bool cplx, const int *perm, int k, double *basis);

}  // namespace tnh
