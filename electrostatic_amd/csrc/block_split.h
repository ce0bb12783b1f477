// block_split.h -- launchers of the two-part block chain kernels
// (block_split.hip), called by the dense-block C ABI.
#pragma once

#include <hip/hip_runtime.h>

namespace negf {

// A chain whose coupling T connects only the second part of a block (orbitals
// h .. m-1) with the first part (0 .. h-1) of the next: a chain of twice as
// many blocks of at most 16 orbitals.
struct SplitChain {
    int m = 0, nb = 0, h = 0;      // orbitals per block, blocks, first part (0: not splittable)
    const double* mats = nullptr;  // device: H_00, H_11, H_01, T_10, each 16 x 16 row-major, zero padded
    const double* v = nullptr;     // device: [nb][32] orbital potentials
};

// Part size h for which T is zero outside rows >= h, columns < h and both
// parts have 1..16 orbitals (the most even choice), or 0.  T: m x m row-major
// with row stride ld.
int split_part_size(int m, const double* T, int ld);
// The four 16 x 16 matrices of a split chain from H0 and T (row stride ld).
void split_matrices(int m, int h, const double* H0, const double* T, int ld, double* mats);

constexpr int SPLIT_SIGMA = 512;  // doubles per (energy, lead): the self-energy on its part
// Lead self-energies: sigma [nE][2][256 complex], lane order of the sweep.
hipError_t split_sancho_rubio(const SplitChain& c, int nE, const double2* E, double Uc0, double Uc1, double tol,
                              int max_iter, double* sigma, int* iters, hipStream_t st);
// Element (i, j) of a stored self-energy: index of its complex value.
inline int split_sigma_index(int i, int j) { return (j >> 2) * 64 + (j & 3) * 16 + i; }
// Bytes of scratch per energy of the sweep.
inline size_t split_scratch_per_energy(int nb) { return (size_t)nb * 2 * 256 * sizeof(double2); }
// Energies e0 .. e0 + n - 1: part[e][nb * m] = Im(coef_e G_oo) and, if diag, G_oo.
hipError_t split_rgf(const SplitChain& c, int e0, int n, const double2* E, const double2* coef, const double* sigma,
                     double2* scratch, double* part, double2* diag, hipStream_t st);

}  // namespace negf
