// Dense kernels of the batched SCF (batch.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "devtypes.hpp"

namespace uno {

// one molecule's n x n matrix of one spin: its first element in every store
struct MatSlot {
    long long off;
    int n, nocc, spin;
};
// the two spins' stores of a quantity (a launch takes the slots of both)
struct Store {
    double* s[2];
};
// one 32 x 32 output tile of a slot's product
struct GemmTile {
    int slot, ti, tj;
};
// C = op(A) op(B) for the slots of the tiles; occ: summed over the slot's occupied columns only
hipError_t grouped_gemm(int ntiles, const GemmTile* tiles, const MatSlot* slots, bool ta, bool tb, bool occ, Store A, Store B,
                        Store C, hipStream_t st);

// symmetric matrices of n <= 256 (maxn the largest): A (destroyed), V (work), evals (n values at the
// slot's offset, ascending), Z (eigenvectors in the columns)
hipError_t batched_jacobi(int nslot, const MatSlot* slots, Store A, Store V, Store evals, Store Z, int maxn, int max_sweeps,
                          hipStream_t st);

// the eigenvectors (columns of Z, n <= 256) of levels that coincide across a slot's Fermi level, in the
// order of Z's rows, which rounding does not decide
hipError_t batch_ties(int nslot, const MatSlot* slots, Store evals, Store Z, hipStream_t st);

// out[q nslot + k] = sum_ij A_q,ij B_q,ij over slot k, for the pairs q that name stores of its spin
constexpr int kMaxDots = 12;
struct DotPairs {
    int n;
    const double* a[kMaxDots][2];
    const double* b[kMaxDots][2];
    void add(const double* a0, const double* a1, const double* b0, const double* b1) {
        a[n][0] = a0, a[n][1] = a1, b[n][0] = b0, b[n][1] = b1;
        ++n;
    }
};
hipError_t batch_dots(int nslot, const MatSlot* slots, const DotPairs& q, double* out, hipStream_t st);
hipError_t batch_diffnorm(int nslot, const MatSlot* slots, Store A, Store B, double* out, hipStream_t st);
// G = W + W^T
hipError_t batch_sym(int nslot, const MatSlot* slots, Store W, Store G, hipStream_t st);
// F = H + G
hipError_t batch_add(int nslot, const MatSlot* slots, const double* H, Store G, Store F, hipStream_t st);
// out = W - W^T
hipError_t batch_antisym(int nslot, const MatSlot* slots, Store W, Store out, hipStream_t st);
// over whole stores: D0 = P0 + P1, and the copies of P0, P1
hipError_t batch_densities(long long len, Store P, double* D0, Store Pold, hipStream_t st);
hipError_t batch_shell_max(int nmol, int maxsh, const MolDesc* mols, const int* shoff, const int* active,
                           const int* sh_off, const int* sh_n, const double* D, const double* D1, const double* D2,
                           double* Dsh, double* dmax, hipStream_t st);
// F_k = sum_j coef[k kMaxLin + j] src_j
constexpr int kMaxLin = 8;
struct LinSources {
    const double* s[kMaxLin][2];
};
hipError_t batch_lincomb(int nslot, const MatSlot* slots, const double* coef, const LinSources& src, Store F, hipStream_t st);

}  // namespace uno
