// Host-callable launchers of the device kernels (all asynchronous on the given stream).
#pragma once
#include <hip/hip_runtime.h>
#include "devtypes.hpp"

namespace uno {

// ERIs of explicit quartet lists, block and Schwarz modes, FP64 (eri.hip)
hipError_t eri_launch(int mode, int bra_class, int ket_class, const EriArgs& a, hipStream_t st);
int eri_class_ncomp(int bra_class, int ket_class);

// Fock-build launches (fock_core.hpp).  Classes above kLaneMaxComp components run one quartet per
// wave (fock_is_wave); the others one ket per lane with the exchange rows of the bra merged in
// LDS (variant 1 every bra row and the Rys table in LDS, 2 every bra row, 3 the first bra
// shell's rows, 0 none: every output straight to W), the bra's exchange density rows (dlds) and
// shell maxima (mlds) staged there where they fit.
struct FockConfig {
    int variant = 0, dlds = 0, mlds = 0;
};
constexpr int kLaneBlock = 256;   // lanes of a block of the lane kernels
constexpr int kWaveSeg = 8;       // kets of a block of the wave kernels
bool fock_is_wave(int bra_class, int ket_class);
// the first of (force, 1, 2, 3) that fits the LDS budget at ncols columns (rows false: 0), with
// what else fits; density rows: dens 0 none, 1 where they fit, -1 where they pay
FockConfig fock_default(int bra_class, int ket_class, int mode, int ncols, int nsh, bool fp32, bool rows, int force,
                        int dens);
bool fock_config_fits(int bra_class, int ket_class, const FockConfig& f, int mode, int ncols, int nsh, bool fp32);
hipError_t fock_launch(int mode, bool fp32, int bra_class, int ket_class, FockArgs a, const FockConfig& f, int ncols,
                       hipStream_t st);
// lists the tasks of nsrc launches that hold a quartet (a: the build's thresholds, bounds and
// density maxima); nblocks of kTaskThreads candidates in all, the counters zeroed
hipError_t fock_tasks(int nsrc, const FockTaskSource* src, int nblocks, const char* tables, const FockArgs& a,
                      FockCounter* ctr, int* lists, hipStream_t st);
// the Fock kernels' copies of the pair data (device arrays), runs sorted by off
hipError_t pair_store(int np, int nrun, const PairRun* runs, const PairHdr* pairs, const PrimPair* prims,
                      const int* colmap, BraPrim* bprim, double* kprim, long long kps, double* kgeo, int4* kidx, int4* kjo,
                      int* knp, int2* kcol, hipStream_t st);
// up to six buffers of 64-bit words zeroed in one launch
struct ClearList {
    unsigned long long* p[6];
    long long len[6];
    int n = 0;
    template <class T>
    void add(T* q, long long count) {
        static_assert(sizeof(T) % 8 == 0, "64-bit words");
        p[n] = reinterpret_cast<unsigned long long*>(q);
        len[n++] = count * (long long)(sizeof(T) / 8);
    }
};
hipError_t fock_clear(const ClearList& c, hipStream_t st);
// dp = D0 in pair-major blocks, dpair = every pair's own entry of dsh (mols / pmol: batched
// stores and every pair's molecule, or null)
hipError_t pair_density(int npairs, const int4* kidx, const int4* kjo, const double* D0, const double* dsh, int n,
                        int nsh, const MolDesc* mols, const int* pmol, double* dp, double* dpair, hipStream_t st);
// the pair-major jp added into W (and W1)
hipError_t jp_scatter(int npairs, const int4* kidx, const int4* kjo, const double* jp, double* W0, double* W1, int n,
                      const MolDesc* mols, const int* pmol, hipStream_t st);
// new pair k = old pair order[k], its primitives at prim0[k] (device arrays; new ones must not
// overlap the old)
hipError_t permute_pairs(int np, const int* order, const int* prim0, const PairHdr* oldp, const PrimPair* oldq,
                         PairHdr* newp, PrimPair* newq, hipStream_t st);
// deterministic builds: W accumulated in fixed point (entry i: int64 words i and i + lo_off)
// back to FP64 in place, first nn entries
hipError_t fixed_to_f64(long long nn, double* W, long long lo_off, hipStream_t st);
hipError_t rys_eval_launch(int n, int npts, const double* x, double* u, double* w, hipStream_t st, bool fp32 = false,
                           bool ref2 = false);

// dense helpers (linalg.hip); matrices are row-major n x n
hipError_t k_unpack(int n, const double* packed, double* dense, hipStream_t st);       // symmetric fill
hipError_t k_pack(int n, const double* dense, double* packed, hipStream_t st);         // lower triangle
hipError_t k_pack_sym_add(int n, const double* W, double* packed, hipStream_t st);     // packed += (W+W^T)_lower
// G = W + W^T, or G += W + W^T when accumulating
hipError_t k_sym_w(int n, const double* W, double* G, hipStream_t st, bool accumulate = false);
hipError_t k_axpby(long len, double a, const double* x, double b, const double* y, double* z, hipStream_t st);
hipError_t k_fill(long len, double v, double* x, hipStream_t st);
// X[i][j] = Z[i][j] f[j] (n x n, f on the device)
hipError_t k_scale_cols(int n, const double* Z, const double* f, double* X, hipStream_t st);
// out[0] += sum_ij A_ij B_ij (full matrices); deterministic two-pass reduction whose
// workspace ws holds kRedBlocks partial sums (one workspace per stream)
constexpr int kRedBlocks = 240;
hipError_t k_dot(long len, const double* A, const double* B, double* out, double* ws, hipStream_t st);
// out[0] = sqrt(sum (A-B)^2) / n
hipError_t k_diffnorm(long len, int n, const double* A, const double* B, double* out, double* ws, hipStream_t st);
// Dsh[s][t] = max |D_ij| over the function block of shells s, t of up to three matrices;
// dmax (zeroed by the caller) = the largest of them
hipError_t k_shell_max(int n, int nsh, const int* sh_off, const int* sh_n, const double* D, const double* D1,
                       const double* D2, double* Dsh, double* dmax, hipStream_t st);
// out[0] = max |x|
hipError_t k_absmax(long len, const double* x, double* out, hipStream_t st);
// A_ii += alpha (n x n)
hipError_t k_shift_diag(int n, double alpha, double* A, hipStream_t st);
// purification: Gershgorin bounds of F (lohi: 2n work, bounds: 2 doubles) and
// X = (hi I - F) / (hi - lo); out[0] = tr(A)
hipError_t sp2_init(int n, const double* F, double* X, double* lohi, double* bounds, hipStream_t st);
hipError_t k_trace(int n, const double* A, double* out, hipStream_t st);
// launch-chained purification steps (linalg.hip): states is an array of step states
// (sp2_state_bytes() each); sp2_start fills state 0 and X0's tile sums (part0: 2 doubles per
// upper-triangle 64 x 64 tile); sp2_steps enqueues steps k0 .. k0+count-1; sp2_state_read
// waits for the stream and reads state k (cur = buffer holding X, done 1 = converged,
// 2 = failed, steps = steps taken, t1 = tr(X))
size_t sp2_state_bytes();
hipError_t sp2_start(int n, const double* X0, double* part0, void* st0, hipStream_t st);
hipError_t sp2_steps(int n, int nocc, double thr, void* states, int k0, int count, double* buf0, double* buf1,
                     double* part0, double* part1, hipStream_t st);
hipError_t sp2_state_read(const void* states, int k, int* cur, int* done, int* steps, double* t1, hipStream_t st);
// C = alpha op(A) op(B) + beta C  (FP64 MFMA 16x16x4)
hipError_t gemm_f64(bool ta, bool tb, int m, int n, int k, double alpha, const double* A, int lda, const double* B,
                    int ldb, double beta, double* C, int ldc, hipStream_t st);
// 1: this thread's gemm_f64 calls give bitwise-repeatable products (no split K, whose
// chunks are added with atomics); returns the previous setting
int gemm_deterministic(int on);
struct GemmDetScope {
    int prev;
    explicit GemmDetScope(bool on) : prev(gemm_deterministic(on ? 1 : 0)) {}
    ~GemmDetScope() { gemm_deterministic(prev); }
    GemmDetScope(const GemmDetScope&) = delete;
    GemmDetScope& operator=(const GemmDetScope&) = delete;
};

// eigensolver pieces (linalg.hip), 3 <= n <= kEigMaxN
constexpr int kEigMaxN = 6752;   // where a block's LDS ends (linalg.hip)
struct EigWork {
    double* A;      // n x n working copy (destroyed)
    double* V;      // n x n reflector vectors (row k = v_k, zero outside its support)
    double* tau;    // n
    double* p;      // n
    double* d;      // n, and zeros up to a multiple of 16: diagonal of T
    double* e;      // the same: off-diagonal of T
    double* scal;   // 4 scalars
    double* evals;  // n  eigenvalues of T (ascending)
    double* Y;      // n x n eigenvectors of T, one per column (Yt)
    double* wk;     // work space of at least eig_work_doubles(n), at most 5 n^2
};
size_t eig_work_doubles(int n);
hipError_t householder_tridiag(int n, EigWork& w, hipStream_t st);
// Z <- Q Z with Q = H_0 ... H_{n-3} from the reflectors in w.V / w.tau (uses w.wk)
hipError_t apply_q(int n, EigWork& w, double* Z, hipStream_t st);
// nclusters < 0: multisection for w.evals; otherwise inverse iteration into the columns of
// w.Y followed by Gram-Schmidt inside the given clusters ({first, end} pairs, device memory)
hipError_t tridiag_eigen(int n, EigWork& w, int nclusters, const int* clusters, hipStream_t st);

// streaming copy of `bytes` (read + write), reps times; total milliseconds in *ms
hipError_t copy_probe(size_t bytes, int reps, float* ms, hipStream_t st);

}  // namespace uno
