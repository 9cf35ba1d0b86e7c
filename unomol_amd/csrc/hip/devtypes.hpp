// Device-side data layout of the direct-SCF engine (shared by host builders and kernels).
//
// Shell pairs (a >= b by shell index) are stored with the higher-l shell first, so every
// quartet class (la,lb|lc,ld) has la >= lb and lc >= ld like the reference's swapped
// shell quartets (TwoElectronInts.cpp:563-580).  Each pair owns a contiguous run of
// primitive pairs.  Both records are 64 bytes so a lane fetches them as 4 x dwordx4.
#pragma once
#include <cstdint>

namespace uno {

struct alignas(16) PairHdr {
    double A[3];    // centre of the first (higher-l) shell
    double AB[3];   // A - B
    int f1, f2;     // first basis function of shell 1 and shell 2
    int prim0;      // first primitive pair
    int nprim;      // number of primitive pairs
    int same;       // both shells are the same shell (a == b)
    int sh1, sh2;   // shell indices (first, second)
    int pad;
};

struct alignas(16) PrimPair {
    double p, ip;   // exponent sum and its inverse
    double P[3];    // Gaussian product centre
    double K;       // c_i c_j (x2 for off-diagonal same-shell pairs) exp(-ab/p |AB|^2)
    double s;       // bare exp(-ab/p |AB|^2) for the primitive prefactor cut
    double pad;
};

// slot pairs of the evaluated-quartet counters of one launch (spread to avoid contention)
constexpr int kCounterSlots = 64;

// pair class index for (l1 >= l2), l <= 2: ss=0 ps=1 pp=2 ds=3 dp=4 dd=5
constexpr int pair_class(int l1, int l2) { return l1 * (l1 + 1) / 2 + l2; }
constexpr int kMaxL = 2;
constexpr int kNumPairClasses = 6;

// digest modes of the ERI kernels
enum DigestMode : int {
    kDigestRHF = 0,      // W += 4 J'[P] - K'[P]
    kDigestUHF = 1,      // Wa += 2 J'[Pa+Pb] - K'[Pa], Wb likewise
    kDigestBlock = 2,    // write the contracted, normalised ERI block
    kDigestSchwarz = 3,  // max |(ij|ij)| of a diagonal quartet
};

// one molecule of a batched launch: its dense matrices start at moff of every store,
// its shell-block density maxima at dshoff
struct MolDesc {
    long long moff;
    long long dshoff;
    int n, nsh;
};

// explicit quartet lists (block and Schwarz modes)
struct EriArgs {
    const PairHdr* pairs;
    const PrimPair* prims;
    const int2* explicit_q;   // (bra, ket) pairs
    long long nquart;
    int qpb;                  // quartets per block of the launch
    int rys2_exact;           // 1: exact two-root Rys quadrature; 0: the reference's
                              // two-root quadrature (Rys.cpp:413-631), the default
    double primcut;           // bare primitive prefactor cut (reference 1e-12)
    double* out;              // block / Schwarz output
};

// ---- Fock builds --------------------------------------------------------------------
// primitive pair as a bra: read whole, through the scalar cache.  K and s carry the bra's
// share of the quartet prefactor, 2 pi^(5/2) / p (the ket's is 1 / q)
struct alignas(16) BraPrim {
    double p, ip, K, s;
    double P[3], PA[3];   // product centre, and relative to the first shell's centre
};
// fields of a primitive pair as a ket, stored field by field: q, 1/q, K/q, s/q, P
constexpr int kKetFields = 7;

// One space of a Fock-build launch: the bra run [bra_off, bra_off + nbra) against the ket run
// [ket_off, ket_off + nket) of the pair array, both sorted by Schwarz bound (descending).  Its
// candidates are first + bra * nseg + segment; same: both are the same run (kets up to the bra).
struct FockSpace {
    int first;
    int bra_off, nbra, ket_off, nket;
    int nseg, seg;        // segments per bra, kets per segment
    int lg;               // 2^lg lanes share a ket (and split its primitives)
    int same, mol;
    int col0, ncols;      // LDS row columns: function of column c at colinv[col0 + c]
    int kstride;          // the ket run's length: primitive j of ket i at kp0 + j kstride + i
    int pad;
    long long kp0;
    long long jo0;        // component c of ket i at jo0 + c kstride + i of the pair-major arrays
};

// a run of the pair array, as the kernel that lays the ket records out needs it
struct PairRun {
    int off, count;
    int col0;             // column of function f at colmap[col0 + f]
    int lcls;
    long long kp0, jo0;
};
// components of a pair class and of its second shell
constexpr int pair_comps(int cls) { return cls == 0 ? 1 : cls == 1 ? 3 : cls == 2 ? 9 : cls == 3 ? 6 : cls == 4 ? 18 : 36; }
constexpr int pair_comps2(int cls) { return cls == 2 || cls == 4 ? 3 : cls == 5 ? 6 : 1; }

constexpr int kQuartSlots = 256;

// A launch as the kernel that lists a build's tasks sees it: candidate c of the launch (a bra and
// a ket segment) is thread (blockIdx - block0) * kTaskThreads + threadIdx
struct FockTaskSource {
    long long sp, blk;        // byte offsets of its tables
    int block0, ncand;
    int list;                 // its list's offset
    int f32;                  // the FP32 half of a mixed build
};
constexpr int kTaskThreads = 1024;
struct alignas(128) FockCounter {   // a cache line each
    int count, head;          // tasks listed, tasks handed out
    int pad[30];
};

struct FockArgs {
    const FockSpace* sp;
    const int* blk;           // space of every 64th block
    // the blocks of a launch take tasks until none is left: the listed ones, or (list null) every
    // candidate 0 .. ncand - 1
    const int* list;
    FockCounter* ctr;
    int ncand;
    const PairHdr* pairs;
    const PrimPair* prims;
    const BraPrim* bprim;
    const double* kprim;      // ket primitive fields, kps apart
    long long kps;
    const double* kgeo;       // kets' A and AB: six fields, npair apart
    long long npair;
    const int4* kidx;         // first functions and shells of the pair
    const int* knp;           // 2 x primitives + (same shell)
    const int2* kcol;         // LDS row columns of the pair's first functions
    const int* colinv;
    const double* pairQ;      // Schwarz bounds
    const double* dpair;      // max |D| of the pair's own shell block
    const double* dp;         // D0 in pair-major blocks
    double* jp;               // pair-major accumulator of the kets' Coulomb outputs
    const double* dsh;        // [nsh x nsh] max |D| of every shell block
    const double* dmax;       // largest of them, per molecule
    double tau, primcut;
    double fp32_thr;          // > 0: mixed build, quartets with a bound below it are FP32's
    int rys2_exact;
    int n, nsh;
    int dlds, mlds;           // density rows / shell maxima of the bra staged in LDS
    const double* D0;         // RHF: P (half density); UHF: Pa + Pb (dense n x n)
    const double* D1;         // UHF: Pa
    const double* D2;         // UHF: Pb
    double* W0;               // RHF: W; UHF: Wa
    double* W1;               // UHF: Wb
    const MolDesc* mols;      // batched launches: the molecules' slices of the stores
    const int* mol_active;    // per molecule: 0 skips its blocks
    unsigned long long* nquart;   // kQuartSlots counters: quartets within the bounds
    unsigned long long* counter;  // evaluated-quartet counters (may be null): kCounterSlots
                                  // (primitive, shell) pairs, summed by the host
    // deterministic accumulation (0: FP64 atomics): every W entry is two int64 words, the
    // word at the entry's own address and one fix_lo entries further on, holding the sum in
    // fixed point (integer additions give the same sum in any order); launches without LDS
    // rows only
    long long fix_lo;
};

}  // namespace uno
