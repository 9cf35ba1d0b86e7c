// Fock-build kernels: screened shell quartets, their ERIs (eri_core.hpp) and the fused J/K
// digestion, one launch per class pair.
//
// The quartet space of a launch is implicit.  A launch walks a short table of spaces
// (FockSpace): a run of bra pairs against a run of ket pairs, both sorted by Schwarz bound,
// descending.  A task is one bra of a space and one segment of its kets.  Which kets of a
// segment belong to the build (Q_ab Q_cd 4 max|D| >= tau, and on which side of the FP32
// threshold they lie) each lane reads off the bounds themselves against the density maximum in
// device memory.  So a build needs no index arrays from the host, no count there and no wait for
// the density bound.  In large builds one kernel first lists the tasks of every launch that
// hold any quartet (k_fock_tasks); a launch's blocks take tasks from a counter until none is
// left.  (Before: prefix and task arrays built and
// uploaded by the host per build, one launch per run pair -- 210 to 245 launches, of which a
// single water's 210 took 8.0 ms one after the other, 38 us each.)
//
// Data: the bra's records are the same for the whole block and read through the scalar cache
// (bra_prim).  The kets' are laid out field by field in run order, a run's primitives with the
// ket index fastest, so the lanes of a wave, consecutive kets, read consecutive addresses.
#pragma once
#include <hip/hip_runtime.h>
#include "eri_core.hpp"

namespace uno {

// classes up to kLaneMaxComp components run one ket per lane (the component block in registers);
// larger ones one quartet per wave
constexpr int kLaneMaxComp = 162;
// Rys tables of up to this many roots are staged in LDS by the kernels without LDS rows
constexpr int kLdsTabMaxRoots = 3;
// every quartet class: pair classes (0 ss, 1 ps, 2 pp, 3 ds, 4 dp, 5 dd) and shells
#define UNO_QUARTET_CLASSES(Q)                                                            \
    Q(0, 0, 0, 0, 0, 0)                                                                   \
    Q(1, 0, 1, 0, 0, 0) Q(1, 1, 1, 0, 1, 0)                                               \
    Q(2, 0, 1, 1, 0, 0) Q(2, 1, 1, 1, 1, 0) Q(2, 2, 1, 1, 1, 1)                           \
    Q(3, 0, 2, 0, 0, 0) Q(3, 1, 2, 0, 1, 0) Q(3, 2, 2, 0, 1, 1) Q(3, 3, 2, 0, 2, 0)       \
    Q(4, 0, 2, 1, 0, 0) Q(4, 1, 2, 1, 1, 0) Q(4, 2, 2, 1, 1, 1) Q(4, 3, 2, 1, 2, 0)       \
    Q(4, 4, 2, 1, 2, 1)                                                                   \
    Q(5, 0, 2, 2, 0, 0) Q(5, 1, 2, 2, 1, 0) Q(5, 2, 2, 2, 1, 1) Q(5, 3, 2, 2, 2, 0)       \
    Q(5, 4, 2, 2, 2, 1) Q(5, 5, 2, 2, 2, 2)

// a uniform read through the scalar cache: constant address space, uniform address
template <class S>
__device__ __forceinline__ const __attribute__((address_space(4))) S* scalar_ptr(const S* p) {
    return (const __attribute__((address_space(4))) S*)(unsigned long long)p;
}

template <class S>
__device__ __forceinline__ S scalar_load(const S* p) {
    static_assert(sizeof(S) % 4 == 0, "read in dwords");
    struct Words { unsigned w[sizeof(S) / 4]; } v;
    const auto* q = scalar_ptr(reinterpret_cast<const unsigned*>(p));
#pragma unroll
    for (unsigned i = 0; i < sizeof(S) / 4; ++i) v.w[i] = q[i];
    return __builtin_bit_cast(S, v);
}

// 64-lane butterfly sum
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    return v;
}

// The space and bra of a task, and its segment's kets [k0, k1) (indices in the ket run);
// false: nothing of it belongs to this build
struct FockTask {
    FockSpace s;
    int bra;          // pair index
    int ibra;         // index in the bra run
    int k0, k1;
    double qi, thr, t32;   // bra bound; kets at or above thr belong to the build, of those the
                           // ones below t32 to its FP32 half
    MolView mv;
    double dm;        // 4 max|D|
};

template <bool F32>
__device__ __forceinline__ bool fock_task(const FockArgs& a, const int b, FockTask& t) {
    // the table brackets the space of every 64th candidate
    const auto* bt = scalar_ptr(a.blk);
    int lo = bt[b >> 6], hi = bt[(b >> 6) + 1];
    const auto* sp = scalar_ptr(a.sp);
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sp[mid].first <= b) lo = mid; else hi = mid - 1;
    }
    t.s = scalar_load(a.sp + lo);
    const int l = b - t.s.first;
    t.ibra = l / t.s.nseg;
    const int seg = l - t.ibra * t.s.nseg;
    t.bra = t.s.bra_off + t.ibra;
    t.k0 = seg * t.s.seg;
    t.k1 = min(t.s.nket, t.k0 + t.s.seg);
    if (t.s.same) t.k1 = min(t.k1, t.ibra + 1);
    if (t.k0 >= t.k1) return false;
    int mol = 0;
    t.mv = MolView{a.D0, a.D1, a.D2, a.W0, a.W1, a.dsh, a.n, a.nsh};
    if (a.mols) {
        mol = t.s.mol;
        if (a.mol_active && !scalar_ptr(a.mol_active)[mol]) return false;   // already converged
        const MolDesc m = scalar_load(a.mols + mol);
        t.mv.D0 = a.D0 + m.moff;
        t.mv.D1 = a.D1 ? a.D1 + m.moff : nullptr;
        t.mv.D2 = a.D2 ? a.D2 + m.moff : nullptr;
        t.mv.W0 = a.W0 + m.moff;
        t.mv.W1 = a.W1 ? a.W1 + m.moff : nullptr;
        t.mv.dsh = a.dsh + m.dshoff;
        t.mv.n = m.n;
        t.mv.nsh = m.nsh;
    }
    t.dm = 4.0 * scalar_ptr(a.dmax)[mol];
    const auto* Q = scalar_ptr(a.pairQ);
    t.qi = Q[t.bra];
    const double qd = t.qi * t.dm;
    if (!(qd > 0.0)) return false;
    t.thr = a.tau / qd;
    if (Q[t.s.ket_off + t.k0] < t.thr) return false;
    t.t32 = 0.0;
    if (a.fp32_thr > 0.0) {
        t.t32 = a.fp32_thr / t.qi;
        if (F32 ? Q[t.s.ket_off + t.k1 - 1] >= t.t32 : Q[t.s.ket_off + t.k0] < t.t32) return false;
    }
    return true;
}

// How a launch's blocks share out its tasks, the costliest first: the first `grid` of them (or, for
// the many short tasks of the wave kernels, half of all) round robin, the rest to whoever asks
// next.  (All of them round robin leaves the launch waiting for its unluckiest block: 66 against
// 55 ms at 64 waters.  Every short task on request keeps thousands of waves on one counter at
// memory-side atomics' pace.)  A block asks for its next task ahead of the work on the current one.
struct FockQueue {
    int total, base;
    __device__ __forceinline__ FockQueue(const FockArgs& a, bool half) {
        total = a.list ? scalar_ptr(&a.ctr->count)[0] : a.ncand;
        const int grid = (int)gridDim.x;
        base = half ? max(grid, total / 2 / grid * grid) : grid;
    }
    __device__ __forceinline__ bool asks(int item) const { return item + (int)gridDim.x >= base && base < total; }
    __device__ __forceinline__ int ask(const FockArgs& a) const { return base + atomicAdd(&a.ctr->head, 1); }
    __device__ __forceinline__ int after(int item) const { return item + (int)gridDim.x; }
};

// whether ket k (bound q) belongs to this launch
template <bool F32>
__device__ __forceinline__ bool fock_ket_in(const FockTask& t, double q) {
    return q >= t.thr && (F32 ? q < t.t32 : q >= t.t32);
}

// ---------------------------------------------------------------------------
// Contracted (un-normalised) ERI block of one shell quartet: ket primitives outside, every
// 2^lg-th of them from `sub` on (the lanes of a group share a ket), the bra's primitives inside,
// from the scalar cache, the next record read while the current one is evaluated.  Returns the
// primitive quartets kept by the cut.
// ---------------------------------------------------------------------------
template <int LA, int LB, int LC, int LD, typename T>
__device__ __forceinline__ unsigned fock_eri(const FockArgs& a, const FockTask& t, int bra_prim0, int bra_nprim,
                                             const T* ab, int kidx, int knprim, int sub, int lg, T* e, const T* tab) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NA = CI::NA, NB = CI::NB, NC = CI::NC, ND = CI::ND, NCOMP = CI::NCOMP, NR = CI::NR;
#pragma unroll
    for (int c = 0; c < NCOMP; ++c) e[c] = 0;
    unsigned nprimq = 0;
    const int pair = t.s.ket_off + kidx;
    double A2[3] = {0.0, 0.0, 0.0};
    T cd[3] = {0, 0, 0};
    if constexpr (LC > 0) {
#pragma unroll
        for (int x = 0; x < 3; ++x) A2[x] = a.kgeo[(long)x * a.npair + pair];
    }
    if constexpr (LD > 0) {
#pragma unroll
        for (int x = 0; x < 3; ++x) cd[x] = (T)a.kgeo[(long)(3 + x) * a.npair + pair];
    }
    const BraPrim* bp = a.bprim + bra_prim0;
    const double* kp = a.kprim + t.s.kp0 + kidx;
    for (int jq = sub; jq < knprim; jq += 1 << lg) {
        const double* r = kp + (long)jq * t.s.kstride;
        const T q = (T)r[0], iq_ = (T)r[a.kps], kk = (T)r[2 * a.kps], sk = (T)r[3 * a.kps];
        const double Q[3] = {r[4 * a.kps], r[5 * a.kps], r[6 * a.kps]};
        // coordinate differences in double, then rounded to the compute type
        T QC[3] = {0, 0, 0};
        if constexpr (LC > 0) {
#pragma unroll
            for (int x = 0; x < 3; ++x) QC[x] = (T)(Q[x] - A2[x]);
        }
        BraPrim nx = scalar_load(bp);
        for (int ip = 0; ip < bra_nprim; ++ip) {
            const BraPrim pp = nx;
            nx = scalar_load(bp + (ip + 1 < bra_nprim ? ip + 1 : ip));
            const T p = (T)pp.p, ip_ = (T)pp.ip;
            // rt = (p+q)^(-1/2), it = 1/(p+q)
            const T rt = rsqrt_nr(p + q), it = rt * rt;
            if ((T)pp.s * sk * rt < (T)a.primcut) continue;
            ++nprimq;
            const T pref = (T)pp.K * kk * rt;
            const T PA[3] = {(T)pp.PA[0], (T)pp.PA[1], (T)pp.PA[2]};
            const T PQ[3] = {(T)(pp.P[0] - Q[0]), (T)(pp.P[1] - Q[1]), (T)(pp.P[2] - Q[2])};
            const T x = p * q * it * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
            T u[NR], w[NR];
            rys_roots<NR, T>(x, u, w, tab);
#pragma unroll
            for (int r2 = 0; r2 < NR; ++r2) {
                const T fff = u[r2] * it;
                const T B00 = (T)0.5 * fff;
                const T B1 = ((T)0.5 - B00 * q) * ip_;
                const T B1p = ((T)0.5 - B00 * p) * iq_;
                T Ix[CI::TBL], Iy[CI::TBL], Iz[CI::TBL];
                axis_table<LA, LB, LC, LD, T>(PA[0] - q * PQ[0] * fff, QC[0] + p * PQ[0] * fff, B00, B1, B1p, ab[0],
                                              cd[0], Ix);
                axis_table<LA, LB, LC, LD, T>(PA[1] - q * PQ[1] * fff, QC[1] + p * PQ[1] * fff, B00, B1, B1p, ab[1],
                                              cd[1], Iy);
                axis_table<LA, LB, LC, LD, T>(PA[2] - q * PQ[2] * fff, QC[2] + p * PQ[2] * fff, B00, B1, B1p, ab[2],
                                              cd[2], Iz);
                const T wr = w[r2] * pref;
#pragma unroll
                for (int i = 0; i < NA; ++i)
#pragma unroll
                    for (int j = 0; j < NB; ++j)
#pragma unroll
                        for (int k = 0; k < NC; ++k)
#pragma unroll
                            for (int l = 0; l < ND; ++l) {
                                const int c = ((i * NB + j) * NC + k) * ND + l;
                                e[c] = fma(wr * Ix[CI::tix(i, j, k, l, 0)], Iy[CI::tix(i, j, k, l, 1)] * Iz[CI::tix(i, j, k, l, 2)], e[c]);
                            }
            }
        }
    }
    // the group's partial blocks, summed into every lane of it
    for (int m = 1; m < 1 << lg; m <<= 1) {
#pragma unroll
        for (int c = 0; c < NCOMP; ++c) e[c] += __shfl_xor(e[c], m, 64);
    }
    return nprimq;
}

// normalisation (AuxFunctions.hpp:49-64) times a factor f
template <int LA, int LB, int LC, int LD, typename T>
__device__ __forceinline__ void normalise_block(T* e, T f) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NA = CI::NA, NB = CI::NB, NC = CI::NC, ND = CI::ND;
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int k = 0; k < NC; ++k)
#pragma unroll
                for (int l = 0; l < ND; ++l)
                    e[((i * NB + j) * NC + k) * ND + l] *=
                        f * (T)(cart_nrm(LA, i) * cart_nrm(LB, j) * cart_nrm(LC, k) * cart_nrm(LD, l));
}

// LDS layouts of the row kernels: kRowsNone every output straight to W, kRowsAll the rows of
// both bra shells merged in LDS, kRowsFirst those of the first shell only
enum RowsMode : int { kRowsNone = 0, kRowsAll = 1, kRowsFirst = 2 };

template <int LA, int LB, int MODE, int ROWS>
__host__ __device__ constexpr int row_count() {
    return ROWS == kRowsNone ? 0
                             : (ncart_c(LA) + (ROWS == kRowsAll ? ncart_c(LB) : 0)) * (MODE == kDigestUHF ? 2 : 1);
}
// rows of the staged exchange density (a.dlds): every bra function, per spin density
template <int LA, int LB, int MODE>
__host__ __device__ constexpr int dens_row_count() {
    return (ncart_c(LA) + ncart_c(LB)) * (MODE == kDigestUHF ? 2 : 1);
}

// four waves a block share its LDS rows (eight: (ds|ss) of 64 waters 6.4 -> 4.9 ms, most other
// classes and 16 waters slower)
constexpr int kRowThreads = 256, kRowWaves = kRowThreads / 64;
// waves per SIMD asked of the registers: the classes that miss two by little, 257 registers of (ds|ds)
// and 312 of (ds|pp), gain from holding to it (64 waters 1.49 -> 1.12 and 2.17 -> 1.76 ms); the ones
// that would spill more, from 350 on, lose (dd|ss 1.14 -> 1.76 ms)
template <int LA, int LB, int LC, int LD>
constexpr int row_min_waves() {
    return LA == 2 && LB == 0 && LC + LD == 2 ? 2 : 1;
}

// ---------------------------------------------------------------------------
// Classes of up to kLaneMaxComp components: one task per block at a time, one lane
// (or a group of 2^lg lanes, each with a share of the ket's primitives) per ket.  The
// exchange contributions all land in the bra's rows of W (rows fa.., fb..), so the block merges
// them in LDS (one row per bra function and spin, a column per function the ket class touches)
// and adds the non-zero entries at the end with row-contiguous atomics; the bra's Coulomb
// outputs are reduced over the block, the kets' go to the pair-major accumulator.  Also in
// LDS: the bra's row of shell-block density maxima (mlds), so that the screen reads one
// coalesced bound per ket and two LDS entries; with dlds the bra's exchange density rows; with
// TL the Rys table.
// ---------------------------------------------------------------------------
template <int LA, int LB, int LC, int LD, int MODE, typename T, int ROWS, bool TL>
__global__ __launch_bounds__(kRowThreads, (row_min_waves<LA, LB, LC, LD>())) void k_fock(const FockArgs a) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NA = CI::NA, NB = CI::NB, NC = CI::NC, ND = CI::ND, NCOMP = CI::NCOMP, NR = CI::NR;
    constexpr bool FB = ROWS == kRowsAll, RW = ROWS != kRowsNone, F32 = sizeof(T) == 4;
    constexpr int NAB = RW ? NA + (FB ? NB : 0) : 0, NROW = row_count<LA, LB, MODE, ROWS>();
    constexpr int NSP = MODE == kDigestUHF ? 2 : 1;
    constexpr int NDR = NA + NB;
    extern __shared__ double rows[];
    __shared__ T tab_lds[TL ? rys_table_size<NR, T>() : 1];
    __shared__ double jred[kRowWaves][NA * NB];
    __shared__ unsigned cred[kRowWaves][3];
    __shared__ int queue[kRowWaves][128];
    __shared__ int upcoming;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const T* tab = rys_table_of<NR, T>(a.rys2_exact);
    if constexpr (TL) {
        for (int i = threadIdx.x; i < rys_table_size<NR, T>(); i += kRowThreads) tab_lds[i] = tab[i];
        tab = tab_lds;
    }
    const FockQueue fq(a, false);
    for (int item = blockIdx.x; item < fq.total;) {
    const bool asks = fq.asks(item);
    if (asks && threadIdx.x == 0) upcoming = fq.ask(a);
    FockTask t;
    if (fock_task<F32>(a, a.list ? scalar_ptr(a.list)[item] : item, t)) {
    const MolView& mv = t.mv;
    const int n = mv.n, ns = mv.nsh, nc = t.s.ncols;
    const PairHdr P1 = scalar_load(a.pairs + t.bra);
    const int fa = P1.f1, fb = P1.f2;
    const int* colinv = a.colinv + t.s.col0;
    double* dlr = rows + NROW * nc;
    const bool dl = RW && a.dlds != 0;
    double* mrow = dlr + (dl ? NDR * NSP * nc : 0);
    const bool ml = a.mlds != 0;
    if constexpr (RW) {
        for (int i = threadIdx.x; i < NROW * nc; i += kRowThreads) rows[i] = 0.0;
        if (dl) {
            for (int i = threadIdx.x; i < NDR * NSP * nc; i += kRowThreads) {
                const int r = i / nc, col = i - r * nc;
                const int sp = r / NDR, rr = r - sp * NDR;
                const double* DK = (MODE == kDigestUHF) ? (sp == 0 ? mv.D1 : mv.D2) : mv.D0;
                const int grow = rr < NA ? fa + rr : fb + rr - NA;
                dlr[i] = DK[(long)grow * n + colinv[col]];
            }
        }
    }
    const double* m1 = mv.dsh + (long)P1.sh1 * ns;
    const double* m2 = mv.dsh + (long)P1.sh2 * ns;
    if (ml)
        for (int s = threadIdx.x; s < ns; s += kRowThreads) mrow[s] = fmax(m1[s], m2[s]);
    __syncthreads();
    const double dab4 = 4.0 * m1[P1.sh2];
    const T ab[3] = {(T)P1.AB[0], (T)P1.AB[1], (T)P1.AB[2]};
    constexpr T jf = (MODE == kDigestRHF) ? 4 : 2;
    double jacc[NA * NB];
    T dab[NA * NB];
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            jacc[i * NB + j] = 0.0;
            dab[i * NB + j] = (T)mv.D0[(long)(fa + i) * n + fb + j];
        }
    unsigned nprim = 0, nshell = 0, nin = 0;
    // Each wave screens its kets 64 at a time (fewer where the segment is short) into a queue of
    // survivors and evaluates them a wavefull at a time, so that the lanes it pays for are
    // busy: of the kets within the bounds two thirds survive the screen of a full build, and a
    // small part that of an incremental one.
    const int lg = t.s.lg, sub = lane & ((1 << lg) - 1), per = 64 >> lg;
    const int step = min(64, max(per, (t.k1 - t.k0 + kRowWaves - 1) / kRowWaves));
    int next = t.k0 + wave * step, nq = 0;
    int* q = queue[wave];
    for (;;) {
        while (nq < per && next < t.k1) {
            const int kk = next + lane;
            bool in = lane < step && kk < t.k1, live = false;
            if (in) {
                const int pcd = t.s.ket_off + kk;
                const double qk = a.pairQ[pcd];
                in = fock_ket_in<F32>(t, qk);
                if (in) {
                    // the density screen of eri_core.hpp's screened()
                    const int4 ki = a.kidx[pcd];
                    double d = fmax(dab4, 4.0 * a.dpair[pcd]);
                    if (ml) d = fmax(d, fmax(mrow[ki.z], mrow[ki.w]));
                    else d = fmax(d, fmax(fmax(m1[ki.z], m1[ki.w]), fmax(m2[ki.z], m2[ki.w])));
                    live = !(t.qi * qk * d < a.tau);
                }
            }
            const unsigned long long m = __ballot(live);
            nin += __popcll(__ballot(in));
            if (live) q[nq + __popcll(m & ((1ull << lane) - 1))] = kk;
            nq += __popcll(m);
            next += kRowWaves * step;
        }
        if (nq == 0) break;
        // the queue is the wave's own: its writes above precede its reads below
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const int take = min(nq, per);
        nq -= take;
        if ((lane >> lg) >= take) continue;
        const int kk = q[nq + (lane >> lg)];
        const int pcd = t.s.ket_off + kk;
        const int4 ki = a.kidx[pcd];   // first functions, shells
        const int kn = a.knp[pcd];     // primitives, twice, plus 1 for a same-shell pair
        T e[NCOMP];
        nprim += fock_eri<LA, LB, LC, LD, T>(a, t, P1.prim0, P1.nprim, ab, kk, kn >> 1, sub, lg, e, tab);
        if (sub) continue;
        ++nshell;
        const T f = (P1.same ? (T)0.5 : (T)1) * ((kn & 1) ? (T)0.5 : (T)1) * (t.bra == pcd ? (T)0.5 : (T)1);
        normalise_block<LA, LB, LC, LD, T>(e, f);
        const int fc = ki.x, fd = ki.y;
        // the ket's entries of the pair-major arrays: component by component over the run, so that
        // a wave's kets meet at consecutive addresses
        const long jo = t.s.jo0 + kk, js = t.s.kstride;
        // Coulomb, bra outputs: kept per thread
        {
            T dcd[NC * ND];
#pragma unroll
            for (int kl = 0; kl < NC * ND; ++kl) dcd[kl] = (T)a.dp[jo + kl * js];
#pragma unroll
            for (int ij = 0; ij < NA * NB; ++ij) {
                T s = 0;
#pragma unroll
                for (int kl = 0; kl < NC * ND; ++kl) s = fma(e[ij * NC * ND + kl], dcd[kl], s);
                jacc[ij] += (double)(jf * s);
            }
        }
        // Coulomb, ket outputs: one atomic each, into the pair-major accumulator (a wave's kets
        // are consecutive there), or in deterministic builds straight into W
#pragma unroll
        for (int kl = 0; kl < NC * ND; ++kl) {
            T s = 0;
#pragma unroll
            for (int ij = 0; ij < NA * NB; ++ij) s = fma(e[ij * NC * ND + kl], dab[ij], s);
            const double v = (double)(jf * s);
            if (RW || a.jp) {
                atomic_add_f64(a.jp + jo + kl * js, v);
            } else {
                const long o = (long)(fc + kl / ND) * n + fd + kl % ND;
                fock_add(a.fix_lo, mv.W0 + o, v);
                if (MODE == kDigestUHF) fock_add(a.fix_lo, mv.W1 + o, v);
            }
        }
        int lc = 0, ld = 0;   // the ket's LDS row columns
        if constexpr (RW) {
            const int2 kc = a.kcol[pcd];
            lc = kc.x;
            ld = kc.y;
        }
        // exchange, once per spin density
#pragma unroll
        for (int sp = 0; sp < NSP; ++sp) {
            const double* DK = (MODE == kDigestUHF) ? (sp == 0 ? mv.D1 : mv.D2) : mv.D0;
            double* R = rows + sp * NAB * nc;
            double* W = (MODE == kDigestUHF && sp) ? mv.W1 : mv.W0;
            T dbd[NB * ND], dbc[NB * NC], dad[NA * ND], dac[NA * NC];
            if (RW && dl) {
                const double* DR = dlr + sp * NDR * nc;
#pragma unroll
                for (int j = 0; j < NB; ++j) {
#pragma unroll
                    for (int l = 0; l < ND; ++l) dbd[j * ND + l] = (T)DR[(NA + j) * nc + ld + l];
#pragma unroll
                    for (int k = 0; k < NC; ++k) dbc[j * NC + k] = (T)DR[(NA + j) * nc + lc + k];
                }
#pragma unroll
                for (int i = 0; i < NA; ++i) {
#pragma unroll
                    for (int l = 0; l < ND; ++l) dad[i * ND + l] = (T)DR[i * nc + ld + l];
#pragma unroll
                    for (int k = 0; k < NC; ++k) dac[i * NC + k] = (T)DR[i * nc + lc + k];
                }
            } else {
#pragma unroll
                for (int j = 0; j < NB; ++j) {
#pragma unroll
                    for (int l = 0; l < ND; ++l) dbd[j * ND + l] = (T)DK[(long)(fb + j) * n + fd + l];
#pragma unroll
                    for (int k = 0; k < NC; ++k) dbc[j * NC + k] = (T)DK[(long)(fb + j) * n + fc + k];
                }
#pragma unroll
                for (int i = 0; i < NA; ++i) {
#pragma unroll
                    for (int l = 0; l < ND; ++l) dad[i * ND + l] = (T)DK[(long)(fa + i) * n + fd + l];
#pragma unroll
                    for (int k = 0; k < NC; ++k) dac[i * NC + k] = (T)DK[(long)(fa + i) * n + fc + k];
                }
            }
            // output (bra function row r of its shell's, ket column): LDS row, or W
            auto put = [&](bool second, int r, int lcol, int gcol, T s) {
                if (RW && (!second || FB)) atomicAdd(R + (second ? NA + r : r) * nc + lcol, (double)(-s));
                else fock_add(RW ? 0 : a.fix_lo, W + (long)((second ? fb : fa) + r) * n + gcol, (double)(-s));
            };
#pragma unroll
            for (int i = 0; i < NA; ++i) {
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    T s = 0;
#pragma unroll
                    for (int j = 0; j < NB; ++j)
#pragma unroll
                        for (int l = 0; l < ND; ++l) s = fma(e[((i * NB + j) * NC + k) * ND + l], dbd[j * ND + l], s);
                    put(false, i, lc + k, fc + k, s);
                }
#pragma unroll
                for (int l = 0; l < ND; ++l) {
                    T s = 0;
#pragma unroll
                    for (int j = 0; j < NB; ++j)
#pragma unroll
                        for (int k = 0; k < NC; ++k) s = fma(e[((i * NB + j) * NC + k) * ND + l], dbc[j * NC + k], s);
                    put(false, i, ld + l, fd + l, s);
                }
            }
#pragma unroll
            for (int j = 0; j < NB; ++j) {
#pragma unroll
                for (int k = 0; k < NC; ++k) {
                    T s = 0;
#pragma unroll
                    for (int i = 0; i < NA; ++i)
#pragma unroll
                        for (int l = 0; l < ND; ++l) s = fma(e[((i * NB + j) * NC + k) * ND + l], dad[i * ND + l], s);
                    put(true, j, lc + k, fc + k, s);
                }
#pragma unroll
                for (int l = 0; l < ND; ++l) {
                    T s = 0;
#pragma unroll
                    for (int i = 0; i < NA; ++i)
#pragma unroll
                        for (int k = 0; k < NC; ++k) s = fma(e[((i * NB + j) * NC + k) * ND + l], dac[i * NC + k], s);
                    put(true, j, ld + l, fd + l, s);
                }
            }
        }
    }
    // bra Coulomb outputs: wave sums, then the four waves
#pragma unroll
    for (int ij = 0; ij < NA * NB; ++ij) {
        const double v = wave_sum(jacc[ij]);
        if (lane == 0) jred[wave][ij] = v;
    }
    if (a.counter) {
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) {
            nprim += __shfl_xor(nprim, m, 64);
            nshell += __shfl_xor(nshell, m, 64);
        }
    }
    if (lane == 0) {
        cred[wave][0] = nin;
        cred[wave][1] = nprim;
        cred[wave][2] = nshell;
    }
    __syncthreads();
    if (threadIdx.x < NA * NB) {
        const int i = threadIdx.x / NB, j = threadIdx.x % NB;
        double v = 0.0;
#pragma unroll
        for (int w = 0; w < kRowWaves; ++w) v += jred[w][threadIdx.x];
        const long o = (long)(fa + i) * n + fb + j;
        fock_add(RW ? 0 : a.fix_lo, mv.W0 + o, v);
        if (MODE == kDigestUHF) fock_add(RW ? 0 : a.fix_lo, mv.W1 + o, v);
    }
    if (threadIdx.x == 0) {
        unsigned long long c0 = 0, c1 = 0, c2 = 0;
        for (int w = 0; w < kRowWaves; ++w) {
            c0 += cred[w][0];
            c1 += cred[w][1];
            c2 += cred[w][2];
        }
        atomicAdd(a.nquart + (item & (kQuartSlots - 1)), c0);
        if (a.counter) {
            unsigned long long* slot = a.counter + 2 * (item & (kCounterSlots - 1));
            atomicAdd(slot, c1);
            atomicAdd(slot + 1, c2);
        }
    }
    // merged exchange rows: consecutive threads take consecutive columns of a row
#pragma unroll
    for (int r = 0; r < NROW; ++r) {
        const int sp = r / (NAB ? NAB : 1), rr = r - sp * NAB;
        const int grow = rr < NA ? fa + rr : fb + rr - NA;
        double* W = (MODE == kDigestUHF && sp) ? mv.W1 : mv.W0;
        for (int col = threadIdx.x; col < nc; col += kRowThreads) {
            const double v = rows[r * nc + col];
            if (v != 0.0) atomic_add_f64(W + (long)grow * n + colinv[col], v);
        }
    }
    }
    __syncthreads();   // every wave is done with this task's LDS
    if (asks) {
        item = __builtin_amdgcn_readfirstlane(upcoming);
        __syncthreads();
    } else {
        item = fq.after(item);
    }
    }
}

template <typename V>
__device__ __forceinline__ V sel3(int ax, V a0, V a1, V a2) {
    return ax == 0 ? a0 : (ax == 1 ? a1 : a2);
}

// ---------------------------------------------------------------------------
// one 64-lane wave (one block) per shell quartet, already resolved (and screened) to its
// bra pair, ket pair, entry and bound
// ---------------------------------------------------------------------------
// One (root, axis) of the wave kernel: the 2-D recurrence G[e][f] scaled by wz (the weight
// times the prefactor on the z axis), the ket transfer H[e][c][d] = sum_j C(d,j) cd^j
// G[e][c+d-j] and the bra transfer I[a][b][c][d] = sum_i C(b,i) ab^i H[a+b-i][c][d], all
// unrolled at compile time, each I entry stored (to LDS) as it is formed
template <int LA, int LB, int LC, int LD, typename T>
__device__ __forceinline__ void wave_axis(T C, T Cp, T B00, T B1, T B1p, T ab, T cd, T wz, T* I) {
    constexpr int E = LA + LB, F = LC + LD;
    T G[E + 1][F + 1];
    G[0][0] = 1;
    if constexpr (E > 0) G[1][0] = C;
#pragma unroll
    for (int e = 1; e < E; ++e) G[e + 1][0] = (T)e * B1 * G[e - 1][0] + C * G[e][0];
#pragma unroll
    for (int f = 0; f < F; ++f)
#pragma unroll
        for (int e = 0; e <= E; ++e) {
            T v = Cp * G[e][f];
            if (f > 0) v = fma((T)f * B1p, G[e][f - 1], v);
            if (e > 0) v = fma((T)e * B00, G[e - 1][f], v);
            G[e][f + 1] = v;
        }
#pragma unroll
    for (int e = 0; e <= E; ++e)
#pragma unroll
        for (int f = 0; f <= F; ++f) G[e][f] *= wz;
    T cdp[LD + 1], abp[LB + 1];
    cdp[0] = 1;
#pragma unroll
    for (int j = 1; j <= LD; ++j) cdp[j] = cdp[j - 1] * cd;
    abp[0] = 1;
#pragma unroll
    for (int i = 1; i <= LB; ++i) abp[i] = abp[i - 1] * ab;
    T H[E + 1][LC + 1][LD + 1];
#pragma unroll
    for (int e = 0; e <= E; ++e)
#pragma unroll
        for (int c = 0; c <= LC; ++c)
#pragma unroll
            for (int d = 0; d <= LD; ++d) {
                T v = 0;
#pragma unroll
                for (int j = 0; j <= d; ++j) v = fma((T)binom_c(d, j) * cdp[j], G[e][c + d - j], v);
                H[e][c][d] = v;
            }
#pragma unroll
    for (int a = 0; a <= LA; ++a)
#pragma unroll
        for (int b = 0; b <= LB; ++b)
#pragma unroll
            for (int c = 0; c <= LC; ++c)
#pragma unroll
                for (int d = 0; d <= LD; ++d) {
                    T v = 0;
#pragma unroll
                    for (int i = 0; i <= b; ++i) v = fma((T)binom_c(b, i) * abp[i], H[a + b - i][c][d], v);
                    I[((a * (LB + 1) + b) * (LC + 1) + c) * (LD + 1) + d] = v;
                }
}

// per component c of a class (the wave kernel's order): its 2-D table index on each
// axis (x | y << 8 | z << 16) and the number of x^2, y^2, z^2 d functions among its four
// (<< 24), fixed at compile time
template <int LA, int LB, int LC, int LD>
struct WaveCompTab {
    int v[ClassInfo<LA, LB, LC, LD>::NCOMP];
    constexpr WaveCompTab() : v() {
        using CI = ClassInfo<LA, LB, LC, LD>;
        for (int c = 0; c < CI::NCOMP; ++c) {
            const int l = c % CI::ND, k = (c / CI::ND) % CI::NC, j = (c / (CI::ND * CI::NC)) % CI::NB,
                      i = c / (CI::ND * CI::NC * CI::NB);
            const int nd2 = (cart_nrm(LA, i) != 1.0) + (cart_nrm(LB, j) != 1.0) + (cart_nrm(LC, k) != 1.0) +
                            (cart_nrm(LD, l) != 1.0);
            v[c] = CI::tix(i, j, k, l, 0) | CI::tix(i, j, k, l, 1) << 8 | CI::tix(i, j, k, l, 2) << 16 | nd2 << 24;
        }
    }
};

// ---------------------------------------------------------------------------
// One shell quartet by one 64-lane wave (one block): the component block, normalised and times
// f, in LDS.  The two pairs are uniform, their records read through the scalar cache.  Lanes < NR
// compute a root and weight each, lanes < 3 NR a (root, axis) recurrence and transfer, and the
// components are split over all lanes.  Returns the primitive quartets kept by the cut.
// ---------------------------------------------------------------------------
template <int LA, int LB, int LC, int LD, typename T>
__device__ __forceinline__ unsigned wave_eri(const PairHdr& P1, const PairHdr& P2, const PrimPair* prims, double primcut,
                                             int rys2_exact, T f, T* sE) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NCOMP = CI::NCOMP, NR = CI::NR, TBL = CI::TBL;
    constexpr int PER = (NCOMP + 63) / 64;
    __shared__ T sUW[2 * NR];
    __shared__ T sI[NR * 3][TBL];
    const int lane = threadIdx.x;
    // each lane owns components lane + 64 m: their table indices from the class's table
    static constexpr WaveCompTab<LA, LB, LC, LD> kComp{};
    // (kept packed, one register per component, unpacked where used)
    int cix[PER];
    T acc[PER];
#pragma unroll
    for (int m = 0; m < PER; ++m) {
        acc[m] = 0;
        const int c = lane + 64 * m;
        cix[m] = kComp.v[c < NCOMP ? c : 0];
    }
    // a (root, axis) lane's axis, picked by selects, not by a dynamic index (which would put the
    // records in scratch memory)
    const int rr = lane / 3, ax = lane - 3 * rr;
    const T abx = (T)sel3(ax, P1.AB[0], P1.AB[1], P1.AB[2]), cdx = (T)sel3(ax, P2.AB[0], P2.AB[1], P2.AB[2]);
    unsigned nprimq = 0;
    for (int ip = 0; ip < P1.nprim; ++ip) {
        const PrimPair pp = scalar_load(prims + P1.prim0 + ip);
        for (int iq = 0; iq < P2.nprim; ++iq) {
            const PrimPair qq = scalar_load(prims + P2.prim0 + iq);
            const T p = (T)pp.p, q = (T)qq.p, ip_ = (T)pp.ip, iq_ = (T)qq.ip;
            const T rt = rsqrt_nr(p + q), it = rt * rt;
            const T bare = (T)kTwoPi25 * (T)pp.s * (T)qq.s * ip_ * iq_ * rt;
            if (bare < (T)primcut) continue;   // uniform across the block
            ++nprimq;
            const T pref = (T)kTwoPi25 * (T)pp.K * (T)qq.K * ip_ * iq_ * rt;
            const T PQ[3] = {(T)(pp.P[0] - qq.P[0]), (T)(pp.P[1] - qq.P[1]), (T)(pp.P[2] - qq.P[2])};
            const T x = p * q * it * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
            if (lane < NR) {
                // root lane
                T u, w;
                rys_root_one<NR, T>(x, lane, u, w, rys_table_of<NR, T>(rys2_exact));
                sUW[lane] = u;
                sUW[NR + lane] = w * pref;
            }
            __syncthreads();
            if (lane < 3 * NR) {
                // (root, axis): recurrence and transfer in registers, the transferred table into
                // LDS
                const T fff = sUW[rr] * it;
                const T B00 = (T)0.5 * fff, B1 = ((T)0.5 - B00 * q) * ip_, B1p = ((T)0.5 - B00 * p) * iq_;
                const T pqa = sel3(ax, PQ[0], PQ[1], PQ[2]);
                const T C = (T)sel3(ax, pp.P[0] - P1.A[0], pp.P[1] - P1.A[1], pp.P[2] - P1.A[2]) - q * pqa * fff;
                const T Cp = (T)sel3(ax, qq.P[0] - P2.A[0], qq.P[1] - P2.A[1], qq.P[2] - P2.A[2]) + p * pqa * fff;
                const T wz = (ax == 2) ? sUW[NR + rr] : (T)1;   // weight x prefactor folded into z
                wave_axis<LA, LB, LC, LD, T>(C, Cp, B00, B1, B1p, abx, cdx, wz, sI[lane]);
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < PER; ++m) {
                if (lane + 64 * m < NCOMP) {
                    const int ix = cix[m] & 255, iy = (cix[m] >> 8) & 255, iz = (cix[m] >> 16) & 255;
                    T s = acc[m];
#pragma unroll
                    for (int r = 0; r < NR; ++r) s = fma(sI[3 * r][ix] * sI[3 * r + 1][iy], sI[3 * r + 2][iz], s);
                    acc[m] = s;
                }
            }
            __syncthreads();
        }
    }
#pragma unroll
    for (int m = 0; m < PER; ++m) {
        const int c = lane + 64 * m;
        if (c < NCOMP) {
            // component normalisation: 1/sqrt(3) per x^2, y^2 or z^2 d function among the four
            T cn = 1;
            for (int q = kComp.v[c] >> 24; q > 0; --q) cn *= 0.57735026918962576451;
            sE[c] = acc[m] * f * cn;
        }
    }
    __syncthreads();
    return nprimq;
}

// waves per SIMD the register allocation must allow: three up to 324 components ((dp|dp),
// (dd|pp) then fit without spilling), two up to 648, one for (dd|dd)
template <int LA, int LB, int LC, int LD>
constexpr int wave_min_waves() {
    return ClassInfo<LA, LB, LC, LD>::NCOMP <= 324 ? 3 : ClassInfo<LA, LB, LC, LD>::NCOMP <= 648 ? 2 : 1;
}

// ---------------------------------------------------------------------------
// Larger classes: one wave (one block) per task (a segment of up to 64 kets, the host's choice is
// kWaveSeg).  Lane i screens ket i, then the wave evaluates the survivors one after another and
// adds their outputs to W.  Segments stay short: the blocks are many, so enough waves are in
// flight to cover each one's serial latency (64 per block was measured 2.5x slower).
// ---------------------------------------------------------------------------
template <int LA, int LB, int LC, int LD, int MODE, typename T>
__global__ __launch_bounds__(64, (wave_min_waves<LA, LB, LC, LD>())) void k_fock_wave(const FockArgs a) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NA = CI::NA, NB = CI::NB, NC = CI::NC, ND = CI::ND, NCOMP = CI::NCOMP;
    constexpr bool F32 = sizeof(T) == 4;
    __shared__ T sE[NCOMP];
    const int lane = threadIdx.x;
    const FockQueue fq(a, true);
    for (int item = blockIdx.x; item < fq.total;) {
    const bool asks = fq.asks(item);
    int upcoming = 0;
    if (asks && lane == 0) upcoming = fq.ask(a);
    FockTask t;
    if (fock_task<F32>(a, a.list ? scalar_ptr(a.list)[item] : item, t)) {
    const MolView& mv = t.mv;
    const PairHdr P1 = scalar_load(a.pairs + t.bra);
    const int pcd = t.s.ket_off + t.k0 + lane;
    bool in = false, live = false;
    if (t.k0 + lane < t.k1) {
        const double qk = a.pairQ[pcd];
        in = fock_ket_in<F32>(t, qk);
        const int4 ki = a.kidx[pcd];
        live = in && !screened(a.tau, mv, P1.sh1, P1.sh2, ki.z, ki.w, t.qi * qk);
    }
    const int nin = __popcll(__ballot(in));
    unsigned long long todo = __ballot(live);
    unsigned long long nprim = 0, nshell = 0;
    while (todo) {
        const int src = __builtin_ctzll(todo);
        todo &= todo - 1;
        const int qcd = t.s.ket_off + t.k0 + src;
        const PairHdr P2 = scalar_load(a.pairs + qcd);
        const T f = (P1.same ? (T)0.5 : (T)1) * (P2.same ? (T)0.5 : (T)1) * (t.bra == qcd ? (T)0.5 : (T)1);
        nprim += wave_eri<LA, LB, LC, LD, T>(P1, P2, a.prims, a.primcut, a.rys2_exact, f, sE);
        ++nshell;
        const int n = mv.n;
        const int fa = P1.f1, fb = P1.f2, fc = P2.f1, fd = P2.f2;
        constexpr T jf = (MODE == kDigestRHF) ? 4 : 2;
        // Coulomb outputs: NA*NB (bra) + NC*ND (ket)
        for (int o = lane; o < NA * NB + NC * ND; o += 64) {
            T s = 0;
            if (o < NA * NB) {
                const int i = o / NB, j = o % NB;
                for (int k = 0; k < NC; ++k)
                    for (int l = 0; l < ND; ++l)
                        s = fma(sE[((i * NB + j) * NC + k) * ND + l], (T)mv.D0[(long)(fc + k) * n + fd + l], s);
                fock_add(a.fix_lo, mv.W0 + (long)(fa + i) * n + fb + j, (double)(jf * s));
                if (MODE == kDigestUHF) fock_add(a.fix_lo, mv.W1 + (long)(fa + i) * n + fb + j, (double)(jf * s));
            } else {
                const int kl = o - NA * NB, k = kl / ND, l = kl % ND;
                for (int i = 0; i < NA; ++i)
                    for (int j = 0; j < NB; ++j)
                        s = fma(sE[((i * NB + j) * NC + k) * ND + l], (T)mv.D0[(long)(fa + i) * n + fb + j], s);
                // straight into W (a wave's lanes already cover the ket block's contiguous rows)
                fock_add(a.fix_lo, mv.W0 + (long)(fc + k) * n + fd + l, (double)(jf * s));
                if (MODE == kDigestUHF) fock_add(a.fix_lo, mv.W1 + (long)(fc + k) * n + fd + l, (double)(jf * s));
            }
        }
        constexpr int NK = NA * NC + NA * ND + NB * NC + NB * ND;
        for (int sp = 0; sp < (MODE == kDigestUHF ? 2 : 1); ++sp) {
            const double* DK = (MODE == kDigestUHF) ? (sp == 0 ? mv.D1 : mv.D2) : mv.D0;
            double* W = sp == 0 ? mv.W0 : mv.W1;
            for (int o = lane; o < NK; o += 64) {
                T s = 0;
                if (o < NA * NC) {                       // (a,c) <- D_bd
                    const int i = o / NC, k = o % NC;
                    for (int j = 0; j < NB; ++j)
                        for (int l = 0; l < ND; ++l)
                            s = fma(sE[((i * NB + j) * NC + k) * ND + l], (T)DK[(long)(fb + j) * n + fd + l], s);
                    fock_add(a.fix_lo, W + (long)(fa + i) * n + fc + k, (double)(-s));
                } else if (o < NA * NC + NA * ND) {      // (a,d) <- D_bc
                    const int q = o - NA * NC, i = q / ND, l = q % ND;
                    for (int j = 0; j < NB; ++j)
                        for (int k = 0; k < NC; ++k)
                            s = fma(sE[((i * NB + j) * NC + k) * ND + l], (T)DK[(long)(fb + j) * n + fc + k], s);
                    fock_add(a.fix_lo, W + (long)(fa + i) * n + fd + l, (double)(-s));
                } else if (o < NA * NC + NA * ND + NB * NC) {   // (b,c) <- D_ad
                    const int q = o - NA * NC - NA * ND, j = q / NC, k = q % NC;
                    for (int i = 0; i < NA; ++i)
                        for (int l = 0; l < ND; ++l)
                            s = fma(sE[((i * NB + j) * NC + k) * ND + l], (T)DK[(long)(fa + i) * n + fd + l], s);
                    fock_add(a.fix_lo, W + (long)(fb + j) * n + fc + k, (double)(-s));
                } else {                                 // (b,d) <- D_ac
                    const int q = o - NA * NC - NA * ND - NB * NC, j = q / ND, l = q % ND;
                    for (int i = 0; i < NA; ++i)
                        for (int k = 0; k < NC; ++k)
                            s = fma(sE[((i * NB + j) * NC + k) * ND + l], (T)DK[(long)(fa + i) * n + fc + k], s);
                    fock_add(a.fix_lo, W + (long)(fb + j) * n + fd + l, (double)(-s));
                }
            }
        }
        __syncthreads();
    }
    if (lane == 0) {
        atomicAdd(a.nquart + (item & (kQuartSlots - 1)), (unsigned long long)nin);
        if (a.counter && nshell) {
            unsigned long long* slot = a.counter + 2 * (item & (kCounterSlots - 1));
            atomicAdd(slot, nprim);
            atomicAdd(slot + 1, nshell);
        }
    }
    }
    item = asks ? __builtin_amdgcn_readfirstlane(upcoming) : fq.after(item);
    }
}

}  // namespace uno
