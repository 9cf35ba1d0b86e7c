// ERI kernels of explicit quartet lists (blocks, Schwarz bounds), the Fock-build launch
// configuration, and the small kernels around a Fock build.  See eri_core.hpp for the
// mathematics, fock_core.hpp for the Fock kernels.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "fock_core.hpp"
#include "kernels.hpp"

namespace uno {

// ---------------------------------------------------------------------------
// contracted (un-normalised) ERI block of one shell quartet in one lane.  Ket primitives outside, bra primitives inside; the
// next bra primitive record is fetched while the current one is evaluated.  tab is the
// Rys table of this class's root count (global or an LDS copy).
// ---------------------------------------------------------------------------
template <int LA, int LB, int LC, int LD, typename T>
__device__ __forceinline__ void eri_block(const EriArgs& a, const PairHdr& P1, const PairHdr& P2, T* e,
                                              const T* tab) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NA = CI::NA, NB = CI::NB, NC = CI::NC, ND = CI::ND, NCOMP = CI::NCOMP, NR = CI::NR;
#pragma unroll
    for (int c = 0; c < NCOMP; ++c) e[c] = 0;
    const T ab[3] = {(T)P1.AB[0], (T)P1.AB[1], (T)P1.AB[2]};
    const T cd[3] = {(T)P2.AB[0], (T)P2.AB[1], (T)P2.AB[2]};
    const PrimPair* bp = a.prims + P1.prim0;
    for (int iq = 0; iq < P2.nprim; ++iq) {
        const PrimPair qq = a.prims[P2.prim0 + iq];
        const T q = (T)qq.p, iq_ = (T)qq.ip, sq = (T)qq.s, Kq = (T)qq.K;
        // coordinate differences in double, then rounded to the compute type
        const T QC[3] = {(T)(qq.P[0] - P2.A[0]), (T)(qq.P[1] - P2.A[1]), (T)(qq.P[2] - P2.A[2])};
        PrimPair nx;
        if (P1.nprim > 0) nx = bp[0];
        for (int ip = 0; ip < P1.nprim; ++ip) {
            const PrimPair pp = nx;
            if (ip + 1 < P1.nprim) nx = bp[ip + 1];
            const T p = (T)pp.p, ip_ = (T)pp.ip;
            // rt = (p+q)^(-1/2), it = 1/(p+q)
            const T rt = rsqrt_nr(p + q), it = rt * rt;
            const T bare = (T)kTwoPi25 * (T)pp.s * sq * ip_ * iq_ * rt;
            if (bare < (T)a.primcut) continue;
            const T pref = (T)kTwoPi25 * (T)pp.K * Kq * ip_ * iq_ * rt;
            const T PA[3] = {(T)(pp.P[0] - P1.A[0]), (T)(pp.P[1] - P1.A[1]), (T)(pp.P[2] - P1.A[2])};
            const T PQ[3] = {(T)(pp.P[0] - qq.P[0]), (T)(pp.P[1] - qq.P[1]), (T)(pp.P[2] - qq.P[2])};
            const T x = p * q * it * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
            T u[NR], w[NR];
            rys_roots<NR, T>(x, u, w, tab);
#pragma unroll
            for (int r = 0; r < NR; ++r) {
                const T fff = u[r] * it;
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
                const T wr = w[r] * pref;
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
}

// ---------------------------------------------------------------------------
// one lane per shell quartet of an explicit list (block / Schwarz modes)
// ---------------------------------------------------------------------------
template <int LA, int LB, int LC, int LD, typename T>
__global__ __launch_bounds__(256) void k_eri_lane(const EriArgs a) {
    constexpr int NCOMP = ClassInfo<LA, LB, LC, LD>::NCOMP;
    const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= a.nquart) return;
    const PairHdr P1 = a.pairs[a.explicit_q[g].x];
    const PairHdr P2 = a.pairs[a.explicit_q[g].y];
    T e[NCOMP];
    eri_block<LA, LB, LC, LD, T>(a, P1, P2, e, rys_table_of<ClassInfo<LA, LB, LC, LD>::NR, T>(a.rys2_exact));
    normalise_block<LA, LB, LC, LD, T>(e, (T)1);
#pragma unroll
    for (int c = 0; c < NCOMP; ++c) a.out[g * NCOMP + c] = (double)e[c];
}

// Schwarz bound of a pair: only the diagonal components (ij|ij), and each unordered pair of its
// primitives once (a product pair and its exchange give the same diagonal).  Bound by its longest
// chain, the 36 x 36 primitives of two first-row core shells, so kSchwarzLanes lanes share a pair's
// primitive quartets: 32 waters (ss|ss) 15 us, (ps|ps) 14 us (a pair per lane, whole blocks:
// 246 and 451 us).
constexpr int kSchwarzLanes = 16;
template <int LA, int LB>
__global__ __launch_bounds__(256) void k_schwarz(const EriArgs a) {
    using CI = ClassInfo<LA, LB, LA, LB>;
    constexpr int NA = CI::NA, NB = CI::NB, NR = CI::NR;
    const long long gt = (long long)blockIdx.x * 256 + threadIdx.x;
    const long long g = gt / kSchwarzLanes;
    const int sub = (int)(gt % kSchwarzLanes);
    if (g >= a.nquart) return;   // the group's lanes together
    const int pair = a.explicit_q[g].x;
    const PairHdr P = a.pairs[pair];
    const double* tab = rys_table_of<NR, double>(a.rys2_exact);
    double e[NA * NB];
#pragma unroll
    for (int c = 0; c < NA * NB; ++c) e[c] = 0.0;
    // row i, column j <= i of the primitive triangle, kSchwarzLanes entries at a time
    int i = 0, j = sub;
    for (;;) {
        while (i < P.nprim && j > i) j -= ++i;
        if (i >= P.nprim) break;
        const PrimPair pp = a.prims[P.prim0 + i], qq = a.prims[P.prim0 + j];
        const double p = pp.p, q = qq.p;
        const double rt = rsqrt_nr(p + q), it = rt * rt;
        const double pref = kTwoPi25 * pp.K * qq.K * pp.ip * qq.ip * rt * (i == j ? 1.0 : 2.0);
        const double PQ[3] = {pp.P[0] - qq.P[0], pp.P[1] - qq.P[1], pp.P[2] - qq.P[2]};
        const double x = p * q * it * (PQ[0] * PQ[0] + PQ[1] * PQ[1] + PQ[2] * PQ[2]);
        double u[NR], w[NR];
        rys_roots<NR, double>(x, u, w, tab);
#pragma unroll
        for (int r = 0; r < NR; ++r) {
            const double fff = u[r] * it;
            const double B00 = 0.5 * fff, B1 = (0.5 - B00 * q) * pp.ip, B1p = (0.5 - B00 * p) * qq.ip;
            double I[3][CI::TBL];
#pragma unroll
            for (int ax = 0; ax < 3; ++ax)
                axis_table<LA, LB, LA, LB, double>(pp.P[ax] - P.A[ax] - q * PQ[ax] * fff, qq.P[ax] - P.A[ax] + p * PQ[ax] * fff,
                                                   B00, B1, B1p, P.AB[ax], P.AB[ax], I[ax]);
            const double wr = w[r] * pref;
#pragma unroll
            for (int ca = 0; ca < NA; ++ca)
#pragma unroll
                for (int cb = 0; cb < NB; ++cb)
                    e[ca * NB + cb] = fma(wr * I[0][CI::tix(ca, cb, ca, cb, 0)],
                                          I[1][CI::tix(ca, cb, ca, cb, 1)] * I[2][CI::tix(ca, cb, ca, cb, 2)], e[ca * NB + cb]);
        }
        j += kSchwarzLanes;
    }
    double m = 0.0;
#pragma unroll
    for (int ca = 0; ca < NA; ++ca)
#pragma unroll
        for (int cb = 0; cb < NB; ++cb) {
            double v = e[ca * NB + cb];
#pragma unroll
            for (int o = 1; o < kSchwarzLanes; o <<= 1) v += __shfl_xor(v, o, kSchwarzLanes);
            // each function's normalisation stands twice in (ij|ij)
            const double nrm = cart_nrm(LA, ca) * cart_nrm(LB, cb);
            m = fmax(m, fabs(v * (nrm * nrm)));
        }
    if (sub == 0) a.out[pair] = sqrt(m);
}

// one quartet of an explicit list per wave (classes of more than kLaneMaxComp components)
template <int LA, int LB, int LC, int LD, int MODE, typename T>
__global__ __launch_bounds__(64, (wave_min_waves<LA, LB, LC, LD>())) void k_eri_wave(const EriArgs a) {
    using CI = ClassInfo<LA, LB, LC, LD>;
    constexpr int NA = CI::NA, NB = CI::NB, NC = CI::NC, ND = CI::ND, NCOMP = CI::NCOMP;
    __shared__ T sE[NCOMP];
    const int lane = threadIdx.x;
    const long long g1 = min(a.nquart, ((long long)blockIdx.x + 1) * a.qpb);
    for (long long g = (long long)blockIdx.x * a.qpb; g < g1; ++g) {
        const int2 q = scalar_load(a.explicit_q + g);
        const PairHdr P1 = scalar_load(a.pairs + q.x), P2 = scalar_load(a.pairs + q.y);
        wave_eri<LA, LB, LC, LD, T>(P1, P2, a.prims, a.primcut, a.rys2_exact, (T)1, sE);
        if constexpr (MODE == kDigestBlock) {
            for (int c = lane; c < NCOMP; c += 64) a.out[g * NCOMP + c] = (double)sE[c];
        } else {
            static_assert(NA * NB <= 64, "one diagonal component per lane");
            const int i = lane / NB, j = lane - i * NB;
            double m = lane < NA * NB ? fabs((double)sE[((i * NB + j) * NC + i) * ND + j]) : 0.0;
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) m = fmax(m, __shfl_xor(m, o, 64));
            if (lane == 0) a.out[q.x] = sqrt(m);
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// launchers of the explicit lists: dispatch on the class and mode
// ---------------------------------------------------------------------------
// blocks: a quartet per lane; per wave 8 quartets in turn, or one where only a bound is wanted (a list
// of pairs, not of quartets)
template <int LA, int LB, int LC, int LD>
static hipError_t launch_block(const EriArgs& a, hipStream_t st) {
    if (a.nquart <= 0) return hipSuccess;
    EriArgs b = a;
    constexpr bool lane = ClassInfo<LA, LB, LC, LD>::NCOMP <= kLaneMaxComp;
    b.qpb = lane ? 256 : 8;
    const unsigned nb = (unsigned)((a.nquart + b.qpb - 1) / b.qpb);
    if constexpr (lane) hipLaunchKernelGGL((k_eri_lane<LA, LB, LC, LD, double>), dim3(nb), dim3(256), 0, st, b);
    else hipLaunchKernelGGL((k_eri_wave<LA, LB, LC, LD, kDigestBlock, double>), dim3(nb), dim3(64), 0, st, b);
    return hipGetLastError();
}

template <int LA, int LB>
static hipError_t launch_schwarz(const EriArgs& a, hipStream_t st) {
    if (a.nquart <= 0) return hipSuccess;
    EriArgs b = a;
    b.qpb = 1;
    if constexpr (ClassInfo<LA, LB, LA, LB>::NCOMP <= kLaneMaxComp) {
        const unsigned nb = (unsigned)((a.nquart * kSchwarzLanes + 255) / 256);
        hipLaunchKernelGGL((k_schwarz<LA, LB>), dim3(nb), dim3(256), 0, st, b);
    } else {
        hipLaunchKernelGGL((k_eri_wave<LA, LB, LA, LB, kDigestSchwarz, double>), dim3((unsigned)a.nquart), dim3(64), 0, st, b);
    }
    return hipGetLastError();
}

hipError_t eri_launch(int mode, int cb, int ck, const EriArgs& a, hipStream_t st) {
    if (mode == kDigestBlock) {
#define UNO_Q(X, Y, LA, LB, LC, LD) \
    if (cb == X && ck == Y) return launch_block<LA, LB, LC, LD>(a, st);
        UNO_QUARTET_CLASSES(UNO_Q)
#undef UNO_Q
    }
    // Schwarz: diagonal classes only
    if (mode != kDigestSchwarz || cb != ck) return hipErrorInvalidValue;
    switch (cb) {
        case 0: return launch_schwarz<0, 0>(a, st);
        case 1: return launch_schwarz<1, 0>(a, st);
        case 2: return launch_schwarz<1, 1>(a, st);
        case 3: return launch_schwarz<2, 0>(a, st);
        case 4: return launch_schwarz<2, 1>(a, st);
        case 5: return launch_schwarz<2, 2>(a, st);
    }
    return hipErrorInvalidValue;
}

int eri_class_ncomp(int cb, int ck) {
    static const int nab[6] = {1, 3, 9, 6, 18, 36};
    return nab[cb] * nab[ck];
}

// ---------------------------------------------------------------------------
// Fock-build launches: the kernels are instantiated per (mode, precision) in fock_*.hip
// ---------------------------------------------------------------------------
hipError_t fock_launch_rhf64(int, int, const FockArgs&, int, size_t, hipStream_t);
hipError_t fock_launch_uhf64(int, int, const FockArgs&, int, size_t, hipStream_t);
hipError_t fock_launch_rhf32(int, int, const FockArgs&, int, size_t, hipStream_t);
hipError_t fock_launch_uhf32(int, int, const FockArgs&, int, size_t, hipStream_t);

bool fock_is_wave(int cb, int ck) { return eri_class_ncomp(cb, ck) > kLaneMaxComp; }

// LDS a block may take (rows, then the Rys table if it still fits): two blocks per compute unit,
// or nearly all of it for the classes whose registers leave one wave per SIMD, so one block per
// compute unit, anyway
static size_t row_lds_budget(int cb, int ck) {
    return (eri_class_ncomp(cb, ck) >= 54 || cb == 5 ? 156 : 80) * 1024;
}

// the LDS a block of this launch needs: dynamic part, and whether all of it fits the budget
static size_t fock_lds(int cb, int ck, const FockConfig& f, int mode, int ncols, int nsh, bool fp32, bool& fits) {
    static const int na[6] = {1, 3, 3, 6, 6, 6};          // functions of the first bra shell
    static const int nb[6] = {1, 1, 3, 1, 3, 6};          // and of the second
    static const int lsum[6] = {0, 1, 2, 2, 3, 4};
    const int nr = (lsum[cb] + lsum[ck]) / 2 + 1;
    const size_t tab = fp32 ? (size_t)kRysAsym[nr] * 2 * nr * UNO_RYS_NCOEF_F * sizeof(float)
                            : (size_t)kRysAsym[nr] * 2 * nr * UNO_RYS_NCOEF * sizeof(double);
    // beside it: the waves' ket queues and the reductions of the bra's Coulomb block
    const size_t sp = mode == kDigestUHF ? 2 : 1, reserve = 8 * (128 * sizeof(int) + na[cb] * nb[cb] * sizeof(double)) + 256;
    const size_t all = (size_t)(na[cb] + nb[cb]) * sp * ncols * sizeof(double);
    size_t dyn = f.mlds ? (size_t)nsh * sizeof(double) : 0;
    if (f.variant == 1 || f.variant == 2) dyn += all;
    if (f.variant == 3) dyn += (size_t)na[cb] * sp * ncols * sizeof(double);
    if (f.variant && f.dlds) dyn += all;
    const bool table = f.variant == 1 || (f.variant == 0 && nr <= kLdsTabMaxRoots);
    fits = dyn + (table ? tab : 0) + reserve <= row_lds_budget(cb, ck);
    return dyn;
}

bool fock_config_fits(int cb, int ck, const FockConfig& f, int mode, int ncols, int nsh, bool fp32) {
    bool fits = false;
    fock_lds(cb, ck, f, mode, ncols, nsh, fp32, fits);
    return fits;
}

FockConfig fock_default(int cb, int ck, int mode, int ncols, int nsh, bool fp32, bool rows, int force, int dens) {
    FockConfig f;
    if (fock_is_wave(cb, ck)) return f;
    auto ok = [&](const FockConfig& g) { return fock_config_fits(cb, ck, g, mode, ncols, nsh, fp32); };
    if (rows) {
        for (int v : {force, 1, 2, 3}) {
            if (v < 1 || v > 3) continue;
            f.variant = v;
            if (ok(f)) break;
            f.variant = 0;
        }
    }
    f.mlds = 1;
    if (!ok(f)) f.mlds = 0;
    // (the exchange density rows in LDS cost a class the blocks they displace: only (ss|ss), which
    // keeps its five blocks per compute unit with them, is faster, 3.63 -> 3.48 ms at 64 waters; of
    // the others (ds|ss) goes 4.56 -> 3.96 ms without, the whole build 56.0 -> 54.8, the FP32 build
    // of 37 waters 17.8 -> 16.7)
    if (f.variant && (dens > 0 || (dens < 0 && cb == 0))) {
        f.dlds = 1;
        if (!ok(f)) f.dlds = 0;
    }
    return f;
}

hipError_t fock_launch(int mode, bool fp32, int cb, int ck, FockArgs a, const FockConfig& f, int ncols, hipStream_t st) {
    if (a.ncand <= 0) return hipSuccess;
    // the rows merge in LDS with FP64 atomics: no deterministic form
    if (!a.sp || !a.blk || !a.ctr || !a.nquart || (f.variant && (a.fix_lo || !a.jp || ncols <= 0)) || f.variant < 0 || f.variant > 3)
        return hipErrorInvalidValue;
    bool fits = false;
    const size_t dyn = fock_lds(cb, ck, f, mode, ncols, a.nsh, fp32, fits);
    if (!fits && !fock_is_wave(cb, ck)) return hipErrorInvalidValue;
    a.mlds = f.mlds;
    a.dlds = f.dlds;
    if (mode == kDigestRHF) return fp32 ? fock_launch_rhf32(cb, ck, a, f.variant, dyn, st)
                                        : fock_launch_rhf64(cb, ck, a, f.variant, dyn, st);
    if (mode == kDigestUHF) return fp32 ? fock_launch_uhf32(cb, ck, a, f.variant, dyn, st)
                                        : fock_launch_uhf64(cb, ck, a, f.variant, dyn, st);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------
// around a Fock build
// ---------------------------------------------------------------------------
// every accumulator of a build cleared in one launch (one buffer per row of the grid)
__global__ __launch_bounds__(256) void k_clear(const ClearList c) {
    unsigned long long* p = c.p[blockIdx.y];
    const long long len = c.len[blockIdx.y];
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < len; i += (long long)gridDim.x * 256) p[i] = 0ULL;
}

hipError_t fock_clear(const ClearList& c, hipStream_t st) {
    long long most = 0;
    for (int k = 0; k < c.n; ++k) most = std::max(most, c.len[k]);
    if (most <= 0) return hipSuccess;
    const long long nb = std::min<long long>((most + 1023) / 1024, 2048);
    hipLaunchKernelGGL(k_clear, dim3((unsigned)nb, (unsigned)c.n), dim3(256), 0, st, c);
    return hipGetLastError();
}

// The tasks of every launch that hold a quartet of this build: a candidate segment counts when
// its first ket (the largest bound) is within the build and, in a mixed build, some of it lies
// on the launch's side of the FP32 threshold (fock_task's tests).  Half the candidates are
// above the diagonal or below the threshold in a full 64-water build and nearly all of them in
// an incremental one; as blocks of their own each cost a launch slot and a chain of
// scalar loads.
__global__ __launch_bounds__(kTaskThreads) void k_fock_tasks(int nsrc, const FockTaskSource* __restrict__ src,
                                                             const char* __restrict__ tables, const FockArgs a,
                                                             FockCounter* ctr, int* __restrict__ lists) {
    __shared__ int wtot[kTaskThreads / 64], base;
    int lo = 0, hi = nsrc - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (src[mid].block0 <= (int)blockIdx.x) lo = mid; else hi = mid - 1;
    }
    const FockTaskSource S = src[lo];
    const int c = ((int)blockIdx.x - S.block0) * kTaskThreads + (int)threadIdx.x;
    bool live = false;
    if (c < S.ncand) {
        const FockSpace* sp = reinterpret_cast<const FockSpace*>(tables + S.sp);
        const int* blk = reinterpret_cast<const int*>(tables + S.blk);
        int x = blk[c >> 6], y = blk[(c >> 6) + 1];
        while (x < y) {
            const int mid = (x + y + 1) >> 1;
            if (sp[mid].first <= c) x = mid; else y = mid - 1;
        }
        const FockSpace& s = sp[x];
        const int l = c - s.first, ibra = l / s.nseg, k0 = (l - ibra * s.nseg) * s.seg;
        int k1 = min(s.nket, k0 + s.seg);
        if (s.same) k1 = min(k1, ibra + 1);
        const int mol = a.mols ? s.mol : 0;
        if (k0 < k1 && !(a.mol_active && !a.mol_active[mol])) {
            const double qi = a.pairQ[s.bra_off + ibra], qd = qi * (4.0 * a.dmax[mol]);
            const double q0 = a.pairQ[s.ket_off + k0];
            live = qd > 0.0 && q0 >= a.tau / qd;
            if (live && a.fp32_thr > 0.0) {
                const double t32 = a.fp32_thr / qi;
                live = S.f32 ? a.pairQ[s.ket_off + k1 - 1] < t32 : q0 >= t32;
            }
        }
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned long long m = __ballot(live);
    if (lane == 0) wtot[wave] = __popcll(m);
    __syncthreads();
    if (threadIdx.x == 0) {
        int t = 0;
        for (int w = 0; w < kTaskThreads / 64; ++w) {
            const int v = wtot[w];
            wtot[w] = t;
            t += v;
        }
        base = t ? atomicAdd(&ctr[lo].count, t) : 0;
    }
    __syncthreads();
    if (live) lists[S.list + base + wtot[wave] + __popcll(m & ((1ull << lane) - 1))] = c;
}

hipError_t fock_tasks(int nsrc, const FockTaskSource* src, int nblocks, const char* tables, const FockArgs& a,
                      FockCounter* ctr, int* lists, hipStream_t st) {
    if (nsrc <= 0 || nblocks <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fock_tasks, dim3((unsigned)nblocks), dim3(kTaskThreads), 0, st, nsrc, src, tables, a, ctr, lists);
    return hipGetLastError();
}

// the molecule's slice of a batched store, or the store itself
__device__ __forceinline__ MolDesc mol_of(const MolDesc* mols, const int* pmol, int p, int n, int nsh) {
    return mols ? mols[pmol[p]] : MolDesc{0, 0, n, nsh};
}
// D0 in pair-major blocks (a wave of kets then reads its density blocks at consecutive
// addresses) and each pair's own shell-block maximum, for the kernels' screen
__global__ __launch_bounds__(256) void k_pair_density(int np, const int4* __restrict__ kidx, const int4* __restrict__ kjo,
                                                      const double* __restrict__ D0, const double* __restrict__ dsh,
                                                      int n, int nsh, const MolDesc* mols, const int* pmol,
                                                      double* __restrict__ dp, double* __restrict__ dpair) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int4 h = kidx[p], o = kjo[p];
    const MolDesc m = mol_of(mols, pmol, p, n, nsh);
    const double* D = D0 + m.moff + (long)h.x * m.n + h.y;
    for (int kl = 0; kl < o.z; ++kl) dp[o.x + (long)kl * o.y] = D[(long)(kl / o.w) * m.n + kl % o.w];
    dpair[p] = dsh[m.dshoff + (long)h.z * m.nsh + h.w];
}

hipError_t pair_density(int npairs, const int4* kidx, const int4* kjo, const double* D0, const double* dsh, int n,
                        int nsh, const MolDesc* mols, const int* pmol, double* dp, double* dpair, hipStream_t st) {
    if (npairs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_density, dim3((npairs + 255) / 256), dim3(256), 0, st, npairs, kidx, kjo, D0, dsh, n, nsh, mols,
                       pmol, dp, dpair);
    return hipGetLastError();
}

// pair-major Coulomb accumulator into W (pair blocks are disjoint: plain adds)
__global__ __launch_bounds__(256) void k_jp_scatter(int np, const int4* __restrict__ kidx, const int4* __restrict__ kjo,
                                                    const double* __restrict__ jp, double* W0, double* W1, int n,
                                                    const MolDesc* mols, const int* pmol) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    const int4 h = kidx[p], o = kjo[p];
    const MolDesc m = mol_of(mols, pmol, p, n, 0);
    for (int kl = 0; kl < o.z; ++kl) {
        const double v = jp[o.x + (long)kl * o.y];
        if (v == 0.0) continue;
        const long w = m.moff + (long)(h.x + kl / o.w) * m.n + h.y + kl % o.w;
        W0[w] += v;
        if (W1) W1[w] += v;
    }
}

hipError_t jp_scatter(int npairs, const int4* kidx, const int4* kjo, const double* jp, double* W0, double* W1, int n,
                      const MolDesc* mols, const int* pmol, hipStream_t st) {
    if (npairs <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_jp_scatter, dim3((npairs + 255) / 256), dim3(256), 0, st, npairs, kidx, kjo, jp, W0, W1, n, mols, pmol);
    return hipGetLastError();
}

// the Fock kernels' copies of the pair data, from the pair and primitive arrays: bra
// primitives with their share of the prefactor, the kets' fields one after another
__global__ __launch_bounds__(256) void k_pair_store(int np, int nrun, const PairRun* __restrict__ runs,
                                                    const PairHdr* __restrict__ pairs, const PrimPair* __restrict__ prims,
                                                    const int* __restrict__ colmap, BraPrim* __restrict__ bprim,
                                                    double* __restrict__ kprim, long long kps, double* __restrict__ kgeo,
                                                    int4* __restrict__ kidx, int4* __restrict__ kjo, int* __restrict__ knp,
                                                    int2* __restrict__ kcol) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= np) return;
    int lo = 0, hi = nrun - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (runs[mid].off <= p) lo = mid; else hi = mid - 1;
    }
    const PairRun r = runs[lo];
    const PairHdr h = pairs[p];
    for (int x = 0; x < 3; ++x) {
        kgeo[(long)x * np + p] = h.A[x];
        kgeo[(long)(3 + x) * np + p] = h.AB[x];
    }
    kidx[p] = make_int4(h.f1, h.f2, h.sh1, h.sh2);
    kjo[p] = make_int4((int)(r.jo0 + (p - r.off)), r.count, pair_comps(r.lcls), pair_comps2(r.lcls));
    knp[p] = 2 * h.nprim + (h.same ? 1 : 0);
    kcol[p] = make_int2(colmap[r.col0 + h.f1], colmap[r.col0 + h.f2]);
    for (int j = 0; j < h.nprim; ++j) {
        const PrimPair q = prims[h.prim0 + j];
        BraPrim b;
        b.p = q.p;
        b.ip = q.ip;
        b.K = kTwoPi25 * q.K * q.ip;
        b.s = kTwoPi25 * q.s * q.ip;
        for (int x = 0; x < 3; ++x) {
            b.P[x] = q.P[x];
            b.PA[x] = q.P[x] - h.A[x];
        }
        bprim[h.prim0 + j] = b;
        double* k = kprim + r.kp0 + (long)j * r.count + (p - r.off);
        k[0] = q.p;
        k[kps] = q.ip;
        k[2 * kps] = q.K * q.ip;
        k[3 * kps] = q.s * q.ip;
        for (int x = 0; x < 3; ++x) k[(4 + x) * kps] = q.P[x];
    }
}

hipError_t pair_store(int np, int nrun, const PairRun* runs, const PairHdr* pairs, const PrimPair* prims,
                      const int* colmap, BraPrim* bprim, double* kprim, long long kps, double* kgeo, int4* kidx, int4* kjo,
                      int* knp, int2* kcol, hipStream_t st) {
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_pair_store, dim3((np + 255) / 256), dim3(256), 0, st, np, nrun, runs, pairs, prims, colmap, bprim,
                       kprim, kps, kgeo, kidx, kjo, knp, kcol);
    return hipGetLastError();
}

// the pair and primitive arrays reordered on the device: new pair k is old pair order[k],
// its primitive records moved to prim0[k]
__global__ __launch_bounds__(256) void k_permute_pairs(int np, const int* __restrict__ order,
                                                       const int* __restrict__ prim0,
                                                       const PairHdr* __restrict__ oldp,
                                                       const PrimPair* __restrict__ oldq, PairHdr* __restrict__ newp,
                                                       PrimPair* __restrict__ newq) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= np) return;
    PairHdr h = oldp[order[k]];
    const int p0 = h.prim0;
    h.prim0 = prim0[k];
    newp[k] = h;
    for (int q = 0; q < h.nprim; ++q) newq[h.prim0 + q] = oldq[p0 + q];
}

hipError_t permute_pairs(int np, const int* order, const int* prim0, const PairHdr* oldp, const PrimPair* oldq,
                         PairHdr* newp, PrimPair* newq, hipStream_t st) {
    if (np <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_permute_pairs, dim3((unsigned)((np + 255) / 256)), dim3(256), 0, st, np, order, prim0,
                       oldp, oldq, newp, newq);
    return hipGetLastError();
}

// fixed-point W (two int64 words per entry, fix_lo entries apart) to FP64, in place
__global__ __launch_bounds__(256) void k_fixed_to_f64(long long nn, double* W, long long lo_off) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nn) return;
    const long long* w = reinterpret_cast<const long long*>(W);
    const long long hi = w[i], lo = w[i + lo_off];
    W[i] = (double)hi * (1.0 / kFixHiScale) + (double)lo * (1.0 / kFixLoScale);
}

hipError_t fixed_to_f64(long long nn, double* W, long long lo_off, hipStream_t st) {
    if (nn <= 0) return hipSuccess;
    if (lo_off < nn) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_fixed_to_f64, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, nn, W, lo_off);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Rys-table evaluation for the parity tests
// ---------------------------------------------------------------------------
template <int NR, typename T>
__global__ void k_rys_eval(int npts, const double* x, double* u, double* w, int ref2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npts) return;
    T uu[NR], ww[NR];
    rys_roots<NR, T>((T)x[i], uu, ww, rys_table_of<NR, T>(!ref2));
    for (int r = 0; r < NR; ++r) { u[i * NR + r] = (double)uu[r]; w[i * NR + r] = (double)ww[r]; }
}

template <typename T>
static hipError_t rys_eval_t(int n, int npts, const double* x, double* u, double* w, hipStream_t st, int ref2) {
    const dim3 g((npts + 255) / 256), b(256);
    switch (n) {
        case 1: hipLaunchKernelGGL((k_rys_eval<1, T>), g, b, 0, st, npts, x, u, w, ref2); break;
        case 2: hipLaunchKernelGGL((k_rys_eval<2, T>), g, b, 0, st, npts, x, u, w, ref2); break;
        case 3: hipLaunchKernelGGL((k_rys_eval<3, T>), g, b, 0, st, npts, x, u, w, ref2); break;
        case 4: hipLaunchKernelGGL((k_rys_eval<4, T>), g, b, 0, st, npts, x, u, w, ref2); break;
        case 5: hipLaunchKernelGGL((k_rys_eval<5, T>), g, b, 0, st, npts, x, u, w, ref2); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t rys_eval_launch(int n, int npts, const double* x, double* u, double* w, hipStream_t st, bool fp32,
                           bool ref2) {
    return fp32 ? rys_eval_t<float>(n, npts, x, u, w, st, ref2) : rys_eval_t<double>(n, npts, x, u, w, st, ref2);
}

}  // namespace uno
