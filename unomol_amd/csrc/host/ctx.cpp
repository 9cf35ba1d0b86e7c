// Context build (shell pairs, primitive pairs, Schwarz bounds, quartet spaces) and
// the direct Fock build.  Replaces the reference's store-then-replay design
// (TwoElectronInts.cpp:511-697 computes every unique ERI once into an 8 GiB buffer
// spilling to MINTS.DAT; formGmatrix replays it each iteration, :822-869) with a direct
// build: every iteration recomputes the significant shell quartets on the GPU and
// contracts them with the density on the fly.
#include <algorithm>
#include <chrono>
#include <cstdint>
#include <cstring>
#include <cmath>
#include <numeric>
#include "engine.hpp"
#include "../hip/kernels.hpp"

namespace uno {

static thread_local std::string g_err;
void set_error(const std::string& m) { g_err = m; }
const std::string& get_error() { return g_err; }

static constexpr double kTwoPi25 = 34.986836655249725;

static int ensure_device() {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) {
        set_error("no HIP device is visible (the engine needs a gfx950 GPU)");
        return UNO_EDEVICE;
    }
    return UNO_OK;
}

EriArgs base_args(uno_ctx* c) {
    EriArgs a{};
    a.pairs = c->d_pairs.p;
    a.prims = c->d_prims.p;
    a.primcut = c->primcut;
    a.rys2_exact = c->rys2_exact;
    return a;
}

// order: the pairs by run key ascending, then bound descending, ties in their own order: a radix sort of
// the bounds' bits (positive numbers order like their bits), 11 at a time, and a last pass by
// run key.  On one thread: a parallel region that finds its threads asleep costs milliseconds (a
// parallel merge sort: 19 ms in a new program's context of 16 waters, 0.6 warm).  The stage around it,
// 32 waters: 1.05 ms, with one stable sort of the indices through the two arrays 2.1.
static void sort_runs(const std::vector<int>& runkey, const std::vector<double>& q, std::vector<int>& order) {
    struct Rec {
        std::uint64_t key;
        int pair;
    };
    const int np = (int)runkey.size();
    constexpr int kBits = 11, kDigits = 1 << kBits;
    static_assert(kNumPairClasses * kNumBuckets <= kDigits, "run keys are one digit");
    std::vector<Rec> v(np), w(np);
    for (int p = 0; p < np; ++p) {
        std::uint64_t b;
        std::memcpy(&b, &q[p], sizeof b);
        v[p] = Rec{~b, p};
    }
    std::vector<int> at(kDigits + 1);
    auto pass = [&](auto digit) {
        std::fill(at.begin(), at.end(), 0);
        for (const Rec& r : v) ++at[digit(r) + 1];
        if (np && at[digit(v[0]) + 1] == np) return;   // all alike
        for (int k = 0; k < kDigits; ++k) at[k + 1] += at[k];
        for (const Rec& r : v) w[at[digit(r)]++] = r;
        v.swap(w);
    };
    for (int s = 0; s < 64; s += kBits) pass([s](const Rec& r) { return (int)(r.key >> s & (kDigits - 1)); });
    pass([&](const Rec& r) { return runkey[r.pair]; });
    for (int p = 0; p < np; ++p) order[p] = v[p].pair;
}

int ctx_build(uno_ctx* c, const uno_basis* b, int start_shell) {
    using bclk = std::chrono::steady_clock;
    auto since = [](bclk::time_point t) { return std::chrono::duration<double, std::milli>(bclk::now() - t).count(); };
    const auto b0 = bclk::now();
    if (int rc = ensure_device()) return rc;
    std::string err;
    if (!make_basis(b, c->B, err)) {
        set_error(err);
        return UNO_EINVAL;
    }
    if (c->B.maxl > kMaxL) {
        set_error("the device ERI kernels cover s, p and d shells (l <= 2); this basis has l = " +
                  std::to_string(c->B.maxl));
        return UNO_EINVAL;
    }
    const Basis& B = c->B;
    c->n = B.norb;
    c->nsh = (int)B.sh.size();
    c->start_shell = start_shell;
    if (!c->st) UNO_HIP(hipStreamCreate(&c->st));
    hipStream_t st = c->st;
    const int nsh = c->nsh;
    // smallest exponent sum a ket pair can have: bounds the bare prefactor from above
    double amin = 1e300;
    for (const Shell& s : B.sh)
        for (double a : s.a) amin = std::min(amin, a);
    const double qmin = 2.0 * amin;
    std::vector<double> low(nsh);   // a shell's most diffuse exponent
    for (int a = 0; a < nsh; ++a) low[a] = *std::min_element(B.sh[a].a.begin(), B.sh[a].a.end());
    c->pairs.clear();
    c->prims.clear();
    c->pair_of.assign((size_t)nsh * nsh, -1);
    // shell pairs (a, b <= a), built per first shell a in parallel into lists of their own,
    // then laid out in the serial order (a, then b, ascending) at prefix-sum offsets
    std::vector<std::vector<PairHdr>> hpa(nsh);
    std::vector<std::vector<PrimPair>> ppa(nsh);
    std::vector<std::vector<int>> bpa(nsh);
#pragma omp parallel for schedule(dynamic, 4)
    for (int a = 0; a < nsh; ++a) {
        std::vector<PairHdr>& hv = hpa[a];
        std::vector<PrimPair>& pv = ppa[a];
        for (int bsh = 0; bsh <= a; ++bsh) {
            const int s1 = (B.sh[a].l >= B.sh[bsh].l) ? a : bsh;
            const int s2 = (s1 == a) ? bsh : a;
            const Shell& S1 = B.sh[s1];
            const Shell& S2 = B.sh[s2];
            const double* A = &B.xyz[3 * S1.cen];
            const double* Bc = &B.xyz[3 * S2.cen];
            PairHdr h{};
            double ab2 = 0.0;
            for (int x = 0; x < 3; ++x) {
                h.A[x] = A[x];
                h.AB[x] = A[x] - Bc[x];
                ab2 += h.AB[x] * h.AB[x];
            }
            // no primitive pair of distant shells passes the bound below where the largest overlap
            // and the smallest exponent sum together do not (1e-6 for the roundings)
            const double plow = low[a] + low[bsh];
            if (kTwoPi25 * std::exp(-low[a] * low[bsh] / plow * ab2) / (plow * qmin * std::sqrt(plow + qmin)) <
                c->primcut * (1.0 - 1e-6))
                continue;
            h.f1 = B.off[s1];
            h.f2 = B.off[s2];
            h.prim0 = (int)pv.size();   // within this shell's list; made global below
            h.same = (a == bsh);
            h.sh1 = s1;
            h.sh2 = s2;
            for (int i = 0; i < S1.npr; ++i) {
                // same shell: lower triangle of primitive pairs, off-diagonal doubled
                // (TwoElectronInts.cpp:444-449)
                const int jend = h.same ? i + 1 : S2.npr;
                for (int j = 0; j < jend; ++j) {
                    const double al = S1.a[i], be = S2.a[j], p = al + be, ip = 1.0 / p;
                    const double s = std::exp(-al * be * ip * ab2);
                    // every quartet with this primitive pair has a bare prefactor below
                    // this bound; drop it when the reference cut would reject them all
                    const double bound = kTwoPi25 * s * ip / (qmin * std::sqrt(p + qmin));
                    if (bound < c->primcut) continue;
                    PrimPair pp{};
                    pp.p = p;
                    pp.ip = ip;
                    for (int x = 0; x < 3; ++x) pp.P[x] = (al * A[x] + be * Bc[x]) * ip;
                    pp.K = S1.c[i] * S2.c[j] * ((h.same && i != j) ? 2.0 : 1.0) * s;
                    pp.s = s;
                    pv.push_back(pp);
                }
            }
            h.nprim = (int)pv.size() - h.prim0;
            if (h.nprim == 0) continue;
            hv.push_back(h);
            bpa[a].push_back(bsh);
        }
    }
    {
        std::vector<long long> hoff(nsh + 1, 0), poff(nsh + 1, 0);
        for (int a = 0; a < nsh; ++a) {
            hoff[a + 1] = hoff[a] + (long long)hpa[a].size();
            poff[a + 1] = poff[a] + (long long)ppa[a].size();
        }
        if (poff[nsh] > (long long)INT32_MAX) {
            set_error("too many primitive pairs for 32-bit offsets");
            return UNO_EINVAL;
        }
        c->pairs.resize((size_t)hoff[nsh]);
        c->prims.resize((size_t)poff[nsh]);
#pragma omp parallel for schedule(dynamic, 4)
        for (int a = 0; a < nsh; ++a) {
            for (size_t k = 0; k < hpa[a].size(); ++k) {
                PairHdr h = hpa[a][k];
                h.prim0 += (int)poff[a];
                c->pairs[(size_t)hoff[a] + k] = h;
                c->pair_of[(size_t)a * nsh + bpa[a][k]] = (int)(hoff[a] + (long long)k);
            }
            std::copy(ppa[a].begin(), ppa[a].end(), c->prims.begin() + poff[a]);
        }
    }
    const int np = (int)c->pairs.size();
    UNO_HIP(c->d_pairs.upload(c->pairs.data(), np, st));
    UNO_HIP(c->d_prims.upload(c->prims.data(), c->prims.size(), st));
    c->ctx_ms[0] = since(b0);
    const auto b1 = bclk::now();
    // Schwarz bounds Q_ab = sqrt(max |(ij|ij)|) from diagonal quartets, per pair class
    c->pairQ.assign(np, 0.0);
    DBuf<double> dq;
    UNO_HIP(dq.alloc(np));
    std::vector<int> pcls(np);
    for (int p = 0; p < np; ++p) pcls[p] = pair_class(B.sh[c->pairs[p].sh1].l, B.sh[c->pairs[p].sh2].l);
    // the pairs class by class, one list and one launch per class
    std::vector<int2> ql((size_t)np);
    int q0[kNumPairClasses + 1] = {};
    for (int p = 0; p < np; ++p) ++q0[pcls[p] + 1];
    for (int X = 0; X < kNumPairClasses; ++X) q0[X + 1] += q0[X];
    {
        int at[kNumPairClasses];
        std::copy(q0, q0 + kNumPairClasses, at);
        for (int p = 0; p < np; ++p) ql[(size_t)at[pcls[p]]++] = make_int2(p, p);
    }
    DBuf<int2> dql;
    UNO_HIP(dql.upload(ql.data(), ql.size(), st));
    for (int X = 0; X < kNumPairClasses; ++X) {
        EriArgs a = base_args(c);
        a.explicit_q = dql.p + q0[X];
        a.nquart = q0[X + 1] - q0[X];
        a.out = dq.p;
        // bounds from the uncut integrals: with the primitive cut a pair of distant
        // tight primitives can lose its whole diagonal quartet while its quartets with
        // diffuse partners survive the cut, so a cut diagonal would under-bound them
        a.primcut = 0.0;
        UNO_HIP(eri_launch(kDigestSchwarz, X, X, a, st));
    }
    UNO_HIP(hipMemcpyAsync(c->pairQ.data(), dq.p, np * sizeof(double), hipMemcpyDeviceToHost, st));
    UNO_HIP(hipStreamSynchronize(st));
    // Reorder the pair and primitive arrays into runs of (angular class, primitive-count
    // bucket), each sorted by Schwarz bound: a launch then walks contiguous memory, and the
    // lanes of a wave see alike primitive loops.
    c->ctx_ms[1] = since(b1);
    const auto b2 = bclk::now();
    // run key of every pair, taken before the arrays are permuted
    std::vector<int> runkey(np);
    for (int p = 0; p < np; ++p) runkey[p] = pcls[p] * kNumBuckets + prim_bucket(c->pairs[p].nprim);
    std::vector<int> order(np);
    sort_runs(runkey, c->pairQ, order);
    // new primitive offsets, in run order
    std::vector<int> nprim0(np);
    for (int k = 0, tp = 0; k < np; ++k) {
        nprim0[k] = tp;
        tp += c->pairs[order[k]].nprim;
    }
    std::vector<PairHdr> pairs2(np);
    std::vector<PrimPair> prims2(c->prims.size());
    std::vector<double> q2(np);
    std::vector<int> newidx(np);
    // all threads from 32768 pairs on; below, one is done before the others wake.  The stage on one
    // thread and on all, ms: 22849 pairs 0.8 and 1.4 when contexts follow each other, 1.6-1.9 and 1.5 for
    // one after a pause; 31839 pairs 1.1 and 1.8, 2.3-3.4 and 2.1; 52064 pairs 2.9-3.5 and 2.8-3.1, 4.7
    // and 3.4
#pragma omp parallel for schedule(static) if (np >= 32768)
    for (int k = 0; k < np; ++k) {
        PairHdr h = c->pairs[order[k]];
        const int p0 = h.prim0;
        h.prim0 = nprim0[k];
        std::copy(c->prims.begin() + p0, c->prims.begin() + p0 + h.nprim, prims2.begin() + h.prim0);
        pairs2[k] = h;
        q2[k] = c->pairQ[order[k]];
        newidx[order[k]] = k;
    }
    for (int& p : c->pair_of)
        if (p >= 0) p = newidx[p];
    c->pairs.swap(pairs2);
    c->prims.swap(prims2);
    c->pairQ.swap(q2);
    // the device copies: the same permutation applied to the arrays uploaded above (the
    // two index arrays go up instead of the records themselves)
    {
        DBuf<int> dorder, dp0;
        DBuf<PairHdr> np_d;
        DBuf<PrimPair> nq_d;
        UNO_HIP(dorder.upload(order.data(), np, st));
        UNO_HIP(dp0.upload(nprim0.data(), np, st));
        UNO_HIP(np_d.alloc(np));
        UNO_HIP(nq_d.alloc(c->prims.size()));
        UNO_HIP(permute_pairs(np, dorder.p, dp0.p, c->d_pairs.p, c->d_prims.p, np_d.p, nq_d.p, st));
        UNO_HIP(hipStreamSynchronize(st));
        c->d_pairs = std::move(np_d);
        c->d_prims = std::move(nq_d);
    }
    UNO_HIP(c->d_pairQ.upload(c->pairQ.data(), np, st));
    c->cls.clear();
    for (int k = 0; k < np;) {
        const int r = runkey[order[k]];
        PairClassList L;
        L.lcls = r / kNumBuckets;
        L.bucket = r % kNumBuckets;
        L.off = k;
        while (k < np && runkey[order[k]] == r) L.Q.push_back(c->pairQ[k++]);
        L.count = k - L.off;
        c->cls.push_back(std::move(L));
    }
    // one run per (angular class, bucket) at most, each sorted by bound
    if ((int)c->cls.size() > kNumPairClasses * kNumBuckets) {
        set_error("internal error: pair runs are not grouped (" + std::to_string(c->cls.size()) + " runs)");
        return UNO_EINVAL;
    }
    for (const PairClassList& L : c->cls)
        for (size_t i = 1; i < L.Q.size(); ++i)
            if (L.Q[i] > L.Q[i - 1]) {
                set_error("internal error: pair run is not sorted by Schwarz bound");
                return UNO_EINVAL;
            }
    c->ctx_ms[2] = since(b2);
    const auto b3 = bclk::now();
    {
        FockMol m;
        m.n = c->n;
        m.runs = &c->cls;
        m.pairs = c->pairs.data();
        if (int rc = c->fs.build({m}, c->d_pairs.p, c->d_prims.p, np, (long long)c->prims.size(), st)) return rc;
    }
    recall_tuning(c);
    std::vector<int> shoff(nsh), shn(nsh);
    for (int s = 0; s < nsh; ++s) {
        shoff[s] = B.off[s];
        shn[s] = ncart(B.sh[s].l);
    }
    UNO_HIP(c->d_shoff.upload(shoff.data(), nsh, st));
    UNO_HIP(c->d_shn.upload(shn.data(), nsh, st));
    // one-electron data: shells with their normalised primitives, centres, and the shell
    // pairs of each class with the higher-l shell first
    {
        std::vector<OneIntShell> hs(nsh);
        std::vector<double> al, co;
        for (int s = 0; s < nsh; ++s) {
            hs[s] = OneIntShell{B.sh[s].l, B.sh[s].npr, B.sh[s].cen, (int)al.size(), B.off[s]};
            al.insert(al.end(), B.sh[s].a.begin(), B.sh[s].a.end());
            co.insert(co.end(), B.sh[s].c.begin(), B.sh[s].c.end());
        }
        std::vector<std::vector<int2>> pl(kNumPairClasses);
        for (int a = 0; a < nsh; ++a)
            for (int bs = 0; bs <= a; ++bs) {
                const int s1 = B.sh[a].l >= B.sh[bs].l ? a : bs, s2 = s1 == a ? bs : a;
                pl[pair_class(B.sh[s1].l, B.sh[s2].l)].push_back(int2{s1, s2});
            }
        UNO_HIP(c->oi_shells.upload(hs.data(), hs.size(), st));
        UNO_HIP(c->oi_alpha.upload(al.data(), al.size(), st));
        UNO_HIP(c->oi_coef.upload(co.data(), co.size(), st));
        UNO_HIP(c->oi_xyz.upload(B.xyz.data(), B.xyz.size(), st));
        UNO_HIP(c->oi_charge.upload(B.q.data(), B.q.size(), st));
        for (int k = 0; k < kNumPairClasses; ++k) {
            c->oi_npair[k] = (int)pl[k].size();
            // longest primitive loops first (a counting sort): a wave's pairs are alike, and the
            // long ones start early
            auto nprim = [&](const int2& p) { return B.sh[p.x].npr * B.sh[p.y].npr; };
            std::vector<int> at;
            for (const int2& p : pl[k]) {
                if ((int)at.size() < nprim(p) + 2) at.resize(nprim(p) + 2);
                ++at[nprim(p)];
            }
            for (int q = (int)at.size() - 2; q >= 0; --q) at[q] += at[q + 1];   // pairs of at least q
            c->oi_many[k] = (int)at.size() > kOiMany ? at[kOiMany] : 0;
            std::vector<int2> sorted(pl[k].size());
            for (const int2& p : pl[k]) sorted[at[nprim(p) + 1]++] = p;
            pl[k].swap(sorted);
            UNO_HIP(c->oi_pairs[k].upload(pl[k].data(), pl[k].size(), st));
        }
    }
    const size_t nn = (size_t)c->n * c->n;
    UNO_HIP(c->D0.alloc(nn));
    UNO_HIP(c->D1.alloc(nn));
    UNO_HIP(c->D2.alloc(nn));
    UNO_HIP(c->W0.alloc(nn));
    UNO_HIP(c->W1.alloc(nn));
    UNO_HIP(c->Dsh.alloc((size_t)nsh * nsh));
    UNO_HIP(c->pk.alloc((size_t)c->n * (c->n + 1)));
    UNO_HIP(c->scal.alloc(16));
    UNO_HIP(c->red.alloc(kRedBlocks));
    UNO_HIP(hipStreamSynchronize(st));
    c->ctx_ms[3] = since(b3);
    return UNO_OK;
}

int oneint_device(uno_ctx* c, double* S, double* T, double* H) {
    OneIntArgs a{};
    a.shells = c->oi_shells.p;
    a.alpha = c->oi_alpha.p;
    a.coef = c->oi_coef.p;
    a.xyz = c->oi_xyz.p;
    a.charge = c->oi_charge.p;
    a.ncen = c->B.ncen;
    a.n = c->n;
    a.skip = c->skip_center;
    a.S = S;
    a.T = T;
    a.H = H;
    static const int kl[kNumPairClasses][2] = {{0, 0}, {1, 0}, {1, 1}, {2, 0}, {2, 1}, {2, 2}};
    for (int k = 0; k < kNumPairClasses; ++k)
        UNO_HIP(oneint_launch(kl[k][0], kl[k][1], c->oi_npair[k], c->oi_many[k], c->oi_pairs[k].p, a, c->st));
    return UNO_OK;
}

// Positron model potential (GDPMInts.cpp:6-146): the positron's charge as six s Gaussians
// c_k exp(-a_k |r - R|^2) at R; every shell pair's (ab|g_k) from the FP64 ERI kernels in
// block mode with the Gaussians as a six-primitive ket pair, no primitive cut (the
// reference applies none there).  The expansion is the reference's fitted table.
int gdpm_matrix(uno_ctx* c, const double* R, std::vector<double>& dh) {
    static const double kAlf[6] = {6.8505018000, 4.0491646000, 3.5941062989, 1.2478274000, 0.7927690989, 0.3377107978};
    static const double kCof[6] = {0.0766926784, 0.1483475912, 0.0462334641, 0.0717376427, 0.0447149792, 0.0069678529};
    const int n = c->n;
    dh.assign((size_t)n * (n + 1) / 2, 0.0);
    std::vector<PairHdr> pairs(c->pairs);
    std::vector<PrimPair> prims(c->prims);
    PairHdr g{};
    for (int x = 0; x < 3; ++x) g.A[x] = R[x];
    g.prim0 = (int)prims.size();
    g.nprim = 6;
    g.sh1 = g.sh2 = -1;
    const int gi = (int)pairs.size();
    pairs.push_back(g);
    for (int k = 0; k < 6; ++k) {
        PrimPair q{};
        q.p = kAlf[k];
        q.ip = 1.0 / kAlf[k];
        for (int x = 0; x < 3; ++x) q.P[x] = R[x];
        q.K = kCof[k];
        q.s = 1.0;
        prims.push_back(q);
    }
    hipStream_t st = c->st;
    DBuf<PairHdr> dp;
    DBuf<PrimPair> dpr;
    UNO_HIP(dp.upload(pairs.data(), pairs.size(), st));
    UNO_HIP(dpr.upload(prims.data(), prims.size(), st));
    std::vector<std::vector<int2>> lists(kNumPairClasses);
    for (int p = 0; p < gi; ++p) {
        const PairHdr& h = c->pairs[p];
        lists[pair_class(c->B.sh[h.sh1].l, c->B.sh[h.sh2].l)].push_back(make_int2(p, gi));
    }
    for (int X = 0; X < kNumPairClasses; ++X) {
        if (lists[X].empty()) continue;
        const int nc = eri_class_ncomp(X, 0);
        DBuf<int2> dq;
        DBuf<double> dout;
        UNO_HIP(dq.upload(lists[X].data(), lists[X].size(), st));
        UNO_HIP(dout.alloc(lists[X].size() * (size_t)nc));
        EriArgs a = base_args(c);
        a.pairs = dp.p;
        a.prims = dpr.p;
        a.primcut = 0.0;
        a.explicit_q = dq.p;
        a.nquart = (long long)lists[X].size();
        a.out = dout.p;
        UNO_HIP(eri_launch(kDigestBlock, X, 0, a, st));
        std::vector<double> blk(lists[X].size() * (size_t)nc);
        UNO_HIP(hipMemcpyAsync(blk.data(), dout.p, blk.size() * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        for (size_t q = 0; q < lists[X].size(); ++q) {
            const PairHdr& h = c->pairs[lists[X][q].x];
            const int na = ncart(c->B.sh[h.sh1].l), nb = ncart(c->B.sh[h.sh2].l);
            for (int i = 0; i < na; ++i)
                for (int j = 0; j < nb; ++j) {
                    const int r = h.f1 + i, col = h.f2 + j;
                    if (h.sh1 == h.sh2 && col > r) continue;   // same shell: each element once
                    dh[pidx(r, col)] -= blk[q * nc + i * nb + j];
                }
        }
    }
    return UNO_OK;
}

// Every canonical function quartet in the reference's order, evaluated on the device
// shell-quartet blocks.
int eri_emit(uno_ctx* c, long cap, double* val, int* ijkl, long* count) {
    const Basis& B = c->B;
    const int nsh = c->nsh;
    struct Rec {
        int cls;        // index into groups
        long q;         // quartet within the group
        int comp;       // component index within the block
    };
    std::vector<Rec> recs;
    std::vector<int> fq;   // 4 per record
    std::vector<std::vector<int2>> groups(kNumPairClasses * kNumPairClasses);
    long n = 0;
    for (int ish = c->start_shell; ish < nsh; ++ish)
        for (int jsh = 0; jsh <= ish; ++jsh)
            for (int ksh = 0; ksh <= ish; ++ksh)
                for (int lsh = 0; lsh <= ksh; ++lsh) {
                    const int sh[4] = {ish, jsh, ksh, lsh};
                    int nf[4], o[4];
                    for (int x = 0; x < 4; ++x) {
                        nf[x] = ncart(B.sh[sh[x]].l);
                        o[x] = B.off[sh[x]];
                    }
                    const int p1 = c->pair_of[(size_t)ish * nsh + jsh];
                    const int p2 = c->pair_of[(size_t)ksh * nsh + lsh];
                    long qidx = -1;
                    int gidx = -1;
                    bool swap = false;
                    int NBb = 0, NCb = 0, NDb = 0;
                    for (int a = 0; a < nf[0]; ++a) {
                        const int ir = o[0] + a;
                        for (int b = 0; b < nf[1]; ++b) {
                            const int jr = o[1] + b;
                            if (jr > ir) break;
                            for (int cc = 0; cc < nf[2]; ++cc) {
                                const int kr = o[2] + cc;
                                if (kr > ir) break;
                                for (int d = 0; d < nf[3]; ++d) {
                                    const int lr = o[3] + d;
                                    if (lr > kr || (ir == kr && lr > jr)) break;
                                    Rec r{-1, -1, 0};
                                    if (p1 >= 0 && p2 >= 0) {
                                        if (qidx < 0) {
                                            const PairHdr& h1 = c->pairs[p1];
                                            const PairHdr& h2 = c->pairs[p2];
                                            const int X = pair_class(B.sh[h1.sh1].l, B.sh[h1.sh2].l);
                                            const int Y = pair_class(B.sh[h2.sh1].l, B.sh[h2.sh2].l);
                                            swap = X < Y;
                                            const int gb = swap ? Y : X, gk = swap ? X : Y;
                                            gidx = gb * kNumPairClasses + gk;
                                            const PairHdr& hb = swap ? h2 : h1;
                                            const PairHdr& hk = swap ? h1 : h2;
                                            NBb = ncart(B.sh[hb.sh2].l);
                                            NCb = ncart(B.sh[hk.sh1].l);
                                            NDb = ncart(B.sh[hk.sh2].l);
                                            groups[gidx].push_back(swap ? make_int2(p2, p1) : make_int2(p1, p2));
                                            qidx = (long)groups[gidx].size() - 1;
                                        }
                                        const PairHdr& h1 = c->pairs[p1];
                                        const PairHdr& h2 = c->pairs[p2];
                                        // component indices in each pair's stored orientation
                                        const int i1 = (h1.sh1 == ish) ? a : b, i2 = (h1.sh1 == ish) ? b : a;
                                        const int k1 = (h2.sh1 == ksh) ? cc : d, k2 = (h2.sh1 == ksh) ? d : cc;
                                        int comp;
                                        if (!swap) comp = ((i1 * NBb + i2) * NCb + k1) * NDb + k2;
                                        else comp = ((k1 * NBb + k2) * NCb + i1) * NDb + i2;
                                        r = Rec{gidx, qidx, comp};
                                    }
                                    recs.push_back(r);
                                    fq.push_back(ir); fq.push_back(jr); fq.push_back(kr); fq.push_back(lr);
                                    ++n;
                                }
                            }
                        }
                    }
                }
    *count = n;
    if (cap <= 0) return UNO_OK;
    hipStream_t st = c->st;
    std::vector<std::vector<double>> blocks(groups.size());
    for (int g = 0; g < (int)groups.size(); ++g) {
        if (groups[g].empty()) continue;
        const int X = g / kNumPairClasses, Y = g % kNumPairClasses;
        const int nc = eri_class_ncomp(X, Y);
        DBuf<int2> dq;
        DBuf<double> dout;
        UNO_HIP(dq.upload(groups[g].data(), groups[g].size(), st));
        UNO_HIP(dout.alloc(groups[g].size() * (size_t)nc));
        EriArgs a = base_args(c);
        a.explicit_q = dq.p;
        a.nquart = (long long)groups[g].size();
        a.out = dout.p;
        UNO_HIP(eri_launch(kDigestBlock, X, Y, a, st));
        blocks[g].resize(groups[g].size() * (size_t)nc);
        UNO_HIP(hipMemcpyAsync(blocks[g].data(), dout.p, blocks[g].size() * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
    }
    for (long e = 0; e < n && e < cap; ++e) {
        const Rec& r = recs[e];
        double v = 0.0;
        if (r.cls >= 0) {
            const int X = r.cls / kNumPairClasses, Y = r.cls % kNumPairClasses;
            v = blocks[r.cls][(size_t)r.q * eri_class_ncomp(X, Y) + r.comp];
        }
        val[e] = v;
        for (int x = 0; x < 4; ++x) ijkl[4 * e + x] = fq[4 * e + x];
    }
    return UNO_OK;
}

}  // namespace uno
