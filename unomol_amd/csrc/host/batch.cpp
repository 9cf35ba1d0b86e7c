// Batched SCF: many molecules of uneven size (each N <= 256 functions), RHF and UHF mixed,
// iterated in lockstep on one device (no reference counterpart: the reference runs one
// molecule per process).
//
// Every molecule keeps its own context for the pair data (shell pairs, Schwarz bounds,
// runs sorted by bound); their pair and primitive arrays are concatenated into one device
// array.  A Fock build is one launch per (bra class, ket class, RHF/UHF) over all molecules'
// quartet spaces (FockStore), each of which names its molecule's slice of the density and
// accumulator stores.
// Dense steps run as grouped GEMMs over every (molecule, spin) slot and a batched Jacobi
// eigensolver (one block per matrix).  The iteration is the single-molecule one with Pulay
// DIIS (8 vectors, error X^T(FPS - SPF)X); molecules stop updating once converged.
#include <algorithm>
#include <chrono>
#include <cfloat>
#include <cmath>
#include <cstdio>
#include <cstring>
#include "engine.hpp"
#include "../hip/batch_kernels.hpp"
#include "../hip/kernels.hpp"

using namespace uno;

namespace {

struct BatchMol {
    uno_ctx* ctx = nullptr;
    int nelec = 0, n = 0, nsh = 0, nocc[2] = {0, 0};
    bool uhf = false;
    long long moff = 0, dshoff = 0;
    int shoff = 0, pair_off = 0;
    // state
    bool active = true, converged = false;
    int iterations = 0;
    double energy = 0.0, eold = 0.0, ediff = 0.0, pdiff = 0.0, nuc = 0.0, init_energy = 0.0;
};

constexpr int kBatchDiis = 8;

using clk = std::chrono::steady_clock;
double secs(clk::time_point a, clk::time_point b) { return std::chrono::duration<double>(b - a).count(); }


// Device copies of the small per-iteration arrays (GEMM groups and tiles, matrix lists,
// quartet entries, DIIS coefficients): the k-th upload of an iteration reuses slot k,
// grown when needed, so the steady state allocates nothing.  Every iteration ends with a
// stream synchronisation before reset() hands the slots out again.
struct Scratch {
    std::vector<DBuf<char>> slot;
    size_t next = 0;
    void reset() { next = 0; }
    template <class T>
    hipError_t upload(const T* h, size_t n, hipStream_t st, T** out) {
        if (next == slot.size()) slot.emplace_back();
        DBuf<char>& s = slot[next++];
        hipError_t e = s.alloc(std::max<size_t>(n, 1) * sizeof(T));
        if (e != hipSuccess) return e;
        *out = reinterpret_cast<T*>(s.p);
        return n ? hipMemcpyAsync(s.p, h, n * sizeof(T), hipMemcpyHostToDevice, st) : hipSuccess;
    }
};

}  // namespace

struct uno_batch {
    std::vector<BatchMol> mol;
    hipStream_t st = nullptr;
    long long store = 0, dsh_total = 0;
    DBuf<PairHdr> pairs;
    DBuf<PrimPair> prims;
    DBuf<double> pairQ;
    DBuf<int> sh_off, sh_n;
    DBuf<MolDesc> mdesc;
    DBuf<int> mshoff;           // per molecule: its first shell in the shell tables
    // stores (each sum_m N_m^2 doubles); index 0 alpha / closed shell, 1 beta
    DBuf<double> H, S, X, P[2], Pold[2], F[2], G[2], C[2], Fp, Tm, Tm2, V, Z, D0, D1, D2, W0, W1, Dsh, ev[2];
    // per spin: the last eigenvectors of X^T F X (orthogonal basis), the next eigensolve's
    // starting basis once warm[spin] is set
    DBuf<double> Wp[2];
    bool warm[2] = {false, false};
    DBuf<double> dF[kBatchDiis][2], dE[kBatchDiis][2];
    DBuf<double> red;
    Scratch scratch;
    // the Fock kernels' pair data and launches over all molecules, every pair's molecule, the
    // per-molecule active flags, and the build captured as a HIP graph (replayed every
    // iteration of a run)
    FockStore fs;
    DBuf<int> pmol, active_d;
    int maxn = 0, maxsh = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t gexec = nullptr;
    int use_graph = 1;
    int use_queue = 1;   // accepted and read back; the launches take no work from a queue
    // the launches go round-robin over st and launch_streams - 1 worker streams (forked from st
    // and joined back; under capture the graph then holds parallel branches)
    int launch_streams = 3;
    LaunchStreams ls;
    int graph_builds = 0, graph_replays = 0, space_builds = 0;
    void drop_graph() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        gexec = nullptr;
        graph = nullptr;
    }
    ~uno_batch() {
        drop_graph();
        for (BatchMol& m : mol)
            if (m.ctx) uno_ctx_destroy(m.ctx);
        if (st) (void)hipStreamSynchronize(st);
        if (st) (void)hipStreamDestroy(st);
    }
};

namespace {

// slots: per (molecule, spin) matrix; spin 1 only for UHF molecules
void make_slots(const uno_batch* b, bool only_active, int spin, std::vector<MatSlot>& out, std::vector<int>& who) {
    out.clear();
    who.clear();
    for (int m = 0; m < (int)b->mol.size(); ++m) {
        const BatchMol& x = b->mol[m];
        if (only_active && !x.active) continue;
        if (spin == 1 && !x.uhf) continue;
        out.push_back(MatSlot{x.moff, x.n});
        who.push_back(m);
    }
}

struct GemmBatch {
    std::vector<GemmGroup> g;
    std::vector<GemmTile> t;
    Scratch* sc;
    explicit GemmBatch(Scratch& s) : sc(&s) {}
    void add(int m, int n, int k, bool ta, bool tb, const double* A, const double* B, double* C, int lda, int ldb,
             int ldc) {
        if (m <= 0 || n <= 0 || k <= 0) return;
        const int gi = (int)g.size();
        g.push_back(GemmGroup{m, n, k, ta ? 1 : 0, tb ? 1 : 0, A, B, C, lda, ldb, ldc});
        for (int i = 0; i < (m + 31) / 32; ++i)
            for (int j = 0; j < (n + 31) / 32; ++j) t.push_back(GemmTile{gi, i, j});
    }
    int run(double alpha, double beta, hipStream_t st) {
        if (t.empty()) return UNO_OK;
        GemmGroup* dg = nullptr;
        GemmTile* dt = nullptr;
        UNO_HIP(sc->upload(g.data(), g.size(), st, &dg));
        UNO_HIP(sc->upload(t.data(), t.size(), st, &dt));
        UNO_HIP(grouped_gemm((int)t.size(), dt, dg, alpha, beta, st));
        // the group / tile arrays are pageable host memory: keep them alive until done
        UNO_HIP(hipStreamSynchronize(st));
        return UNO_OK;
    }
};

// Z, evals of every slot's symmetric matrix A (destroyed), A given per slot
int batch_eigh(uno_batch* b, const std::vector<MatSlot>& sl, double* A, double* evals_base,
               const std::vector<long long>& evoff) {
    std::vector<BatchMat> bm(sl.size());
    for (size_t k = 0; k < sl.size(); ++k)
        bm[k] = BatchMat{sl[k].n, A + sl[k].off, b->V.p + sl[k].off, evals_base + evoff[k], b->Z.p + sl[k].off};
    BatchMat* d = nullptr;
    UNO_HIP(b->scratch.upload(bm.data(), bm.size(), b->st, &d));
    UNO_HIP(batched_jacobi((int)bm.size(), d, b->maxn, 50, nullptr, b->st));
    UNO_HIP(hipStreamSynchronize(b->st));
    return UNO_OK;
}

}  // namespace

namespace uno {

// the launches of one build: accumulators and density maxima cleared by a fill kernel (no memset
// nodes when captured), the densities in the pairs' order, one launch per class pair and shell
// kind, and the Coulomb accumulator into W
static int enqueue_fock(uno_batch* b) {
    hipStream_t st = b->st;
    FockStore& fs = b->fs;
    const int np = fs.npair, nm = (int)b->mol.size();
    ClearList cl;
    cl.add(b->W0.p, b->store);
    cl.add(b->W1.p, b->store);
    cl.add(fs.jp.p, fs.njp);
    cl.add(fs.dmax.p, nm);
    cl.add(fs.ctr.p, 2 * (long long)fs.launches.size());
    UNO_HIP(fock_clear(cl, st));
    UNO_HIP(batch_shell_max(nm, b->maxsh, b->mdesc.p, b->mshoff.p, b->active_d.p, b->sh_off.p, b->sh_n.p, b->D0.p, b->D1.p, b->D2.p,
                            b->Dsh.p, fs.dmax.p, st));
    UNO_HIP(pair_density(np, fs.kidx.p, fs.kjo.p, b->D0.p, b->Dsh.p, 0, 0, b->mdesc.p, b->pmol.p, fs.dp.p, fs.dpair.p, st));
    const uno_ctx* c0 = b->mol[0].ctx;
    if (!fs.launches.empty()) {
        FockArgs a = fs.args(0, 0, false, b->pairs.p, b->prims.p, b->pairQ.p);
        a.tau = c0->tau;
        a.mols = b->mdesc.p;
        a.mol_active = b->active_d.p;
        if (int rc = fs.list_tasks(false, a, st)) return rc;
    }
    const int nls = std::max(1, std::min(kMaxLaunchStreams, b->launch_streams));
    if (int rc = b->ls.begin(nls, st)) return rc;
    for (size_t k = 0; k < fs.launches.size(); ++k) {
        const FockLaunch& l = fs.launches[k];
        const bool uhf = l.group != 0;
        FockArgs a = fs.args((int)k, 0, false, b->pairs.p, b->prims.p, b->pairQ.p);
        a.tau = c0->tau;
        a.primcut = c0->primcut;
        a.rys2_exact = c0->rys2_exact;
        a.n = b->maxn;
        a.nsh = b->maxsh;
        a.dsh = b->Dsh.p;
        a.jp = fs.jp.p;
        a.nquart = fs.nquart.p;
        a.D0 = b->D0.p;
        a.W0 = b->W0.p;
        if (uhf) {
            a.D1 = b->D1.p;
            a.D2 = b->D2.p;
            a.W1 = b->W1.p;
        }
        a.mols = b->mdesc.p;
        a.mol_active = b->active_d.p;
        const int mode = uhf ? kDigestUHF : kDigestRHF;
        const FockConfig f = fock_default(l.cx, l.cy, mode, l.ncols, b->maxsh, false, true, 0, -1);
        UNO_HIP(fock_launch(mode, false, l.cx, l.cy, a, f, l.ncols, b->ls.of((int)(k % (size_t)nls), st)));
    }
    if (int rc = b->ls.end(nls, st)) return rc;
    UNO_HIP(jp_scatter(np, fs.kidx.p, fs.kjo.p, fs.jp.p, b->W0.p, b->W1.p, 0, b->mdesc.p, b->pmol.p, st));
    return UNO_OK;
}

// batched Fock build on the densities in D0 (D1, D2): W0 (W1) accumulators
static int batch_fock(uno_batch* b) {
    hipStream_t st = b->st;
    const int nm = (int)b->mol.size();
    std::vector<int> act(nm);
    for (int m = 0; m < nm; ++m) act[m] = b->mol[m].active ? 1 : 0;
    UNO_HIP(hipMemcpyAsync(b->active_d.p, act.data(), nm * sizeof(int), hipMemcpyHostToDevice, st));
    if (int rc = b->ls.prepare(std::max(1, std::min(kMaxLaunchStreams, b->launch_streams)))) return rc;
    if (b->use_graph) {
        if (!b->gexec) {
            UNO_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            const int rc = enqueue_fock(b);
            hipGraph_t g = nullptr;
            const hipError_t ee = hipStreamEndCapture(st, &g);
            if (rc || ee != hipSuccess) {
                if (g) (void)hipGraphDestroy(g);
                if (rc) return rc;
                UNO_HIP(ee);
            }
            b->graph = g;
            UNO_HIP(hipGraphInstantiate(&b->gexec, b->graph, nullptr, nullptr, 0));
            ++b->graph_builds;
        }
        UNO_HIP(hipGraphLaunch(b->gexec, st));
        ++b->graph_replays;
    } else {
        if (int rc = enqueue_fock(b)) return rc;
    }
    UNO_HIP(hipStreamSynchronize(st));
    return UNO_OK;
}

}  // namespace uno

extern "C" {

int uno_batch_create(int nmol, const uno_basis* bases, const int* nelec, uno_batch** out) {
    if (nmol <= 0 || !bases || !nelec || !out) { set_error("bad argument"); return UNO_EINVAL; }
    auto* b = new uno_batch;
    b->mol.resize(nmol);
    std::vector<PairHdr> pairs;
    std::vector<PrimPair> prims;
    std::vector<double> q;
    std::vector<int> shoff, shn;
    std::vector<MolDesc> md;
    std::vector<int> pmol, mshoff;
    for (int m = 0; m < nmol; ++m) {
        BatchMol& x = b->mol[m];
        if (int rc = uno_ctx_create(&bases[m], 0, &x.ctx)) { delete b; return rc; }
        uno_ctx* c = x.ctx;
        x.n = c->n;
        x.nsh = c->nsh;
        x.nelec = nelec[m];
        x.uhf = nelec[m] % 2 != 0;
        x.nocc[0] = x.uhf ? nelec[m] - nelec[m] / 2 : nelec[m] / 2;
        x.nocc[1] = nelec[m] / 2;
        if (x.n > 256 || nelec[m] <= 0 || x.nocc[0] > x.n) {
            set_error("batched SCF: molecule " + std::to_string(m) + " has more than 256 functions or a bad "
                      "electron count");
            delete b;
            return UNO_EINVAL;
        }
        x.moff = b->store;
        b->store += (long long)x.n * x.n;
        x.dshoff = b->dsh_total;
        b->dsh_total += (long long)x.nsh * x.nsh;
        x.shoff = (int)shoff.size();
        for (int s = 0; s < x.nsh; ++s) {
            shoff.push_back(c->B.off[s]);
            shn.push_back(ncart(c->B.sh[s].l));
        }
        x.pair_off = (int)pairs.size();
        const int p0 = (int)prims.size();
        for (PairHdr h : c->pairs) {
            h.prim0 += p0;
            pairs.push_back(h);
            pmol.push_back(m);
        }
        mshoff.push_back(x.shoff);
        b->maxn = std::max(b->maxn, x.n);
        b->maxsh = std::max(b->maxsh, x.nsh);
        prims.insert(prims.end(), c->prims.begin(), c->prims.end());
        q.insert(q.end(), c->pairQ.begin(), c->pairQ.end());
        md.push_back(MolDesc{x.moff, x.dshoff, x.n, x.nsh});
        for (int i = 0; i < c->B.ncen; ++i)
            for (int j = i + 1; j < c->B.ncen; ++j) {
                const double* r1 = &c->B.xyz[3 * i];
                const double* r2 = &c->B.xyz[3 * j];
                const double dx = r1[0] - r2[0], dy = r1[1] - r2[1], dz = r1[2] - r2[2];
                x.nuc += c->B.q[i] * c->B.q[j] / std::sqrt(dx * dx + dy * dy + dz * dz);
            }
    }
    int ndev = 0;
    (void)hipGetDeviceCount(&ndev);
    hipError_t e = hipStreamCreate(&b->st);
    if (e != hipSuccess) { set_error("HIP stream creation failed"); delete b; return UNO_EDEVICE; }
    hipStream_t st = b->st;
    auto up = [&](auto& buf, const auto& v) { return buf.upload(v.data(), v.size(), st); };
    if (up(b->pairs, pairs) != hipSuccess || up(b->prims, prims) != hipSuccess || up(b->pairQ, q) != hipSuccess ||
        up(b->sh_off, shoff) != hipSuccess || up(b->sh_n, shn) != hipSuccess || up(b->mdesc, md) != hipSuccess || up(b->pmol, pmol) != hipSuccess ||
        up(b->mshoff, mshoff) != hipSuccess || b->active_d.alloc(nmol) != hipSuccess) {
        set_error("batched SCF: device upload failed");
        delete b;
        return UNO_ENOMEM;
    }
    {
        std::vector<FockMol> fm(nmol);
        for (int m = 0; m < nmol; ++m) {
            const BatchMol& x = b->mol[m];
            fm[m] = FockMol{x.n, m, x.uhf ? 1 : 0, &x.ctx->cls, x.pair_off, pairs.data() + x.pair_off};
        }
        if (int rc = b->fs.build(fm, b->pairs.p, b->prims.p, (int)pairs.size(), (long long)prims.size(), st)) {
            delete b;
            return rc;
        }
    }
    const size_t S = (size_t)b->store;
    DBuf<double>* stores[] = {&b->H, &b->S, &b->X, &b->P[0], &b->P[1], &b->Pold[0], &b->Pold[1], &b->F[0], &b->F[1],
                              &b->G[0], &b->G[1], &b->C[0], &b->C[1], &b->Fp, &b->Tm, &b->Tm2, &b->V, &b->Z,
                              &b->D0, &b->D1, &b->D2, &b->W0, &b->W1, &b->Wp[0], &b->Wp[1]};
    for (DBuf<double>* p : stores)
        if (p->alloc(S) != hipSuccess) { set_error("batched SCF: device allocation failed"); delete b; return UNO_ENOMEM; }
    for (int k = 0; k < kBatchDiis; ++k)
        for (int s = 0; s < 2; ++s)
            if (b->dF[k][s].alloc(S) != hipSuccess || b->dE[k][s].alloc(S) != hipSuccess) {
                set_error("batched SCF: device allocation failed");
                delete b;
                return UNO_ENOMEM;
            }
    if (b->Dsh.alloc(std::max<long long>(1, b->dsh_total)) != hipSuccess || b->ev[0].alloc(S) != hipSuccess ||
        b->ev[1].alloc(S) != hipSuccess || b->red.alloc(8 * (size_t)nmol * (kBatchDiis + 4)) != hipSuccess) {
        set_error("batched SCF: device allocation failed");
        delete b;
        return UNO_ENOMEM;
    }
    *out = b;
    return UNO_OK;
}

int uno_batch_destroy(uno_batch* b) {
    delete b;
    return UNO_OK;
}

int uno_batch_nmol(const uno_batch* b) { return b ? (int)b->mol.size() : 0; }

int uno_batch_set(uno_batch* b, const char* key, double v) {
    if (!b || !key) { set_error("null argument"); return UNO_EINVAL; }
    const std::string k(key);
    if (k == "graph") b->use_graph = (int)v;
    else if (k == "queue") b->use_queue = (int)v;
    else if (k == "launch_streams") {
        b->launch_streams = std::max(1, std::min(kMaxLaunchStreams, (int)v));
        b->drop_graph();   // a captured build keeps the stream layout it was captured with
    }
    else { set_error("unknown batch option " + k); return UNO_EINVAL; }
    b->drop_graph();
    return UNO_OK;
}

int uno_batch_get(const uno_batch* b, const char* key, double* v) {
    if (!b || !key || !v) { set_error("null argument"); return UNO_EINVAL; }
    const std::string k(key);
    if (k == "graph") *v = b->use_graph;
    else if (k == "queue") *v = b->use_queue;
    else if (k == "launch_streams") *v = b->launch_streams;
    else if (k == "space_builds") *v = b->space_builds;
    else if (k == "graph_builds") *v = b->graph_builds;
    else if (k == "graph_replays") *v = b->graph_replays;
    else if (k == "launches_per_build") *v = (double)b->fs.launches.size();
    else { set_error("unknown batch option " + k); return UNO_EINVAL; }
    return UNO_OK;
}

int uno_batch_density(const uno_batch* b, int m, double* P) {
    if (!b || !P || m < 0 || m >= (int)b->mol.size()) { set_error("bad argument"); return UNO_EINVAL; }
    const BatchMol& x = b->mol[m];
    const size_t nn = (size_t)x.n * x.n;
    if (!b->P[0].p) { set_error("the batch has not run"); return UNO_EINVAL; }
    UNO_HIP(hipMemcpyAsync(P, b->P[0].p + x.moff, nn * sizeof(double), hipMemcpyDeviceToHost, b->st));
    if (x.uhf) UNO_HIP(hipMemcpyAsync(P + nn, b->P[1].p + x.moff, nn * sizeof(double), hipMemcpyDeviceToHost, b->st));
    UNO_HIP(hipStreamSynchronize(b->st));
    return UNO_OK;
}

int uno_batch_run(uno_batch* b, const uno_scf_opts* opts, uno_scf_result* res, double* energies) {
    if (!b || !res) { set_error("null argument"); return UNO_EINVAL; }
    uno_scf_opts o;
    if (opts) o = *opts; else uno_scf_defaults(&o);
    if (o.precision || o.incremental || o.guess != 0) {
        set_error("batched SCF: FP64 full builds from the core-Hamiltonian guess only");
        return UNO_EINVAL;
    }
    const auto t0 = clk::now();
    hipStream_t st = b->st;
    b->scratch.reset();
    b->warm[0] = b->warm[1] = false;
    // the captured build belongs to one run
    b->drop_graph();
    b->space_builds = 1;
    b->graph_builds = b->graph_replays = 0;
    {
        ClearList cl;
        cl.add(b->fs.nquart.p, 2 * kQuartSlots);
        UNO_HIP(fock_clear(cl, st));
    }
    const int nm = (int)b->mol.size();
    const long long S = b->store;
    // per-molecule eigenvalue offsets into ev stores: reuse the matrix offsets (n <= n^2)
    // one-electron matrices of every molecule
    for (BatchMol& x : b->mol) {
        x.active = true;
        x.converged = false;
        x.iterations = 0;
        x.eold = x.energy = x.ediff = x.pdiff = 0.0;
        if (int rc = oneint_device(x.ctx, b->S.p + x.moff, b->Tm.p + x.moff, b->H.p + x.moff)) return rc;
        UNO_HIP(hipStreamSynchronize(x.ctx->st));
    }
    for (int s = 0; s < 2; ++s) {
        UNO_HIP(k_fill(S, 0.0, b->P[s].p, st));
        UNO_HIP(k_fill(S, 0.0, b->G[s].p, st));
    }
    std::vector<MatSlot> sl[2];
    std::vector<int> who[2];
    std::vector<DBuf<MatSlot>> dsl(2);
    auto refresh_slots = [&]() -> int {
        for (int s = 0; s < 2; ++s) {
            make_slots(b, true, s, sl[s], who[s]);
            if (!sl[s].empty()) UNO_HIP(dsl[s].upload(sl[s].data(), sl[s].size(), st));
        }
        return UNO_OK;
    };
    if (int rc = refresh_slots()) return rc;
    auto evoff = [&](int s) {
        std::vector<long long> o;
        for (const MatSlot& m : sl[s]) o.push_back(m.off);
        return o;
    };
    // X = U s^-1/2 (RHF.hpp:214-233): Jacobi of S, column scaling on the host read-back
    {
        UNO_HIP(hipMemcpyAsync(b->Tm.p, b->S.p, S * sizeof(double), hipMemcpyDeviceToDevice, st));
        if (int rc = batch_eigh(b, sl[0], b->Tm.p, b->ev[0].p, evoff(0))) return rc;
        std::vector<double> ev(S), Z(S);
        UNO_HIP(hipMemcpyAsync(ev.data(), b->ev[0].p, S * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipMemcpyAsync(Z.data(), b->Z.p, S * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        for (const BatchMol& x : b->mol) {
            for (int j = 0; j < x.n; ++j) {
                double f = ev[x.moff + j];
                if (std::fabs(f) < 1e-7 && f < 0.0) f = -f;
                if (!(f > 0.0)) { set_error("Zero or negative eigenvalue in an overlap matrix"); return UNO_ESINGULAR; }
                const double sc = 1.0 / std::sqrt(f);
                for (int i = 0; i < x.n; ++i) Z[x.moff + (long long)i * x.n + j] *= sc;
            }
        }
        UNO_HIP(b->X.upload(Z.data(), S, st));
    }
    // F (store, per spin) -> P per spin slot: X^T F X, Jacobi, C = X W, P = C_occ C_occ^T
    double diag_s = 0.0;
    auto diag_to_P = [&](int s, const double* Fs) -> int {
        if (sl[s].empty()) return UNO_OK;
        const auto td = clk::now();
        struct Acc { double& t; clk::time_point t0; ~Acc() { t += secs(t0, clk::now()); } } acc{diag_s, td};
        GemmBatch g1(b->scratch), g2(b->scratch);
        for (const MatSlot& m : sl[s]) g1.add(m.n, m.n, m.n, false, false, Fs + m.off, b->X.p + m.off, b->Tm.p + m.off, m.n, m.n, m.n);
        if (int rc = g1.run(1.0, 0.0, st)) return rc;
        for (const MatSlot& m : sl[s]) g2.add(m.n, m.n, m.n, true, false, b->X.p + m.off, b->Tm.p + m.off, b->Fp.p + m.off, m.n, m.n, m.n);
        if (int rc = g2.run(1.0, 0.0, st)) return rc;
        // after their first eigensolve the molecules start from their last eigenvectors Wp:
        // in that basis the matrix is nearly diagonal and the Jacobi sweeps settle in a few
        // rounds (W = Wp Z after)
        std::vector<char> warm(sl[s].size(), 0);
        GemmBatch w1(b->scratch), w2(b->scratch), w3(b->scratch);
        for (size_t k = 0; k < sl[s].size(); ++k) {
            const MatSlot& m = sl[s][k];
            warm[k] = b->warm[s];
            if (warm[k]) {
                w1.add(m.n, m.n, m.n, false, false, b->Fp.p + m.off, b->Wp[s].p + m.off, b->Tm.p + m.off, m.n, m.n, m.n);
                w2.add(m.n, m.n, m.n, true, false, b->Wp[s].p + m.off, b->Tm.p + m.off, b->Tm2.p + m.off, m.n, m.n, m.n);
                w3.add(m.n, m.n, m.n, false, false, b->Wp[s].p + m.off, b->Z.p + m.off, b->Tm.p + m.off, m.n, m.n, m.n);
            }
        }
        if (int rc = w1.run(1.0, 0.0, st)) return rc;
        if (int rc = w2.run(1.0, 0.0, st)) return rc;
        {
            std::vector<BatchMat> bm(sl[s].size());
            for (size_t k = 0; k < sl[s].size(); ++k) {
                const MatSlot& m = sl[s][k];
                bm[k] = BatchMat{m.n, (warm[k] ? b->Tm2.p : b->Fp.p) + m.off, b->V.p + m.off, b->ev[s].p + m.off,
                                 b->Z.p + m.off};
            }
            BatchMat* d = nullptr;
            UNO_HIP(b->scratch.upload(bm.data(), bm.size(), st, &d));
            UNO_HIP(batched_jacobi((int)bm.size(), d, b->maxn, 50, nullptr, st));
            // bm is pageable host memory: its upload must be done before it goes
            UNO_HIP(hipStreamSynchronize(st));
        }
        if (int rc = w3.run(1.0, 0.0, st)) return rc;
        // the new starting bases in one launch: Wp Z (warm, in Tm) or Z (cold)
        {
            std::vector<double> coef(2 * sl[s].size());
            for (size_t k = 0; k < sl[s].size(); ++k) {
                coef[2 * k] = warm[k] ? 1.0 : 0.0;
                coef[2 * k + 1] = warm[k] ? 0.0 : 1.0;
            }
            const double* src[2] = {b->Tm.p, b->Z.p};
            double* dcoef = nullptr;
            const double** dsrc = nullptr;
            UNO_HIP(b->scratch.upload(coef.data(), coef.size(), st, &dcoef));
            UNO_HIP(b->scratch.upload(src, 2, st, &dsrc));
            UNO_HIP(batch_lincomb((int)sl[s].size(), dsl[s].p, 2, dcoef, dsrc, b->Wp[s].p, st));
            UNO_HIP(hipStreamSynchronize(st));
        }
        b->warm[s] = true;
        GemmBatch g3(b->scratch), g4(b->scratch);
        for (const MatSlot& m : sl[s]) g3.add(m.n, m.n, m.n, false, false, b->X.p + m.off, b->Wp[s].p + m.off, b->C[s].p + m.off, m.n, m.n, m.n);
        if (int rc = g3.run(1.0, 0.0, st)) return rc;
        for (size_t k = 0; k < sl[s].size(); ++k) {
            const MatSlot& m = sl[s][k];
            g4.add(m.n, m.n, b->mol[who[s][k]].nocc[s], false, true, b->C[s].p + m.off, b->C[s].p + m.off,
                   b->P[s].p + m.off, m.n, m.n, m.n);
        }
        return g4.run(1.0, 0.0, st);
    };
    // core-Hamiltonian guess (UHF beta reuses the alpha orbitals, UHF.hpp:206-215)
    if (int rc = diag_to_P(0, b->H.p)) return rc;
    if (!sl[1].empty()) {
        GemmBatch g(b->scratch);
        for (size_t k = 0; k < sl[1].size(); ++k) {
            const MatSlot& m = sl[1][k];
            g.add(m.n, m.n, b->mol[who[1][k]].nocc[1], false, true, b->C[0].p + m.off, b->C[0].p + m.off,
                  b->P[1].p + m.off, m.n, m.n, m.n);
        }
        if (int rc = g.run(1.0, 0.0, st)) return rc;
    }
    double eps = o.eps;
    std::vector<double> hs(4 * (size_t)nm + 8);
    int ndiis = 0, slot_next = 0;
    std::vector<double> Bm((size_t)nm * kBatchDiis * kBatchDiis, 0.0);
    int iteration = 0;
    double fock_s = 0.0;
    int nstopped = 0;
    double wall99 = -1.0;
    while (true) {
        b->scratch.reset();   // the previous iteration ended synchronised
        // densities of the build: D1 = Pa, D2 = Pb (zero for closed shells), D0 = D1 + D2
        const auto tf = clk::now();
        UNO_HIP(hipMemcpyAsync(b->D1.p, b->P[0].p, S * sizeof(double), hipMemcpyDeviceToDevice, st));
        UNO_HIP(hipMemcpyAsync(b->D2.p, b->P[1].p, S * sizeof(double), hipMemcpyDeviceToDevice, st));
        UNO_HIP(k_axpby(S, 1.0, b->D1.p, 1.0, b->D2.p, b->D0.p, st));
        if (int rc = batch_fock(b)) return rc;
        UNO_HIP(batch_sym((int)sl[0].size(), dsl[0].p, b->W0.p, b->G[0].p, false, st));
        if (!sl[1].empty()) UNO_HIP(batch_sym((int)sl[1].size(), dsl[1].p, b->W1.p, b->G[1].p, false, st));
        fock_s += secs(tf, clk::now());
        // energies: e1 = tr(Pa H) + tr(Pb H), e2 = tr(Pa Ga) + tr(Pb Gb)
        double* r = b->red.p;
        const int n0 = (int)sl[0].size();
        UNO_HIP(batch_dot(n0, dsl[0].p, b->P[0].p, b->H.p, r, false, st));
        UNO_HIP(batch_dot(n0, dsl[0].p, b->P[1].p, b->H.p, r, true, st));
        UNO_HIP(batch_dot(n0, dsl[0].p, b->P[0].p, b->G[0].p, r + nm, false, st));
        UNO_HIP(batch_dot(n0, dsl[0].p, b->P[1].p, b->G[1].p, r + nm, true, st));
        UNO_HIP(hipMemcpyAsync(hs.data(), r, 2 * (size_t)nm * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        for (int k = 0; k < n0; ++k) {
            BatchMol& x = b->mol[who[0][k]];
            const double e1 = hs[k], e2 = hs[nm + k];
            x.energy = x.uhf ? e1 + 0.5 * e2 : 2.0 * e1 + e2;
            x.ediff = x.energy - x.eold;
            x.eold = x.energy;
            if (iteration == 0) x.init_energy = x.energy + x.nuc;
        }
        // F = H + G; DIIS on every active slot (one shared history position per iteration)
        for (int s = 0; s < 2; ++s) UNO_HIP(k_axpby(S, 1.0, b->H.p, 1.0, b->G[s].p, b->F[s].p, st));
        const int slot = slot_next;
        slot_next = (slot_next + 1) % kBatchDiis;
        if (ndiis < kBatchDiis) ++ndiis;
        for (int s = 0; s < 2; ++s) {
            if (sl[s].empty()) continue;
            UNO_HIP(hipMemcpyAsync(b->dF[slot][s].p, b->F[s].p, S * sizeof(double), hipMemcpyDeviceToDevice, st));
            GemmBatch g1(b->scratch), g2(b->scratch), g3(b->scratch), g4(b->scratch);
            for (const MatSlot& m : sl[s]) g1.add(m.n, m.n, m.n, false, false, b->F[s].p + m.off, b->P[s].p + m.off, b->Tm.p + m.off, m.n, m.n, m.n);
            if (int rc = g1.run(1.0, 0.0, st)) return rc;
            for (const MatSlot& m : sl[s]) g2.add(m.n, m.n, m.n, false, false, b->Tm.p + m.off, b->S.p + m.off, b->Fp.p + m.off, m.n, m.n, m.n);
            if (int rc = g2.run(1.0, 0.0, st)) return rc;
            // FPS - SPF = FPS - (FPS)^T
            UNO_HIP(batch_sym((int)sl[s].size(), dsl[s].p, b->Fp.p, b->Tm2.p, false, st));
            UNO_HIP(k_axpby(S, 2.0, b->Fp.p, -1.0, b->Tm2.p, b->Tm2.p, st));
            for (const MatSlot& m : sl[s]) g3.add(m.n, m.n, m.n, false, false, b->Tm2.p + m.off, b->X.p + m.off, b->Tm.p + m.off, m.n, m.n, m.n);
            if (int rc = g3.run(1.0, 0.0, st)) return rc;
            for (const MatSlot& m : sl[s]) g4.add(m.n, m.n, m.n, true, false, b->X.p + m.off, b->Tm.p + m.off, b->dE[slot][s].p + m.off, m.n, m.n, m.n);
            if (int rc = g4.run(1.0, 0.0, st)) return rc;
        }
        // B-matrix row of the new vector: sum over spins of <E_new, E_j>
        std::vector<double> row((size_t)kBatchDiis * nm, 0.0);
        for (int j = 0; j < ndiis; ++j) {
            UNO_HIP(batch_dot(n0, dsl[0].p, b->dE[slot][0].p, b->dE[j][0].p, r, false, st));
            std::vector<double> t0v(n0);
            UNO_HIP(hipMemcpyAsync(t0v.data(), r, n0 * sizeof(double), hipMemcpyDeviceToHost, st));
            std::vector<double> t1v(sl[1].size());
            if (!sl[1].empty()) {
                UNO_HIP(batch_dot((int)sl[1].size(), dsl[1].p, b->dE[slot][1].p, b->dE[j][1].p, r + nm, false, st));
                UNO_HIP(hipMemcpyAsync(t1v.data(), r + nm, t1v.size() * sizeof(double), hipMemcpyDeviceToHost, st));
            }
            UNO_HIP(hipStreamSynchronize(st));
            for (int k = 0; k < n0; ++k) row[(size_t)who[0][k] * kBatchDiis + j] = t0v[k];
            for (size_t k = 0; k < t1v.size(); ++k) row[(size_t)who[1][k] * kBatchDiis + j] += t1v[k];
        }
        std::vector<double> coef((size_t)n0 * kBatchDiis, 0.0);
        bool any = false;
        for (int k = 0; k < n0; ++k) {
            const int m = who[0][k];
            double* Bmm = &Bm[(size_t)m * kBatchDiis * kBatchDiis];
            for (int j = 0; j < ndiis; ++j) Bmm[slot * kBatchDiis + j] = Bmm[j * kBatchDiis + slot] = row[(size_t)m * kBatchDiis + j];
            coef[(size_t)k * kBatchDiis + slot] = 1.0;
            if (ndiis >= 2 && diis_coefficients(Bmm, kBatchDiis, ndiis, slot, &coef[(size_t)k * kBatchDiis]) >= 2)
                any = true;
        }
        if (any) {
            for (int s = 0; s < 2; ++s) {
                if (sl[s].empty()) continue;
                std::vector<const double*> src(kBatchDiis);
                for (int j = 0; j < kBatchDiis; ++j) src[j] = b->dF[j][s].p;
                const double** dsrc = nullptr;
                UNO_HIP(b->scratch.upload(src.data(), src.size(), st, &dsrc));
                // coefficients of slot k of spin s: the molecule's row (spin 1 slots are a subset)
                std::vector<double> cs((size_t)sl[s].size() * kBatchDiis);
                for (size_t k = 0; k < sl[s].size(); ++k) {
                    const int m = who[s][k];
                    const size_t k0 = std::find(who[0].begin(), who[0].end(), m) - who[0].begin();
                    std::copy(&coef[k0 * kBatchDiis], &coef[k0 * kBatchDiis] + kBatchDiis, &cs[k * kBatchDiis]);
                }
                double* dcs = nullptr;
                UNO_HIP(b->scratch.upload(cs.data(), cs.size(), st, &dcs));
                UNO_HIP(batch_lincomb((int)sl[s].size(), dsl[s].p, kBatchDiis, dcs, dsrc, b->F[s].p, st));
                UNO_HIP(hipStreamSynchronize(st));
            }
        }
        // new densities
        for (int s = 0; s < 2; ++s)
            UNO_HIP(hipMemcpyAsync(b->Pold[s].p, b->P[s].p, S * sizeof(double), hipMemcpyDeviceToDevice, st));
        for (int s = 0; s < 2; ++s)
            if (int rc = diag_to_P(s, b->F[s].p)) return rc;
        UNO_HIP(batch_diffnorm(n0, dsl[0].p, b->P[0].p, b->Pold[0].p, r, st));
        if (!sl[1].empty()) UNO_HIP(batch_diffnorm((int)sl[1].size(), dsl[1].p, b->P[1].p, b->Pold[1].p, r + nm, st));
        std::vector<double> pd(2 * (size_t)nm, 0.0);
        UNO_HIP(hipMemcpyAsync(pd.data(), r, 2 * (size_t)nm * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        ++iteration;
        bool changed = false;
        for (int k = 0; k < n0; ++k) {
            BatchMol& x = b->mol[who[0][k]];
            x.pdiff = pd[k];
            x.iterations = iteration;
        }
        for (size_t k = 0; k < sl[1].size(); ++k) b->mol[who[1][k]].pdiff += pd[nm + k];
        for (int k = 0; k < n0; ++k) {
            BatchMol& x = b->mol[who[0][k]];
            bool conv = false;
            if (iteration >= 2) {
                if (o.cflag == 0) conv = x.ediff < eps;
                else if (o.cflag == 1) conv = x.pdiff < eps;
                else if (o.cflag == 3) conv = std::fabs(x.ediff) < eps;
                else conv = x.pdiff < eps && x.ediff < eps;
            }
            if (conv || iteration >= o.maxits) {
                x.converged = conv;
                x.active = false;
                changed = true;
                ++nstopped;
            }
        }
        if (wall99 < 0.0 && 100 * nstopped >= 99 * nm) wall99 = secs(t0, clk::now());
        if (o.verbose)
            fprintf(stderr, "[batch] iteration %d: %d molecules were active, %d stopped; Fock %.3f s, "
                            "eigen/GEMM %.3f s, wall %.3f s\n", iteration, n0, nstopped, fock_s, diag_s,
                    secs(t0, clk::now()));
        bool any_active = false;
        for (const BatchMol& x : b->mol) any_active = any_active || x.active;
        if (!any_active) break;
        if (changed) {
            if (int rc = refresh_slots()) return rc;
        }
    }
    const double wall = secs(t0, clk::now());
    double quartets = 0.0;
    {
        std::vector<unsigned long long> h(2 * kQuartSlots);
        UNO_HIP(hipMemcpyAsync(h.data(), b->fs.nquart.p, h.size() * sizeof(h[0]), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        for (unsigned long long v : h) quartets += (double)v;
    }
    int rc = UNO_OK;
    for (int m = 0; m < nm; ++m) {
        const BatchMol& x = b->mol[m];
        uno_scf_result& r = res[m];
        std::memset(&r, 0, sizeof(r));
        r.energy = x.energy + x.nuc;
        r.init_energy = x.init_energy;
        r.ediff = x.ediff;
        r.pdiff = x.pdiff;
        r.nucrep = x.nuc;
        r.electronic = x.energy;
        r.iterations = x.iterations;
        r.converged = x.converged ? 1 : 0;
        r.uhf = x.uhf ? 1 : 0;
        r.nfock = x.iterations;
        r.wall_s = wall;
        r.wall99_s = wall99 < 0.0 ? wall : wall99;
        r.fock_s = fock_s;
        r.diag_s = diag_s;
        r.quartets = quartets;
        if (energies) energies[m] = r.energy;
        if (!x.converged) rc = UNO_ENOCONV;
    }
    return rc;
}

}  // extern "C"
