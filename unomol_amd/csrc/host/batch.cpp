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


// pinned host memory, so that the small copies of an iteration are asynchronous
struct Pinned {
    char* p = nullptr;
    size_t n = 0;
    Pinned() = default;
    Pinned(const Pinned&) = delete;
    Pinned& operator=(const Pinned&) = delete;
    hipError_t alloc(size_t bytes) { return n = bytes, hipHostMalloc((void**)&p, bytes, hipHostMallocDefault); }
    ~Pinned() { if (p) (void)hipHostFree(p); }
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
    DBuf<double> H, S, X, D0, P[2], Pold[2], F[2], G[2], C[2], Fp[2], Tm[2], Tm2[2], V[2], Z[2], W[2], Dsh, ev[2];
    // per spin: the last eigenvectors of X^T F X (orthogonal basis), the next eigensolve's
    // starting basis once warm[spin] is set, and the buffer the next ones go to
    DBuf<double> Wp[2], Wn[2];
    bool warm[2] = {false, false};
    DBuf<double> dF[kBatchDiis][2], dE[kBatchDiis][2];
    DBuf<double> red, coef;
    // the active slots, those of spin 0 first (nslot[s] of spin s, of molecules who[k]), and their
    // GEMM tiles in the same order; rewritten when a molecule stops
    DBuf<MatSlot> slots;
    DBuf<GemmTile> tiles;
    int nslot[2] = {0, 0}, ntile[2] = {0, 0};
    std::vector<int> who;
    // host sides of the copies, a place each: written or read only while the stream is idle
    Pinned host;
    int* h_active = nullptr;
    MatSlot* h_slots = nullptr;
    GemmTile* h_tiles = nullptr;
    double *h_coef = nullptr, *h_dots = nullptr, *h_pdiff = nullptr;
    hipEvent_t ev_fock[2] = {}, ev_diag[2] = {};
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
        for (hipEvent_t e : {ev_fock[0], ev_fock[1], ev_diag[0], ev_diag[1]})
            if (e) (void)hipEventDestroy(e);
        if (st) (void)hipStreamDestroy(st);
    }
};

namespace {

Store both(DBuf<double>* x) { return Store{{x[0].p, x[1].p}}; }
Store same(const DBuf<double>& x) { return Store{{x.p, x.p}}; }

// the slots and tiles of the active molecules (spin 1 only for UHF molecules), and the active flags
int refresh_slots(uno_batch* b) {
    b->who.clear();
    int nt = 0;
    for (int s = 0; s < 2; ++s) {
        const int k0 = (int)b->who.size(), t0 = nt;
        for (int m = 0; m < (int)b->mol.size(); ++m) {
            const BatchMol& x = b->mol[m];
            b->h_active[m] = x.active ? 1 : 0;
            if (!x.active || (s == 1 && !x.uhf)) continue;
            const int k = (int)b->who.size();
            b->who.push_back(m);
            b->h_slots[k] = MatSlot{x.moff, x.n, x.nocc[s], s};
            const int nb = (x.n + 31) / 32;
            for (int i = 0; i < nb; ++i)
                for (int j = 0; j < nb; ++j) b->h_tiles[nt++] = GemmTile{k, i, j};
        }
        b->nslot[s] = (int)b->who.size() - k0;
        b->ntile[s] = nt - t0;
    }
    hipStream_t st = b->st;
    UNO_HIP(hipMemcpyAsync(b->active_d.p, b->h_active, b->mol.size() * sizeof(int), hipMemcpyHostToDevice, st));
    UNO_HIP(hipMemcpyAsync(b->slots.p, b->h_slots, b->who.size() * sizeof(MatSlot), hipMemcpyHostToDevice, st));
    UNO_HIP(hipMemcpyAsync(b->tiles.p, b->h_tiles, nt * sizeof(GemmTile), hipMemcpyHostToDevice, st));
    return UNO_OK;
}

// C = op(A) op(B) over the active slots of spins [s0, s1)
int gemm(uno_batch* b, int s0, int s1, bool ta, bool tb, bool occ, Store A, Store B, Store C) {
    const int lo = s0 ? b->ntile[0] : 0, hi = s1 > 1 ? b->ntile[0] + b->ntile[1] : b->ntile[0];
    UNO_HIP(grouped_gemm(hi - lo, b->tiles.p + lo, b->slots.p, ta, tb, occ, A, B, C, b->st));
    return UNO_OK;
}

double elapsed(hipEvent_t* e) {
    float ms = 0.f;
    (void)hipEventElapsedTime(&ms, e[0], e[1]);
    return 1e-3 * ms;
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
    cl.add(b->W[0].p, b->store);
    cl.add(b->W[1].p, b->store);
    cl.add(fs.jp.p, fs.njp);
    cl.add(fs.dmax.p, nm);
    cl.add(fs.ctr.p, 2 * (long long)fs.launches.size());
    UNO_HIP(fock_clear(cl, st));
    UNO_HIP(batch_shell_max(nm, b->maxsh, b->mdesc.p, b->mshoff.p, b->active_d.p, b->sh_off.p, b->sh_n.p, b->D0.p, b->P[0].p, b->P[1].p,
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
        a.W0 = b->W[0].p;
        if (uhf) {
            a.D1 = b->P[0].p;
            a.D2 = b->P[1].p;
            a.W1 = b->W[1].p;
        }
        a.mols = b->mdesc.p;
        a.mol_active = b->active_d.p;
        const int mode = uhf ? kDigestUHF : kDigestRHF;
        const FockConfig f = fock_default(l.cx, l.cy, mode, l.ncols, b->maxsh, false, true, 0, -1);
        UNO_HIP(fock_launch(mode, false, l.cx, l.cy, a, f, l.ncols, b->ls.of((int)(k % (size_t)nls), st)));
    }
    if (int rc = b->ls.end(nls, st)) return rc;
    UNO_HIP(jp_scatter(np, fs.kidx.p, fs.kjo.p, fs.jp.p, b->W[0].p, b->W[1].p, 0, b->mdesc.p, b->pmol.p, st));
    return UNO_OK;
}

// batched Fock build on the densities in P, D0 their sum: W accumulators
static int batch_fock(uno_batch* b) {
    hipStream_t st = b->st;
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
        ++b->space_builds;
    }
    const size_t S = (size_t)b->store;
    DBuf<double>* stores[] = {&b->H, &b->S, &b->X, &b->P[0], &b->P[1], &b->Pold[0], &b->Pold[1], &b->F[0], &b->F[1],
                              &b->G[0], &b->G[1], &b->C[0], &b->C[1], &b->Fp[0], &b->Fp[1], &b->Tm[0], &b->Tm[1],
                              &b->Tm2[0], &b->Tm2[1], &b->V[0], &b->V[1], &b->Z[0], &b->Z[1], &b->D0, &b->W[0],
                              &b->W[1], &b->Wp[0], &b->Wp[1], &b->Wn[0], &b->Wn[1]};
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
        b->ev[1].alloc(S) != hipSuccess) {
        set_error("batched SCF: device allocation failed");
        delete b;
        return UNO_ENOMEM;
    }
    // the iteration's small arrays, sized for every slot active
    size_t ns = 0, nt = 0;
    for (const BatchMol& x : b->mol) {
        const size_t nb = (x.n + 31) / 32, k = x.uhf ? 2 : 1;
        ns += k;
        nt += k * nb * nb;
    }
    const size_t sz[6] = {nmol * sizeof(int), ns * sizeof(MatSlot), nt * sizeof(GemmTile), ns * kMaxLin * sizeof(double),
                          ns * kMaxDots * sizeof(double), ns * sizeof(double)};
    size_t at[7] = {};
    for (int k = 0; k < 6; ++k) at[k + 1] = at[k] + (sz[k] + 63) / 64 * 64;
    if (b->slots.alloc(ns) != hipSuccess || b->tiles.alloc(nt) != hipSuccess || b->coef.alloc(ns * kMaxLin) != hipSuccess ||
        b->red.alloc(ns * kMaxDots) != hipSuccess || b->host.alloc(at[6]) != hipSuccess) {
        set_error("batched SCF: allocation failed");
        delete b;
        return UNO_ENOMEM;
    }
    b->h_active = reinterpret_cast<int*>(b->host.p + at[0]);
    b->h_slots = reinterpret_cast<MatSlot*>(b->host.p + at[1]);
    b->h_tiles = reinterpret_cast<GemmTile*>(b->host.p + at[2]);
    b->h_coef = reinterpret_cast<double*>(b->host.p + at[3]);
    b->h_dots = reinterpret_cast<double*>(b->host.p + at[4]);
    b->h_pdiff = reinterpret_cast<double*>(b->host.p + at[5]);
    for (hipEvent_t* ep : {&b->ev_fock[0], &b->ev_fock[1], &b->ev_diag[0], &b->ev_diag[1]})
        if (hipEventCreate(ep) != hipSuccess) {
            set_error("HIP event creation failed");
            delete b;
            return UNO_EDEVICE;
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
    b->warm[0] = b->warm[1] = false;
    // the captured build belongs to one run
    b->drop_graph();
    b->graph_builds = b->graph_replays = 0;
    {
        ClearList cl;
        cl.add(b->fs.nquart.p, 2 * kQuartSlots);
        UNO_HIP(fock_clear(cl, st));
    }
    const int nm = (int)b->mol.size();
    const long long S = b->store;
    // (the eigenvalues of a slot are at its matrix offset: n <= n^2)
    // one-electron matrices of every molecule
    for (BatchMol& x : b->mol) {
        x.active = true;
        x.converged = false;
        x.iterations = 0;
        x.eold = x.energy = x.ediff = x.pdiff = 0.0;
        if (int rc = oneint_device(x.ctx, b->S.p + x.moff, b->Tm[0].p + x.moff, b->H.p + x.moff)) return rc;
    }
    for (BatchMol& x : b->mol) UNO_HIP(hipStreamSynchronize(x.ctx->st));
    for (int s = 0; s < 2; ++s) {
        UNO_HIP(k_fill(S, 0.0, b->P[s].p, st));
        UNO_HIP(k_fill(S, 0.0, b->G[s].p, st));
    }
    if (int rc = refresh_slots(b)) return rc;
    // X = U s^-1/2 (RHF.hpp:214-233): Jacobi of S, column scaling on the host read-back
    {
        UNO_HIP(hipMemcpyAsync(b->Tm[0].p, b->S.p, S * sizeof(double), hipMemcpyDeviceToDevice, st));
        UNO_HIP(batched_jacobi(b->nslot[0], b->slots.p, same(b->Tm[0]), same(b->V[0]), same(b->ev[0]), same(b->Z[0]), b->maxn,
                               50, st));
        std::vector<double> ev(S), Z(S);
        UNO_HIP(hipMemcpyAsync(ev.data(), b->ev[0].p, S * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipMemcpyAsync(Z.data(), b->Z[0].p, S * sizeof(double), hipMemcpyDeviceToHost, st));
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
        UNO_HIP(hipStreamSynchronize(st));   // Z is pageable
    }
    const Store X = same(b->X), Fp = both(b->Fp), Tm = both(b->Tm), Tm2 = both(b->Tm2), Z = both(b->Z), P = both(b->P),
                C = both(b->C);
    // F -> P over the slots of spins [0, ns): X^T F X, Jacobi, C = X W, P = C_occ C_occ^T.  Nothing here
    // waits for the device: the slots, the tiles and the stores are all the launches need.
    auto diag_to_P = [&](int ns, Store F) -> int {
        UNO_HIP(hipEventRecord(b->ev_diag[0], st));
        if (int rc = gemm(b, 0, ns, false, false, false, F, X, Tm)) return rc;
        if (int rc = gemm(b, 0, ns, true, false, false, X, Tm, Fp)) return rc;
        // after their first eigensolve the molecules start from their last eigenvectors Wp:
        // in that basis the matrix is nearly diagonal and the Jacobi sweeps settle in a few
        // rounds (W = Wp Z after; the first one's Z is W).  Spin 0 is warm when spin 1 is.
        const int nw = b->warm[1] ? ns : b->warm[0] ? 1 : 0;
        const Store Wp = both(b->Wp), Wn = both(b->Wn);
        if (nw) {
            if (int rc = gemm(b, 0, nw, false, false, false, Fp, Wp, Tm)) return rc;
            if (int rc = gemm(b, 0, nw, true, false, false, Wp, Tm, Tm2)) return rc;
        }
        Store A, E;
        for (int s = 0; s < 2; ++s) {
            A.s[s] = s < nw ? Tm2.s[s] : Fp.s[s];
            E.s[s] = s < nw ? Z.s[s] : Wn.s[s];
        }
        UNO_HIP(batched_jacobi(b->nslot[0] + (ns > 1 ? b->nslot[1] : 0), b->slots.p, A, both(b->V), both(b->ev), E, b->maxn, 50,
                               st));
        if (nw) {
            // (not for the core Hamiltonian, whose levels come out the same in every run)
            UNO_HIP(batch_ties(b->nslot[0] + (ns > 1 ? b->nslot[1] : 0), b->slots.p, both(b->ev), E, st));
            if (int rc = gemm(b, 0, nw, false, false, false, Wp, Z, Wn)) return rc;
        }
        for (int s = 0; s < ns; ++s) {
            std::swap(b->Wp[s], b->Wn[s]);
            b->warm[s] = true;
        }
        if (int rc = gemm(b, 0, ns, false, false, false, X, Wn, C)) return rc;
        if (int rc = gemm(b, 0, ns, false, true, true, C, C, P)) return rc;
        UNO_HIP(hipEventRecord(b->ev_diag[1], st));
        return UNO_OK;
    };
    // core-Hamiltonian guess (UHF beta reuses the alpha orbitals, UHF.hpp:206-215)
    if (int rc = diag_to_P(1, same(b->H))) return rc;
    if (int rc = gemm(b, 1, 2, false, true, true, same(b->C[0]), same(b->C[0]), P)) return rc;
    UNO_HIP(hipStreamSynchronize(st));
    double diag_s = elapsed(b->ev_diag);
    double eps = o.eps;
    int ndiis = 0, slot_next = 0;
    std::vector<double> Bm((size_t)nm * kBatchDiis * kBatchDiis, 0.0);
    static_assert(kBatchDiis <= kMaxLin && kBatchDiis + 4 <= kMaxDots, "one launch per combination and per row");
    LinSources hist;
    for (int j = 0; j < kBatchDiis; ++j)
        for (int s = 0; s < 2; ++s) hist.s[j][s] = b->dF[j][s].p;
    int iteration = 0;
    double fock_s = 0.0;
    int nstopped = 0;
    double wall99 = -1.0;
    // Two waits an iteration: for the energies and the DIIS row, whose coefficients the host solves
    // for, and for the density changes, which decide who stops.
    while (true) {
        const int n0 = b->nslot[0], n = n0 + b->nslot[1];
        UNO_HIP(hipEventRecord(b->ev_fock[0], st));
        UNO_HIP(batch_densities(S, P, b->D0.p, both(b->Pold), st));
        if (int rc = batch_fock(b)) return rc;
        UNO_HIP(batch_sym(n, b->slots.p, both(b->W), both(b->G), st));
        UNO_HIP(hipEventRecord(b->ev_fock[1], st));
        // F = H + G and its DIIS error X^T (FPS - SPF) X, FPS - SPF = FPS - (FPS)^T, on every active
        // slot (one shared history position per iteration)
        const int slot = slot_next;
        slot_next = (slot_next + 1) % kBatchDiis;
        if (ndiis < kBatchDiis) ++ndiis;
        const Store F = both(b->dF[slot]), E = both(b->dE[slot]);
        UNO_HIP(batch_add(n, b->slots.p, b->H.p, both(b->G), F, st));
        if (int rc = gemm(b, 0, 2, false, false, false, F, P, Tm)) return rc;
        if (int rc = gemm(b, 0, 2, false, false, false, Tm, same(b->S), Fp)) return rc;
        UNO_HIP(batch_antisym(n, b->slots.p, Fp, Tm2, st));
        if (int rc = gemm(b, 0, 2, false, false, false, Tm2, X, Tm)) return rc;
        if (int rc = gemm(b, 0, 2, true, false, false, X, Tm, E)) return rc;
        // energies: e1 = tr(Pa H) + tr(Pb H), e2 = tr(Pa Ga) + tr(Pb Gb), from the slots of spin 0; and
        // the B-matrix row of the new error: sum over spins of <E_new, E_j>
        DotPairs q{};
        q.add(P.s[0], nullptr, b->H.p, nullptr);
        q.add(P.s[1], nullptr, b->H.p, nullptr);
        q.add(P.s[0], nullptr, b->G[0].p, nullptr);
        q.add(P.s[1], nullptr, b->G[1].p, nullptr);
        for (int j = 0; j < ndiis; ++j) q.add(E.s[0], E.s[1], b->dE[j][0].p, b->dE[j][1].p);
        UNO_HIP(batch_dots(n, b->slots.p, q, b->red.p, st));
        UNO_HIP(hipMemcpyAsync(b->h_dots, b->red.p, (size_t)q.n * n * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        fock_s += elapsed(b->ev_fock);
        auto dot = [&](int pair, int k) { return b->h_dots[(size_t)pair * n + k]; };
        std::vector<double> row((size_t)nm * kBatchDiis, 0.0);
        for (int k = 0; k < n; ++k)
            for (int j = 0; j < ndiis; ++j) row[(size_t)b->who[k] * kBatchDiis + j] += dot(4 + j, k);
        std::vector<int> first(nm, -1);   // a molecule's spin-0 slot
        for (int k = 0; k < n0; ++k) {
            const int m = b->who[k];
            BatchMol& x = b->mol[m];
            const double e1 = dot(0, k) + dot(1, k), e2 = dot(2, k) + dot(3, k);
            x.energy = x.uhf ? e1 + 0.5 * e2 : 2.0 * e1 + e2;
            x.ediff = x.energy - x.eold;
            x.eold = x.energy;
            if (iteration == 0) x.init_energy = x.energy + x.nuc;
            double* Bmm = &Bm[(size_t)m * kBatchDiis * kBatchDiis];
            for (int j = 0; j < ndiis; ++j) Bmm[slot * kBatchDiis + j] = Bmm[j * kBatchDiis + slot] = row[(size_t)m * kBatchDiis + j];
            double* ck = b->h_coef + (size_t)k * kMaxLin;
            std::fill(ck, ck + kMaxLin, 0.0);
            ck[slot] = 1.0;
            if (ndiis >= 2) diis_coefficients(Bmm, kBatchDiis, ndiis, slot, ck);
            first[m] = k;
        }
        for (int k = n0; k < n; ++k)
            std::copy_n(b->h_coef + (size_t)first[b->who[k]] * kMaxLin, kMaxLin, b->h_coef + (size_t)k * kMaxLin);
        UNO_HIP(hipMemcpyAsync(b->coef.p, b->h_coef, (size_t)n * kMaxLin * sizeof(double), hipMemcpyHostToDevice, st));
        UNO_HIP(batch_lincomb(n, b->slots.p, b->coef.p, hist, both(b->F), st));
        // new densities
        if (int rc = diag_to_P(2, both(b->F))) return rc;
        UNO_HIP(batch_diffnorm(n, b->slots.p, P, both(b->Pold), b->red.p, st));
        UNO_HIP(hipMemcpyAsync(b->h_pdiff, b->red.p, n * sizeof(double), hipMemcpyDeviceToHost, st));
        UNO_HIP(hipStreamSynchronize(st));
        diag_s += elapsed(b->ev_diag);
        ++iteration;
        bool changed = false;
        for (int k = 0; k < n; ++k) {
            BatchMol& x = b->mol[b->who[k]];
            x.pdiff = k < n0 ? b->h_pdiff[k] : x.pdiff + b->h_pdiff[k];
            x.iterations = iteration;
        }
        for (int k = 0; k < n0; ++k) {
            BatchMol& x = b->mol[b->who[k]];
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
            if (int rc = refresh_slots(b)) return rc;
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
