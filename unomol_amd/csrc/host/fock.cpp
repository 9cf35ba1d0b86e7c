// The direct Fock build: the kernels' pair data and quartet spaces (once per geometry), and the
// launches of a build.  A build's grids do not depend on the density: the kernels find the
// quartets that belong to it from the Schwarz bounds and the density maximum on the device
// (fock_core.hpp), so the host only enqueues one launch per class pair and precision.
#include <algorithm>
#include <array>
#include <climits>
#include <cstdint>
#include <cmath>
#include <mutex>
#include "engine.hpp"

namespace uno {

int LaunchStreams::prepare(int n) {
    for (int k = 0; k + 1 < n; ++k)
        if (!w[k]) {
            UNO_HIP(hipStreamCreate(&w[k]));
            UNO_HIP(hipEventCreateWithFlags(&join[k], hipEventDisableTiming));
        }
    if (n > 1 && !fork) UNO_HIP(hipEventCreateWithFlags(&fork, hipEventDisableTiming));
    return UNO_OK;
}
int LaunchStreams::begin(int n, hipStream_t st) {
    if (n <= 1) return UNO_OK;
    UNO_HIP(hipEventRecord(fork, st));
    for (int k = 0; k + 1 < n; ++k) UNO_HIP(hipStreamWaitEvent(w[k], fork, 0));
    return UNO_OK;
}
int LaunchStreams::end(int n, hipStream_t st) {
    for (int k = 0; k + 1 < n; ++k) {
        UNO_HIP(hipEventRecord(join[k], w[k]));
        UNO_HIP(hipStreamWaitEvent(st, join[k], 0));
    }
    return UNO_OK;
}
LaunchStreams::~LaunchStreams() {
    for (int k = 0; k + 1 < kMaxLaunchStreams; ++k) {
        if (w[k]) {
            (void)hipStreamSynchronize(w[k]);
            (void)hipStreamDestroy(w[k]);
        }
        if (join[k]) (void)hipEventDestroy(join[k]);
    }
    if (fork) (void)hipEventDestroy(fork);
}

// candidate tasks from which a build lists the live ones first (below, the list costs a launch and
// the blocks would find few dead ones)
constexpr long long kListFrom = 8192;

// lanes the chip holds at two waves per SIMD
constexpr double kChipLanes = 2 * 1024 * 64;

// log2 of the lanes that share a ket of kprim primitives against a bra of bprim, in a launch of
// about `prims` primitive quartets: doubled while the split costs next to nothing (the rounds over
// the ket's primitives stay nearly full, and each lane keeps primitive quartets enough that
// adding up the group's blocks does not show), or while one lane's loop over a quartet's
// primitives is longer than the launch could take with its work spread over the chip.  (A third
// of the candidates are taken to survive the screens.)
static int lanes_per_ket(int bprim, int kprim, double prims) {
    const double share = std::max(8.0, 0.3 * prims / kChipLanes);
    int lg = 0;
    while ((1 << lg) < kprim && lg < 6) {
        const int g = 2 << lg, rounds = (kprim + g - 1) / g, now = (kprim + (1 << lg) - 1) >> lg;
        const bool cheap = kprim >= 0.85 * rounds * g && bprim * rounds >= 16;
        if (!cheap && bprim * now <= share) break;
        ++lg;
    }
    return lg;
}

int FockStore::build(const std::vector<FockMol>& mols, const PairHdr* d_pairs, const PrimPair* d_prims, int np,
                     long long nprims, hipStream_t st) {
    static const int kPairL[kNumPairClasses][2] = {{0, 0}, {1, 0}, {1, 1}, {2, 0}, {2, 1}, {2, 2}};
    npair = np;
    njp = 0;
    // runs of the whole array, with their ket layout, and the LDS row columns: per molecule and
    // ket class the functions its pairs touch (whole shells), in function order
    struct Run {
        int off, count, maxprim, lcls;
        long long kp0, jo0;
    };
    std::vector<PairRun> pr;
    std::vector<std::vector<Run>> runs(mols.size());
    std::vector<int> colmap, cinv;
    std::vector<std::array<int, kNumPairClasses>> ncols(mols.size());
    std::vector<int> colbase(mols.size());
    kps = 0;
    for (size_t m = 0; m < mols.size(); ++m) {
        const FockMol& x = mols[m];
        const int base = (int)colmap.size();
        colbase[m] = base;
        colmap.resize(base + (size_t)kNumPairClasses * x.n, -1);
        cinv.resize(colmap.size(), 0);
        std::vector<char> used((size_t)kNumPairClasses * x.n, 0);
        for (const PairClassList& L : *x.runs) {
            Run r{x.pair_off + L.off, L.count, 1, L.lcls, kps, njp};
            const int n1 = ncart(kPairL[L.lcls][0]), n2 = ncart(kPairL[L.lcls][1]);
            char* u = used.data() + (size_t)L.lcls * x.n;
            for (int k = L.off; k < L.off + L.count; ++k) {
                const PairHdr& h = x.pairs[k];
                r.maxprim = std::max(r.maxprim, h.nprim);
                for (int f = 0; f < n1; ++f) u[h.f1 + f] = 1;
                for (int f = 0; f < n2; ++f) u[h.f2 + f] = 1;
            }
            njp += (long long)pair_comps(L.lcls) * L.count;
            kps += (long long)r.maxprim * L.count;
            runs[m].push_back(r);
            pr.push_back(PairRun{r.off, r.count, base + L.lcls * x.n, L.lcls, r.kp0, r.jo0});
        }
        for (int c = 0; c < kNumPairClasses; ++c) {
            int k = 0;
            for (int f = 0; f < x.n; ++f)
                if (used[(size_t)c * x.n + f]) {
                    colmap[base + (size_t)c * x.n + f] = k;
                    cinv[base + (size_t)c * x.n + k] = f;
                    ++k;
                }
            ncols[m][c] = k;
        }
    }
    if (njp > (long long)INT32_MAX) {
        set_error("too many shell pairs for 32-bit offsets");
        return UNO_EINVAL;
    }
    // the launches: per launch group and class pair the spaces of every molecule, the ones with
    // the longest primitive loops first
    launches.clear();
    nspaces = 0;
    std::vector<char> host;
    auto put = [&](const void* p, size_t bytes) {
        const size_t off = (host.size() + 15) / 16 * 16;
        host.resize(off + bytes);
        std::copy((const char*)p, (const char*)p + bytes, host.begin() + off);
        return off;
    };
    for (int g = 0; g < 2; ++g)
        for (int cx = kNumPairClasses - 1; cx >= 0; --cx)
            for (int cy = cx; cy >= 0; --cy) {
                struct Cand {
                    FockSpace s;
                    int bprim, kprim;
                };
                std::vector<Cand> cs;
                double total = 0.0, prims = 0.0;
                FockLaunch L{cx, cy, g, 0, 1, 0, 0, 0, {0, 0}};
                for (size_t m = 0; m < mols.size(); ++m) {
                    if (mols[m].group != g) continue;
                    for (size_t X = 0; X < runs[m].size(); ++X)
                        for (size_t Y = 0; Y <= X; ++Y) {
                            const Run& b = runs[m][X];
                            const Run& k = runs[m][Y];
                            if (b.lcls != cx || k.lcls != cy) continue;
                            FockSpace s{};
                            s.bra_off = b.off;
                            s.nbra = b.count;
                            s.ket_off = k.off;
                            s.nket = k.count;
                            s.same = X == Y;
                            s.mol = mols[m].mol;
                            s.col0 = colbase[m] + cy * mols[m].n;
                            s.ncols = ncols[m][cy];
                            s.kstride = k.count;
                            s.kp0 = k.kp0;
                            s.jo0 = k.jo0;
                            cs.push_back(Cand{s, b.maxprim, k.maxprim});
                            const double nq = (s.same ? 0.5 : 1.0) * s.nbra * (double)s.nket;
                            total += nq;
                            prims += nq * b.maxprim * k.maxprim;
                            L.ncols = std::max(L.ncols, s.ncols);
                            L.nket = std::max(L.nket, s.nket);
                        }
                }
                if (cs.empty()) continue;
                std::stable_sort(cs.begin(), cs.end(), [](const Cand& u, const Cand& v) { return (long)u.bprim * u.kprim > (long)v.bprim * v.kprim; });
                std::vector<FockSpace> sp;
                long long nb = 0;
                // segments as long as leaves about 8192 passes' worth of blocks to balance the
                // launch (and their number within a grid): each block ends by adding its rows to
                // W, an atomic per row and column, which at 1024 kets a block was as many as the
                // kets' own (64 waters, one stream: 93.5 ms at up to 4 passes, 75.0 at up to 32;
                // (ds|ss) 11.2 -> 6.6, (ss|ss) 10.1 -> 6.1)
                for (int longer = 1;; longer *= 2) {
                    sp.clear();
                    nb = 0;
                    for (const Cand& c : cs) {
                        FockSpace s = c.s;
                        if (fock_is_wave(cx, cy)) {
                            s.seg = longer * (int)std::max(1.0, std::min<double>(kWaveSeg, total / 4096.0));
                        } else {
                            s.lg = lanes_per_ket(c.bprim, c.kprim, prims);
                            const int pass = kLaneBlock >> s.lg;
                            s.seg = longer * pass * (int)std::max(1.0, std::min(32.0, total / (pass * 8192.0)));
                        }
                        s.nseg = (s.nket + s.seg - 1) / s.seg;
                        s.first = (int)std::min<long long>(nb, INT32_MAX);
                        nb += (long long)s.nseg * s.nbra;
                        sp.push_back(s);
                    }
                    if (nb < (1LL << 30) && !(fock_is_wave(cx, cy) && longer * kWaveSeg > 64)) break;
                    if (longer > (1 << 20)) {
                        set_error("quartet space too large for one launch");
                        return UNO_EINVAL;
                    }
                }
                L.ncand = (int)nb;
                std::vector<int> blk;
                int k = 0;
                for (long long b = 0; b <= nb + 63; b += 64) {
                    while (k + 1 < (int)sp.size() && sp[k + 1].first <= b) ++k;
                    blk.push_back(k);
                }
                L.sp = put(sp.data(), sp.size() * sizeof(FockSpace));
                nspaces += (int)sp.size();
                L.blk = put(blk.data(), blk.size() * sizeof(int));
                launches.push_back(L);
            }
    // the task lists' sources: counter and list of launch k and precision p (2 k + p in a mixed
    // build, k otherwise)
    long long total = 0;
    for (FockLaunch& l : launches)
        for (int p = 0; p < 2; ++p) {
            l.list[p] = (int)std::min<long long>(total, INT32_MAX);
            total += l.ncand;
        }
    listed = total > 2 * kListFrom && total <= (long long)INT32_MAX;
    std::vector<FockTaskSource> hsrc[2];
    if (listed) {
        for (int m = 0; m < 2; ++m) {
            int nb = 0;
            for (const FockLaunch& l : launches)
                for (int p = 0; p <= m; ++p) {
                    hsrc[m].push_back(FockTaskSource{(long long)l.sp, (long long)l.blk, nb, l.ncand, l.list[p], p});
                    nb += (l.ncand + kTaskThreads - 1) / kTaskThreads;
                }
            nsrc[m] = (int)hsrc[m].size();
            src_blocks[m] = nb;
            UNO_HIP(src[m].upload(hsrc[m].data(), hsrc[m].size(), st));
        }
        UNO_HIP(lists.alloc((size_t)total));
    }
    UNO_HIP(ctr.alloc(2 * launches.size()));
    DBuf<PairRun> dr;
    DBuf<int> dcm;
    UNO_HIP(dr.upload(pr.data(), pr.size(), st));
    UNO_HIP(dcm.upload(colmap.data(), colmap.size(), st));
    UNO_HIP(colinv.upload(cinv.data(), cinv.size(), st));
    UNO_HIP(tables.upload(host.data(), host.size(), st));
    UNO_HIP(bprim.alloc((size_t)std::max(nprims, 1LL)));
    UNO_HIP(kprim.alloc((size_t)std::max(kKetFields * kps, 1LL)));
    UNO_HIP(kgeo.alloc(6 * (size_t)std::max(np, 1)));
    UNO_HIP(kidx.alloc(np));
    UNO_HIP(kjo.alloc(np));
    UNO_HIP(knp.alloc(np));
    UNO_HIP(kcol.alloc(np));
    UNO_HIP(dpair.alloc(np));
    UNO_HIP(dp.alloc((size_t)std::max(njp, 1LL)));
    UNO_HIP(jp.alloc((size_t)std::max(njp, 1LL)));
    UNO_HIP(dmax.alloc(mols.size()));
    UNO_HIP(nquart.alloc(3 * kQuartSlots));
    UNO_HIP(pair_store(np, (int)pr.size(), dr.p, d_pairs, d_prims, dcm.p, bprim.p, kprim.p, kps, kgeo.p, kidx.p, kjo.p,
                       knp.p, kcol.p, st));
    UNO_HIP(hipStreamSynchronize(st));   // the host tables and the scratch buffers go
    return UNO_OK;
}

FockArgs FockStore::args(int k, int prec, bool mixed, const PairHdr* d_pairs, const PrimPair* d_prims,
                         const double* pairQ) const {
    const FockLaunch& l = launches[k];
    FockArgs a{};
    a.sp = reinterpret_cast<const FockSpace*>(tables.p + l.sp);
    a.blk = reinterpret_cast<const int*>(tables.p + l.blk);
    a.list = listed ? lists.p + l.list[prec] : nullptr;
    a.ctr = ctr.p + (mixed ? 2 * k + prec : k);
    a.ncand = l.ncand;
    a.pairs = d_pairs;
    a.prims = d_prims;
    a.bprim = bprim.p;
    a.kprim = kprim.p;
    a.kps = kps;
    a.kgeo = kgeo.p;
    a.npair = npair;
    a.kidx = kidx.p;
    a.knp = knp.p;
    a.kcol = kcol.p;
    a.colinv = colinv.p;
    a.pairQ = pairQ;
    a.dpair = dpair.p;
    a.dp = dp.p;
    a.dmax = dmax.p;
    return a;
}

int FockStore::list_tasks(bool mixed, const FockArgs& a, hipStream_t st) const {
    const int m = mixed ? 1 : 0;
    if (listed) UNO_HIP(fock_tasks(nsrc[m], src[m].p, src_blocks[m], tables.p, a, ctr.p, lists.p, st));
    return UNO_OK;
}

// tuned configurations, shared by every context of the same layout in this process: basis size,
// shells, pairs and the runs' classes and primitive buckets (two contractions of the same shells
// differ in those alone)
static std::map<std::vector<int>, std::map<std::tuple<int, int, int, int>, FockConfig>> g_tuning;
static std::mutex g_tuning_mutex;

static std::vector<int> tuning_key(const uno_ctx* c) {
    std::vector<int> key{c->n, c->nsh, (int)c->pairs.size()};
    for (const PairClassList& L : c->cls) key.push_back(L.lcls * kNumBuckets + L.bucket);
    return key;
}

void remember_tuning(uno_ctx* c) {
    const std::lock_guard<std::mutex> lock(g_tuning_mutex);
    auto& m = g_tuning[tuning_key(c)];
    for (const auto& kv : c->tune) m[kv.first] = kv.second;
}

void recall_tuning(uno_ctx* c) {
    const std::lock_guard<std::mutex> lock(g_tuning_mutex);
    auto it = g_tuning.find(tuning_key(c));
    c->tune.clear();
    if (it != g_tuning.end()) c->tune = it->second;
}

int fock_build(uno_ctx* c, bool uhf, bool mixed) {
    hipStream_t st = c->st;
    FockStore& fs = c->fs;
    const long nn = (long)c->n * c->n;
    // deterministic builds: W holds two int64 words per entry (the second nn entries on), no
    // LDS rows, and the kets' Coulomb outputs go straight to W
    const bool det = c->deterministic != 0;
    const bool rows_on = c->row_merge && !det;
    const long wlen = det ? 2 * nn : nn;
    if (det) {
        UNO_HIP(c->W0.alloc(wlen));
        UNO_HIP(c->W1.alloc(wlen));
    }
    ClearList cl;
    cl.add(c->W0.p, wlen);
    if (uhf) cl.add(c->W1.p, wlen);
    cl.add(fs.jp.p, fs.njp);
    cl.add(fs.nquart.p, 2 * kQuartSlots);
    cl.add(fs.dmax.p, 1);
    cl.add(fs.ctr.p, 2 * (long long)fs.launches.size());
    UNO_HIP(fock_clear(cl, st));
    // shell-block density maxima for the screen, the largest of them, and the densities in the
    // pairs' order
    UNO_HIP(k_shell_max(c->n, c->nsh, c->d_shoff.p, c->d_shn.p, c->D0.p, uhf ? c->D1.p : nullptr,
                        uhf ? c->D2.p : nullptr, c->Dsh.p, fs.dmax.p, st));
    UNO_HIP(pair_density(fs.npair, fs.kidx.p, fs.kjo.p, c->D0.p, c->Dsh.p, c->n, c->nsh, nullptr, nullptr, fs.dp.p,
                         fs.dpair.p, st));
    if (!fs.launches.empty()) {
        FockArgs a = fs.args(0, 0, mixed, c->d_pairs.p, c->d_prims.p, c->d_pairQ.p);
        a.tau = c->tau;
        a.fp32_thr = mixed ? c->fp32_thr : 0.0;
        if (int rc = fs.list_tasks(mixed, a, st)) return rc;
    }
    const int mode = uhf ? kDigestUHF : kDigestRHF;
    // (the tuner times each launch on the context's stream)
    const int nls = c->tuning ? 1 : std::max(1, std::min(kMaxLaunchStreams, c->launch_streams));
    if (int rc = c->ls.prepare(nls)) return rc;
    if (int rc = c->ls.begin(nls, st)) return rc;
    int nlaunch = 0;
    for (int k = 0; k < (int)fs.launches.size(); ++k)
        for (int prec = 0; prec < (mixed ? 2 : 1); ++prec) {
            const FockLaunch& l = fs.launches[k];
            FockArgs a = fs.args(k, prec, mixed, c->d_pairs.p, c->d_prims.p, c->d_pairQ.p);
            a.tau = c->tau;
            a.primcut = c->primcut;
            a.fp32_thr = mixed ? c->fp32_thr : 0.0;
            a.rys2_exact = c->rys2_exact;
            a.n = c->n;
            a.nsh = c->nsh;
            a.dsh = c->Dsh.p;
            a.jp = det ? nullptr : fs.jp.p;
            a.fix_lo = det ? nn : 0;
            a.nquart = fs.nquart.p + prec * kQuartSlots;
            a.D0 = c->D0.p;
            a.W0 = c->W0.p;
            if (uhf) {
                a.D1 = c->D1.p;
                a.D2 = c->D2.p;
                a.W1 = c->W1.p;
            }
            const bool wave = fock_is_wave(l.cx, l.cy);
            const bool rows = rows_on && l.nket >= c->row_min_kets;
            FockConfig f = fock_default(l.cx, l.cy, mode, l.ncols, c->nsh, prec == 1, rows, c->row_variant, c->row_dens);
            const auto key = std::make_tuple(kNumPairClasses * l.cx + l.cy, prec, uhf ? 1 : 0, mixed ? 1 : 0);
            // (a layout that the caller forces, and that fits, goes before the tuned one)
            if (rows && !c->tuning && !(c->row_variant && f.variant == c->row_variant)) {
                auto it = c->tune.find(key);
                if (it != c->tune.end()) {
                    auto fits = [&](const FockConfig& g) { return fock_config_fits(l.cx, l.cy, g, mode, l.ncols, c->nsh, prec == 1); };
                    FockConfig g = it->second;
                    if (c->row_dens == 0) g.dlds = 0;
                    if (fits(g)) f = g;
                    g.dlds = 1;
                    if (c->row_dens > 0 && g.variant && fits(g)) f = g;
                }
            }
            const int ci = prec * kNumPairClasses * kNumPairClasses + l.cx * kNumPairClasses + l.cy;
            auto launch = [&](const FockConfig& g, hipStream_t s) {
                return fock_launch(mode, prec == 1, l.cx, l.cy, a, g, l.ncols, s);
            };
            if (c->tuning && rows && !wave) {
                // time every candidate (each one run three times, the fastest counts)
                float best_ms = 1e30f;
                FockConfig best = f;
                hipEvent_t t0, t1;
                UNO_HIP(hipEventCreate(&t0));
                UNO_HIP(hipEventCreate(&t1));
                unsigned long long* const counted = a.nquart;
                a.nquart = fs.nquart.p + 2 * kQuartSlots;   // the candidates' counts go nowhere
                for (int v = 0; v < 16; ++v) {
                    FockConfig g;
                    g.variant = v & 3;
                    g.dlds = (v >> 2) & 1;
                    g.mlds = (v >> 3) & 1;
                    if (g.dlds && (!g.variant || c->row_dens == 0)) continue;
                    if (!fock_config_fits(l.cx, l.cy, g, mode, l.ncols, c->nsh, prec == 1)) continue;
                    float ms_min = 1e30f;
                    for (int rep = 0; rep < 3; ++rep) {
                        // the tasks from the first one again
                        UNO_HIP(hipMemsetAsync(&a.ctr->head, 0, sizeof(int), st));
                        UNO_HIP(hipEventRecord(t0, st));
                        UNO_HIP(launch(g, st));
                        UNO_HIP(hipEventRecord(t1, st));
                        UNO_HIP(hipEventSynchronize(t1));
                        float ms = 0.f;
                        UNO_HIP(hipEventElapsedTime(&ms, t0, t1));
                        ms_min = std::min(ms_min, ms);
                    }
                    if (ms_min < best_ms) {
                        best_ms = ms_min;
                        best = g;
                    }
                }
                (void)hipEventDestroy(t0);
                (void)hipEventDestroy(t1);
                // once more with the chosen one, which counts
                a.nquart = counted;
                UNO_HIP(hipMemsetAsync(&a.ctr->head, 0, sizeof(int), st));
                UNO_HIP(launch(best, st));
                c->tune[key] = best;
                c->tune_ms += best_ms;
                continue;
            }
            const int slot = f.variant * 2 * kNumPairClasses * kNumPairClasses + ci;
            const bool prof = c->profile && !c->tuning && c->d_counter.p;
            const hipStream_t ls = c->ls.of(nlaunch++ % nls, st);
            hipEvent_t e1 = nullptr;
            if (prof) {
                a.counter = c->d_counter.p + 2 * kCounterSlots * slot;
                const size_t pe = c->prof_pending++;
                while (c->prof_ev.size() < 2 * (pe + 1)) {
                    hipEvent_t e = nullptr;
                    UNO_HIP(hipEventCreate(&e));
                    c->prof_ev.push_back(e);
                }
                if (c->prof_evslot.size() < pe + 1) c->prof_evslot.resize(pe + 1);
                c->prof_evslot[pe] = slot;
                e1 = c->prof_ev[2 * pe + 1];
                UNO_HIP(hipEventRecord(c->prof_ev[2 * pe], ls));
            }
            UNO_HIP(launch(f, ls));
            if (prof) UNO_HIP(hipEventRecord(e1, ls));
        }
    // the context's stream continues once every worker's launches are done
    if (int rc = c->ls.end(nls, st)) return rc;
    if (det) {
        UNO_HIP(fixed_to_f64(nn, c->W0.p, nn, st));
        if (uhf) UNO_HIP(fixed_to_f64(nn, c->W1.p, nn, st));
    } else {
        // the kets' Coulomb outputs, accumulated per pair, into W
        UNO_HIP(jp_scatter(fs.npair, fs.kidx.p, fs.kjo.p, fs.jp.p, c->W0.p, uhf ? c->W1.p : nullptr, c->n, nullptr,
                           nullptr, st));
    }
    c->quartets_known = false;
    return UNO_OK;
}

int fock_quartets(uno_ctx* c) {
    if (c->quartets_known) return UNO_OK;
    unsigned long long h[2 * kQuartSlots];
    UNO_HIP(hipMemcpyAsync(h, c->fs.nquart.p, sizeof(h), hipMemcpyDeviceToHost, c->st));
    UNO_HIP(hipStreamSynchronize(c->st));
    double q[2] = {0.0, 0.0};
    for (int k = 0; k < 2 * kQuartSlots; ++k) q[k / kQuartSlots] += (double)h[k];
    c->last_quartets = q[0] + q[1];
    c->last_quartets32 = q[1];
    c->quartets_known = true;
    return UNO_OK;
}

int profile_reset(uno_ctx* c, bool enable) {
    for (int i = 0; i < kProfSlots; ++i) c->prof_ms[i] = c->prof_launch[i] = c->prof_prim[i] = c->prof_shell[i] = 0.0;
    c->prof_pending = 0;   // pairs of earlier builds are dropped (their events are re-recorded)
    if (enable) {
        // the counters accumulate on the device from here until the next reset
        UNO_HIP(c->d_counter.alloc(2 * kCounterSlots * kProfSlots));
        // (all-zero bits: a fill of 0.0 clears the 64-bit counters)
        UNO_HIP(k_fill(2 * kCounterSlots * kProfSlots, 0.0, reinterpret_cast<double*>(c->d_counter.p), c->st));
    }
    return UNO_OK;
}

int profile_collect(uno_ctx* c) {
    if (!c->d_counter.p) return UNO_OK;
    UNO_HIP(hipStreamSynchronize(c->st));
    for (size_t k = 0; k < c->prof_pending; ++k) {
        float ms = 0.f;
        UNO_HIP(hipEventElapsedTime(&ms, c->prof_ev[2 * k], c->prof_ev[2 * k + 1]));
        c->prof_ms[c->prof_evslot[k]] += ms;
        c->prof_launch[c->prof_evslot[k]] += 1.0;
    }
    c->prof_pending = 0;
    std::vector<unsigned long long> cnt(2 * kCounterSlots * kProfSlots);
    UNO_HIP(hipMemcpy(cnt.data(), c->d_counter.p, cnt.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost));
    // device totals since the last reset
    for (int ci = 0; ci < kProfSlots; ++ci) {
        double pr = 0.0, sh = 0.0;
        for (int sl = 0; sl < kCounterSlots; ++sl) {
            pr += (double)cnt[2 * (kCounterSlots * ci + sl)];
            sh += (double)cnt[2 * (kCounterSlots * ci + sl) + 1];
        }
        c->prof_prim[ci] = pr;
        c->prof_shell[ci] = sh;
    }
    return UNO_OK;
}

}  // namespace uno
