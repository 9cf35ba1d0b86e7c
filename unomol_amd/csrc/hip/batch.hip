// Dense kernels of the batched SCF: many small molecules (N <= 256 functions each) whose
// matrices live back to back in one store, row-major N_m x N_m at offset off[m].
//
// A launch takes the slots (molecule, spin) of both spins: everything an iteration launches is
// described by one list of slots and one of their tiles, which change when a molecule stops.
//
//  * grouped GEMM: C_m = op(A_m) op(B_m) for every slot, one 32 x 32 output tile per
//    256-thread block (2 x 2 outputs per thread, K through LDS in steps of 32);
//  * batched Jacobi eigensolver: one block per molecule, cyclic sweeps in parallel
//    (round-robin) order, each round applying N/2 disjoint rotations to rows, then
//    columns, then the eigenvector columns; eigenvalues ascending with their vectors;
//  * per-molecule reductions (trace products, difference norms) and helpers.
#include <hip/hip_runtime.h>
#include <algorithm>
#include "batch_kernels.hpp"

namespace uno {

// ---------------------------------------------------------------------------
// grouped GEMM
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_grouped_gemm(const GemmTile* __restrict__ tiles, const MatSlot* __restrict__ slots,
                                                      int ta, int tb, int occ, Store As, Store Bs, Store Cs) {
    __shared__ double sA[32][33];
    __shared__ double sB[32][33];
    const GemmTile t = tiles[blockIdx.x];
    const MatSlot m = slots[t.slot];
    const int n = m.n, kn = occ ? m.nocc : n;
    const double* A = As.s[m.spin] + m.off;
    const double* B = Bs.s[m.spin] + m.off;
    double* C = Cs.s[m.spin] + m.off;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;   // 16 x 16 threads, 2 x 2 outputs each
    const int i0 = t.ti * 32, j0 = t.tj * 32;
    double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
    for (int k0 = 0; k0 < kn; k0 += 32) {
        for (int e = threadIdx.x; e < 32 * 32; e += 256) {
            const int r = e >> 5, c = e & 31;
            // op(A)[i][k], i = i0 + r, k = k0 + c
            const int i = i0 + r, k = k0 + c;
            double av = 0.0;
            if (i < n && k < kn) av = ta ? A[k * n + i] : A[i * n + k];
            sA[r][c] = av;
            // op(B)[k][j], k = k0 + r, j = j0 + c
            const int kk = k0 + r, j = j0 + c;
            double bv = 0.0;
            if (kk < kn && j < n) bv = tb ? B[j * n + kk] : B[kk * n + j];
            sB[r][c] = bv;
        }
        __syncthreads();
#pragma unroll 8
        for (int k = 0; k < 32; ++k) {
            const double a0 = sA[ty * 2][k], a1 = sA[ty * 2 + 1][k];
            const double b0 = sB[k][tx * 2], b1 = sB[k][tx * 2 + 1];
            acc[0][0] = fma(a0, b0, acc[0][0]);
            acc[0][1] = fma(a0, b1, acc[0][1]);
            acc[1][0] = fma(a1, b0, acc[1][0]);
            acc[1][1] = fma(a1, b1, acc[1][1]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int i = i0 + ty * 2 + a, j = j0 + tx * 2 + b;
            if (i < n && j < n) C[i * n + j] = acc[a][b];
        }
}

hipError_t grouped_gemm(int ntiles, const GemmTile* tiles, const MatSlot* slots, bool ta, bool tb, bool occ, Store A, Store B,
                        Store C, hipStream_t st) {
    if (ntiles <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_grouped_gemm, dim3(ntiles), dim3(256), 0, st, tiles, slots, ta ? 1 : 0, tb ? 1 : 0, occ ? 1 : 0, A, B, C);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// batched Jacobi: A (destroyed) -> eigenvalues ascending, eigenvectors in the columns of Z
// ---------------------------------------------------------------------------
// Cyclic Jacobi in round-robin order: with m = N rounded up to even (a dummy index N when N
// is odd), round r pairs (m-1, r) and ((r+k) mod (m-1), (r-k) mod (m-1)), k = 1..m/2-1, so
// that each round is a perfect matching and m-1 rounds visit every pair once.  A rotation
// is skipped when |a_pq| <= max(eps/2 sqrt(|a_pp a_qq|), 1e-15 ||A||_F) (it would not change
// the diagonal, or the pair is converged to working accuracy of the whole matrix: the
// relative test alone never settles next to zero diagonal entries, where rounding keeps
// a_pq above it); sweeps stop when none is applied.
constexpr int kJacobiThreads = 1024;
// a rotation of (x, y); the roundings are spelled out because the vectors inside an exactly
// degenerate level follow them, and both kernels have to pick the same
__device__ __forceinline__ double turn_p(double c, double s, double x, double y) { return fma(c, x, -(s * y)); }
__device__ __forceinline__ double turn_q(double c, double s, double x, double y) { return fma(s, x, c * y); }
constexpr int kJacobiLdsN = 140;   // largest matrix of the LDS kernel below
__global__ __launch_bounds__(kJacobiThreads) void k_batched_jacobi(const MatSlot* __restrict__ slots, Store As, Store Vs,
                                                                   Store evals, Store Zs, int max_sweeps) {
    __shared__ double cs[128], sn[128];
    __shared__ int pp[128], qq[128];
    __shared__ int nrot;
    __shared__ double red[kJacobiThreads / 64];
    const MatSlot M = slots[blockIdx.x];
    const int n = M.n;
    if (n <= kJacobiLdsN) return;   // the LDS kernel's
    double* A = As.s[M.spin] + M.off;
    double* V = Vs.s[M.spin] + M.off;
    double* ev = evals.s[M.spin] + M.off;
    double* Z = Zs.s[M.spin] + M.off;
    const int tid = threadIdx.x;
    double f2 = 0.0;
    for (long e = tid; e < (long)n * n; e += blockDim.x) {
        V[e] = (e / n == e % n) ? 1.0 : 0.0;
        f2 = fma(A[e], A[e], f2);
    }
    for (int o = 32; o >= 1; o >>= 1) f2 += __shfl_xor(f2, o, 64);
    if ((tid & 63) == 0) red[tid >> 6] = f2;
    __syncthreads();
    double fro2 = 0.0;
    for (int w = 0; w < kJacobiThreads / 64; ++w) fro2 += red[w];
    const double abs_tol = 1e-15 * sqrt(fro2);
    const int m = n + (n & 1);
    int sweep = 0;
    while (sweep < max_sweeps && n > 1) {
        ++sweep;
        if (tid == 0) nrot = 0;
        __syncthreads();
        for (int r = 0; r < m - 1; ++r) {
            for (int k = tid; k < m / 2; k += blockDim.x) {
                int a, b;
                if (k == 0) { a = m - 1; b = r; }
                else { a = (r + k) % (m - 1); b = (r - k + (m - 1)) % (m - 1); }
                const int p = a < b ? a : b, q = a < b ? b : a;
                double c = 1.0, s = 0.0;
                if (q < n) {
                    const double apq = A[(long)p * n + q];
                    const double app = A[(long)p * n + p], aqq = A[(long)q * n + q];
                    if (fabs(apq) > fmax(1.1102230246251565e-16 * sqrt(fabs(app * aqq)), abs_tol)) {
                        const double theta = (aqq - app) / (2.0 * apq);
                        const double t = fabs(theta) < 1e150
                                             ? (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0))
                                             : 0.5 / theta;
                        c = 1.0 / sqrt(t * t + 1.0);
                        s = t * c;
                        atomicAdd(&nrot, 1);
                    }
                }
                pp[k] = p;
                qq[k] = q;
                cs[k] = c;
                sn[k] = s;
            }
            __syncthreads();
            // rows p, q of A: A <- J^T A
            for (long e = tid; e < (long)(m / 2) * n; e += blockDim.x) {
                const int k = (int)(e / n), j = (int)(e % n);
                const int p = pp[k], q = qq[k];
                if (q >= n || sn[k] == 0.0) continue;
                const double c = cs[k], s = sn[k];
                const double ap = A[(long)p * n + j], aq = A[(long)q * n + j];
                A[(long)p * n + j] = turn_p(c, s, ap, aq);
                A[(long)q * n + j] = turn_q(c, s, ap, aq);
            }
            __syncthreads();
            // columns p, q of A and of V: A <- A J, V <- V J
            for (long e = tid; e < (long)(m / 2) * n; e += blockDim.x) {
                const int k = (int)(e / n), i = (int)(e % n);
                const int p = pp[k], q = qq[k];
                if (q >= n || sn[k] == 0.0) continue;
                const double c = cs[k], s = sn[k];
                const double ap = A[(long)i * n + p], aq = A[(long)i * n + q];
                A[(long)i * n + p] = turn_p(c, s, ap, aq);
                A[(long)i * n + q] = turn_q(c, s, ap, aq);
                const double vp = V[(long)i * n + p], vq = V[(long)i * n + q];
                V[(long)i * n + p] = turn_p(c, s, vp, vq);
                V[(long)i * n + q] = turn_q(c, s, vp, vq);
            }
            __syncthreads();
        }
        const int done = nrot == 0;
        __syncthreads();
        if (done) break;
    }
    __syncthreads();
    // eigenvalues ascending (ties by index) with their vectors as columns of Z
    for (int i = tid; i < n; i += blockDim.x) {
        const double di = A[(long)i * n + i];
        int rank = 0;
        for (int j = 0; j < n; ++j) {
            const double dj = A[(long)j * n + j];
            if (dj < di || (dj == di && j < i)) ++rank;
        }
        ev[rank] = di;
        for (int r = 0; r < n; ++r) Z[(long)r * n + rank] = V[(long)r * n + i];
    }
}

// The same rotations in the same order with the matrix in LDS, for n <= kJacobiLdsN (158 KB of the
// 160 at 140 functions), in the other kernel's arithmetic, so that the vectors it picks inside an
// exactly degenerate level (a linear molecule's pi pairs) are the same.  A round is one pass over
// the matrix, which applies the rotations to both sides of every 2 x 2 block of the pairs (k, l),
// rows first, and one phase in which two waves compute the next round's rotations (a chain of
// divides and square roots) while the others turn the eigenvectors.  These are kept
// transposed (the two vectors of a rotation are rows), in LDS as well while both fit, else in V.
// Bound by latency: a wave reads what all its blocks need before it uses any of it, and a round
// without rotations costs the test alone.  32 molecules of up to 114 functions, mean launch of an SCF
// (most of them warm): 5.7 ms with the matrix in global memory, 1.35 here.
// LDS of a matrix: padded to an even size with zeros (the dummy index of an odd n then needs no
// exceptions), odd row strides so that columns fall on different banks
__host__ __device__ constexpr int jacobi_a(int n) { return (n + (n & 1)) * (n + (n & 1) + 1); }
__host__ __device__ constexpr int jacobi_v(int n) { return n * (n | 1); }
constexpr int kJacobiLds = 19904;   // doubles a block may take (99 functions with their vectors: 19901)
static_assert(jacobi_a(kJacobiLdsN) <= kJacobiLds, "the largest matrix fits");
__host__ __device__ constexpr bool jacobi_v_fits(int n) { return jacobi_a(n) + jacobi_v(n) <= kJacobiLds; }
__global__ __launch_bounds__(kJacobiThreads) void k_batched_jacobi_lds(const MatSlot* __restrict__ slots, Store As, Store Vs,
                                                                       Store evals, Store Zs, int max_sweeps) {
    constexpr int kPairs = kJacobiLdsN / 2, kWaves = kJacobiThreads / 64;
    constexpr int kRotWaves = (kPairs + 63) / 64;                             // waves of the rotations
    constexpr int kPer = 3;                                                   // rows of blocks in flight
    constexpr int kVPer = 5;                                                  // pairs of vectors in flight
    extern __shared__ double lds[];
    // rotations of this round and the next: (c, s), the pair, and how many there are
    __shared__ double2 rot[2][kPairs];
    __shared__ int2 pq[2][kPairs];
    __shared__ int nrot[2];
    __shared__ double red[kWaves];
    const MatSlot M = slots[blockIdx.x];
    const int n = M.n;
    if (n > kJacobiLdsN) return;   // the other kernel's
    const int m = n + (n & 1), mk = m / 2, ld = m + 1, lv = n | 1;
    const double* A0 = As.s[M.spin] + M.off;
    double* ev = evals.s[M.spin] + M.off;
    double* Z = Zs.s[M.spin] + M.off;
    double* A = lds;
    // component i of vector p in V[p ldv + i], in one of two address spaces: the accesses name theirs
    const bool vl = jacobi_v_fits(n);
    typedef __attribute__((address_space(1))) double Global;
    double* const VL = lds + jacobi_a(n);
    Global* const VG = (Global*)(Vs.s[M.spin] + M.off);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    double f2 = 0.0;
    if (n & 1)
        for (int e = tid; e < m; e += kJacobiThreads) A[e * ld + n] = A[n * ld + e] = 0.0;
    for (int e = tid; e < n * n; e += kJacobiThreads) {
        const int i = e / n, j = e - i * n;
        const double v = A0[e];
        A[i * ld + j] = v;
        if (vl) VL[i * lv + j] = i == j ? 1.0 : 0.0;
        else VG[e] = i == j ? 1.0 : 0.0;
        f2 = fma(v, v, f2);
    }
    for (int o = 32; o >= 1; o >>= 1) f2 += __shfl_xor(f2, o, 64);
    if ((tid & 63) == 0) red[tid >> 6] = f2;
    if (tid < 2) nrot[tid] = 0;
    __syncthreads();
    double fro2 = 0.0;
    for (int w = 0; w < kWaves; ++w) fro2 += red[w];
    const double abs_tol = 1e-15 * sqrt(fro2);
    // the rotations of round r into buffer d
    auto rotations = [&](int r, int d) {
        double c = 1.0, s = 0.0;
        if (tid < mk) {
            int a, b;
            if (tid == 0) {
                a = m - 1;
                b = r;
            } else {
                a = r + tid;
                if (a >= m - 1) a -= m - 1;
                b = r - tid;
                if (b < 0) b += m - 1;
            }
            const int p = a < b ? a : b, q = a < b ? b : a;
            if (q < n) {
                const double apq = A[p * ld + q];
                const double app = A[p * ld + p], aqq = A[q * ld + q];
                if (fabs(apq) > fmax(1.1102230246251565e-16 * sqrt(fabs(app * aqq)), abs_tol)) {
                    const double theta = (aqq - app) / (2.0 * apq);
                    const double t = fabs(theta) < 1e150
                                         ? (theta >= 0.0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0))
                                         : 0.5 / theta;
                    c = 1.0 / sqrt(t * t + 1.0);
                    s = t * c;
                }
            }
            rot[d][tid] = make_double2(c, s);
            pq[d][tid] = make_int2(p, q);
        }
        const unsigned long long any = __ballot(s != 0.0);
        if (lane == 0 && any) atomicAdd(&nrot[d], 1);
    };
    // the rotations of buffer d applied to the eigenvectors by the other waves, kVPer of them in flight
    auto turn = [&](auto* V, int ldv, int d) {
        constexpr int kC = (kJacobiLdsN + 63) / 64;
        for (int k0 = wave - kRotWaves; k0 < mk; k0 += (kWaves - kRotWaves) * kVPer) {
            double2 rv[kVPer];
            int2 pv[kVPer];
            double x[kVPer][kC], y[kVPer][kC];
#pragma unroll
            for (int u = 0; u < kVPer; ++u) {
                const int k = k0 + (kWaves - kRotWaves) * u;
                rv[u] = rot[d][min(k, mk - 1)];
                pv[u] = pq[d][min(k, mk - 1)];
                if (k >= mk) rv[u].y = 0.0;
            }
#pragma unroll
            for (int u = 0; u < kVPer; ++u)
                if (rv[u].y != 0.0) {
                    const int vp = __builtin_amdgcn_readfirstlane(pv[u].x) * ldv, vq = __builtin_amdgcn_readfirstlane(pv[u].y) * ldv;
#pragma unroll
                    for (int c = 0; c < kC; ++c)
                        if (lane + 64 * c < n) {
                            x[u][c] = V[vp + lane + 64 * c];
                            y[u][c] = V[vq + lane + 64 * c];
                        }
                }
#pragma unroll
            for (int u = 0; u < kVPer; ++u)
                if (rv[u].y != 0.0) {
                    const int vp = __builtin_amdgcn_readfirstlane(pv[u].x) * ldv, vq = __builtin_amdgcn_readfirstlane(pv[u].y) * ldv;
                    const double c0 = rv[u].x, s0 = rv[u].y;
#pragma unroll
                    for (int c = 0; c < kC; ++c)
                        if (lane + 64 * c < n) {
                            V[vp + lane + 64 * c] = turn_p(c0, s0, x[u][c], y[u][c]);
                            V[vq + lane + 64 * c] = turn_q(c0, s0, x[u][c], y[u][c]);
                        }
                }
        }
    };
    if (n > 1 && wave < kRotWaves) rotations(0, 0);
    __syncthreads();
    int d = 0;
    for (int sweep = 0; sweep < max_sweeps && n > 1; ++sweep) {
        bool turned = false;   // some rotation in this sweep
        for (int r = 0; r < m - 1; ++r, d ^= 1) {
            const bool some = nrot[d] != 0;
            turned = turned || some;
            if (some) {
                // a wave takes whole rows of blocks (pair k, its rotation uniform), kPer at a time, its
                // lanes the pairs l
                for (int l0 = 0; l0 < mk; l0 += 64) {
                    const int l = min(l0 + lane, mk - 1);
                    const bool on = l0 + lane < mk;
                    const double2 rl = rot[d][l];
                    const int2 pl = pq[d][l];
                    const double cl = rl.x, sl = rl.y;
                    double* cp = A + pl.x;
                    double* cq = A + pl.y;
                    for (int k0 = wave; k0 < mk; k0 += kWaves * kPer) {
                        double2 rk[kPer];
                        int2 pk[kPer];
                        double a[kPer][4];
#pragma unroll
                        for (int u = 0; u < kPer; ++u) {
                            const int k = min(k0 + kWaves * u, mk - 1);
                            rk[u] = rot[d][k];
                            pk[u] = pq[d][k];
                        }
#pragma unroll
                        for (int u = 0; u < kPer; ++u) {
                            const int rp = __builtin_amdgcn_readfirstlane(pk[u].x) * ld;
                            const int rq = __builtin_amdgcn_readfirstlane(pk[u].y) * ld;
                            a[u][0] = cp[rp];
                            a[u][1] = cq[rp];
                            a[u][2] = cp[rq];
                            a[u][3] = cq[rq];
                        }
#pragma unroll
                        for (int u = 0; u < kPer; ++u) {
                            const double ck = rk[u].x, sk = rk[u].y;
                            const double r00 = turn_p(ck, sk, a[u][0], a[u][2]), r01 = turn_p(ck, sk, a[u][1], a[u][3]);
                            const double r10 = turn_q(ck, sk, a[u][0], a[u][2]), r11 = turn_q(ck, sk, a[u][1], a[u][3]);
                            if (k0 + kWaves * u < mk && on && (sk != 0.0 || sl != 0.0)) {
                                const int rp = __builtin_amdgcn_readfirstlane(pk[u].x) * ld;
                                const int rq = __builtin_amdgcn_readfirstlane(pk[u].y) * ld;
                                cp[rp] = turn_p(cl, sl, r00, r01);
                                cq[rp] = turn_q(cl, sl, r00, r01);
                                cp[rq] = turn_p(cl, sl, r10, r11);
                                cq[rq] = turn_q(cl, sl, r10, r11);
                            }
                        }
                    }
                }
                __syncthreads();
            }
            // the next round's rotations (the next sweep's first after the last), and the vectors
            if (wave < kRotWaves) {
                rotations(r + 1 < m - 1 ? r + 1 : 0, d ^ 1);
            } else if (some) {
                if (vl) turn(VL, lv, d);
                else turn(VG, n, d);
            }
            if (tid == 0 && some) nrot[d] = 0;   // read by all before the pass, written again after this barrier
            __syncthreads();
        }
        if (!turned) break;
    }
    __syncthreads();
    // eigenvalues ascending (ties by index) with their vectors as columns of Z
    int* rank = reinterpret_cast<int*>(&rot[0][0]);   // n ints in n / 2 (c, s)
    for (int i = tid; i < n; i += kJacobiThreads) {
        const double di = A[i * ld + i];
        int r = 0;
        for (int j = 0; j < n; ++j) {
            const double dj = A[j * ld + j];
            if (dj < di || (dj == di && j < i)) ++r;
        }
        ev[r] = di;
        rank[i] = r;
    }
    __syncthreads();
    for (int e = tid; e < n * n; e += kJacobiThreads) {
        const int i = e / n, r = e - i * n;
        Z[(long)r * n + rank[i]] = vl ? VL[i * lv + r] : VG[e];
    }
}

hipError_t batched_jacobi(int nslot, const MatSlot* slots, Store A, Store V, Store evals, Store Z, int maxn, int max_sweeps,
                          hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    // (a smaller matrix of the launch may keep its vectors in LDS where the largest does not)
    const int nl = std::min(maxn, kJacobiLdsN);
    const size_t need = sizeof(double) * (size_t)(jacobi_v_fits(nl) ? jacobi_a(nl) + jacobi_v(nl) : kJacobiLds);
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&k_batched_jacobi_lds),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kJacobiLds * sizeof(double))))
        return e;
    hipLaunchKernelGGL(k_batched_jacobi_lds, dim3(nslot), dim3(kJacobiThreads), need, st, slots, A, V, evals, Z,
                       max_sweeps);
    if (maxn > kJacobiLdsN)
        hipLaunchKernelGGL(k_batched_jacobi, dim3(nslot), dim3(kJacobiThreads), 0, st, slots, A, V, evals, Z, max_sweeps);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Occupation of coinciding levels.  Where the highest occupied and the lowest empty level lie
// within kTieLevel of each other (a pi pair of a linear molecule that the first builds leave half
// filled: exactly degenerate, 2e-16 apart), rounding decides which of their orbitals Jacobi lists
// first, and with it the order in which the Fock atomics arrived: an HF molecule converged to
// |dE| < 1e-8 then has one of two mirror-image densities, 2.4e-7 apart, and from run to run not the
// same.  Such orbitals keep the order that they had in the iteration before.  Z holds the eigenvectors
// over that iteration's orbitals, so the first of the level becomes the projection into it of the
// first orbital whose projection is at least half as long as the longest, the next the same among
// what is orthogonal to it.  (Exactly equal levels come out in that order anyway, ties by index.)  kTieLevel is
// far above the rounding of the levels (1e-14) and far below what a distortion splits them by.
// One block per slot; without such levels (nearly always) it reads two numbers and ends.
// ---------------------------------------------------------------------------
constexpr double kTieLevel = 1e-10;
__global__ __launch_bounds__(256) void k_batch_ties(const MatSlot* __restrict__ slots, Store evals, Store Zs) {
    __shared__ double red[4], w[256];
    __shared__ int first;
    const MatSlot m = slots[blockIdx.x];
    const int n = m.n;
    if (m.nocc <= 0 || m.nocc >= n) return;
    const double* ev = evals.s[m.spin] + m.off;
    if (!(ev[m.nocc] - ev[m.nocc - 1] <= kTieLevel)) return;
    double* Z = Zs.s[m.spin] + m.off;
    int lo = m.nocc - 1, hi = m.nocc + 1;
    while (lo > 0 && ev[lo] - ev[lo - 1] <= kTieLevel) --lo;
    while (hi < n && ev[hi] - ev[hi - 1] <= kTieLevel) ++hi;
    const int r = threadIdx.x, lane = r & 63;
    double* row = Z + (long)r * n;   // n <= 256: a row per thread
    for (int c0 = lo; c0 < m.nocc; ++c0) {
        double s = 0.0;
        if (r < n)
            for (int c = c0; c < hi; ++c) s = fma(row[c], row[c], s);
        double big = s;
        for (int o = 32; o >= 1; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
        if (lane == 0) red[r >> 6] = big;
        if (r == 0) first = n;
        __syncthreads();
        big = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
        if (r < n && s >= 0.25 * big) atomicMin(&first, r);
        __syncthreads();
        const int f = first;
        if (f >= n) return;   // not a number
        // the reflection of the level's orbitals that takes row f to (|row|, 0, ..): v = row - |row| e
        if (r < hi - c0) w[r] = Z[(long)f * n + c0 + r];
        __syncthreads();
        double tail = 0.0;
        for (int c = 1; c < hi - c0; ++c) tail = fma(w[c], w[c], tail);
        const double x = w[0], len = sqrt(fma(x, x, tail));
        const double v0 = x > 0.0 ? -tail / (x + len) : x - len, v2 = fma(v0, v0, tail);
        if (v2 > 0.0 && r < n) {
            double t = v0 * row[c0];
            for (int c = 1; c < hi - c0; ++c) t = fma(w[c], row[c0 + c], t);
            t *= 2.0 / v2;
            row[c0] = fma(-t, v0, row[c0]);
            for (int c = 1; c < hi - c0; ++c) row[c0 + c] = fma(-t, w[c], row[c0 + c]);
        }
        __syncthreads();
    }
}

hipError_t batch_ties(int nslot, const MatSlot* slots, Store evals, Store Z, hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_ties, dim3(nslot), dim3(256), 0, st, slots, evals, Z);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// per-molecule helpers: one 256-thread block per slot
// ---------------------------------------------------------------------------
__device__ __forceinline__ double block_reduce_sum(double v, double* red) {
    for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    for (int k = 0; k < (int)(blockDim.x >> 6); ++k) s += red[k];
    __syncthreads();
    return s;
}

// out[q nslot + k] = sum_ij A_q,ij B_q,ij over slot k's n x n matrices
__global__ __launch_bounds__(256) void k_batch_dots(const MatSlot* __restrict__ slots, DotPairs q, double* __restrict__ out) {
    __shared__ double red[4];
    const MatSlot m = slots[blockIdx.x];
    const double* A = q.a[blockIdx.y][m.spin];
    const double* B = q.b[blockIdx.y][m.spin];
    if (!A || !B) return;
    double s = 0.0;
    for (int e = threadIdx.x; e < m.n * m.n; e += 256) s += A[m.off + e] * B[m.off + e];
    s = block_reduce_sum(s, red);
    if (threadIdx.x == 0) out[blockIdx.y * gridDim.x + blockIdx.x] = s;
}

// out[k] = sqrt(sum (A - B)^2) / n over slot k
__global__ __launch_bounds__(256) void k_batch_diffnorm(const MatSlot* __restrict__ slots, Store A, Store B,
                                                        double* __restrict__ out) {
    __shared__ double red[4];
    const MatSlot m = slots[blockIdx.x];
    const double* a = A.s[m.spin] + m.off;
    const double* b = B.s[m.spin] + m.off;
    double s = 0.0;
    for (int e = threadIdx.x; e < m.n * m.n; e += 256) {
        const double d = a[e] - b[e];
        s += d * d;
    }
    s = block_reduce_sum(s, red);
    if (threadIdx.x == 0) out[blockIdx.x] = sqrt(s) / m.n;
}

// element-wise kernels: kSlotBlocks blocks share a slot's matrix
constexpr int kSlotBlocks = 8;

// G = W + W^T, or W - W^T as 2 W - (W + W^T)
template <bool ANTI>
__global__ __launch_bounds__(256) void k_batch_sym(const MatSlot* __restrict__ slots, Store W, Store G) {
    const MatSlot m = slots[blockIdx.x];
    const double* w = W.s[m.spin] + m.off;
    double* g = G.s[m.spin] + m.off;
    for (int e = blockIdx.y * 256 + threadIdx.x; e < m.n * m.n; e += 256 * kSlotBlocks) {
        const int i = e / m.n, j = e - i * m.n;
        const double x = w[e], v = x + w[j * m.n + i];
        g[e] = ANTI ? fma(2.0, x, -v) : v;
    }
}

__global__ __launch_bounds__(256) void k_batch_add(const MatSlot* __restrict__ slots, const double* __restrict__ H, Store G,
                                                   Store F) {
    const MatSlot m = slots[blockIdx.x];
    const double* h = H + m.off;
    const double* g = G.s[m.spin] + m.off;
    double* f = F.s[m.spin] + m.off;
    for (int e = blockIdx.y * 256 + threadIdx.x; e < m.n * m.n; e += 256 * kSlotBlocks) f[e] = h[e] + g[e];
}

__global__ __launch_bounds__(256) void k_batch_densities(long long len, Store P, double* __restrict__ D0, Store Pold) {
    const long long e = (long long)blockIdx.x * 256 + threadIdx.x;
    if (e >= len) return;
    const double a = P.s[0][e], b = P.s[1][e];
    D0[e] = a + b;
    Pold.s[0][e] = a;
    Pold.s[1][e] = b;
}

// Dsh_m[s][t] = max |D| over the function block of shells s, t of every active molecule m (D1,
// D2 optional further densities of the same layout), dmax[m] (zeroed) the largest of them
__global__ __launch_bounds__(256) void k_batch_shell_max(const MolDesc* __restrict__ mols, const int* __restrict__ shoff,
                                                         const int* __restrict__ active, const int* __restrict__ sh_off,
                                                         const int* __restrict__ sh_n, const double* __restrict__ D,
                                                         const double* __restrict__ D1, const double* __restrict__ D2,
                                                         double* __restrict__ Dsh, unsigned long long* __restrict__ dmax) {
    const int mol = blockIdx.y;
    if (!active[mol]) return;
    const MolDesc m = mols[mol];
    const int ns = m.nsh;
    double big = 0.0;
    const int st = blockIdx.x * 256 + threadIdx.x;
    if (st < ns * ns) {
        const int s = st / ns, t = st % ns;
        const int o1 = sh_off[shoff[mol] + s], n1 = sh_n[shoff[mol] + s];
        const int o2 = sh_off[shoff[mol] + t], n2 = sh_n[shoff[mol] + t];
        double v = 0.0;
        for (int a = 0; a < n1; ++a)
            for (int b = 0; b < n2; ++b) {
                const long ij = m.moff + (long)(o1 + a) * m.n + o2 + b;
                v = fmax(v, fabs(D[ij]));
                if (D1) v = fmax(v, fabs(D1[ij]));
                if (D2) v = fmax(v, fabs(D2[ij]));
            }
        Dsh[m.dshoff + st] = v;
        big = v;
    }
    for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
    if ((threadIdx.x & 63) == 0 && big > 0.0) atomicMax(dmax + mol, (unsigned long long)__double_as_longlong(big));
}

// F_k = sum_j c[k kMaxLin + j] H_j,k: a linear combination of stores per slot
__global__ __launch_bounds__(256) void k_batch_lincomb(const MatSlot* __restrict__ slots, const double* __restrict__ coef,
                                                       LinSources src, Store F) {
    const MatSlot m = slots[blockIdx.x];
    double* f = F.s[m.spin] + m.off;
    for (int e = blockIdx.y * 256 + threadIdx.x; e < m.n * m.n; e += 256 * kSlotBlocks) {
        double v = 0.0;
#pragma unroll
        for (int j = 0; j < kMaxLin; ++j) {
            const double cj = coef[blockIdx.x * kMaxLin + j];
            if (cj != 0.0) v = fma(cj, src.s[j][m.spin][m.off + e], v);
        }
        f[e] = v;
    }
}

hipError_t batch_dots(int nslot, const MatSlot* slots, const DotPairs& q, double* out, hipStream_t st) {
    if (nslot <= 0 || q.n <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_dots, dim3(nslot, q.n), dim3(256), 0, st, slots, q, out);
    return hipGetLastError();
}
hipError_t batch_diffnorm(int nslot, const MatSlot* slots, Store A, Store B, double* out, hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_diffnorm, dim3(nslot), dim3(256), 0, st, slots, A, B, out);
    return hipGetLastError();
}
hipError_t batch_sym(int nslot, const MatSlot* slots, Store W, Store G, hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    hipLaunchKernelGGL((k_batch_sym<false>), dim3(nslot, kSlotBlocks), dim3(256), 0, st, slots, W, G);
    return hipGetLastError();
}
hipError_t batch_antisym(int nslot, const MatSlot* slots, Store W, Store out, hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    hipLaunchKernelGGL((k_batch_sym<true>), dim3(nslot, kSlotBlocks), dim3(256), 0, st, slots, W, out);
    return hipGetLastError();
}
hipError_t batch_add(int nslot, const MatSlot* slots, const double* H, Store G, Store F, hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_add, dim3(nslot, kSlotBlocks), dim3(256), 0, st, slots, H, G, F);
    return hipGetLastError();
}
hipError_t batch_densities(long long len, Store P, double* D0, Store Pold, hipStream_t st) {
    hipLaunchKernelGGL(k_batch_densities, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, len, P, D0, Pold);
    return hipGetLastError();
}
hipError_t batch_shell_max(int nmol, int maxsh, const MolDesc* mols, const int* shoff, const int* active,
                           const int* sh_off, const int* sh_n, const double* D, const double* D1, const double* D2,
                           double* Dsh, double* dmax, hipStream_t st) {
    if (nmol <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_shell_max, dim3((maxsh * maxsh + 255) / 256, nmol), dim3(256), 0, st, mols, shoff, active,
                       sh_off, sh_n, D, D1, D2, Dsh, reinterpret_cast<unsigned long long*>(dmax));
    return hipGetLastError();
}
hipError_t batch_lincomb(int nslot, const MatSlot* slots, const double* coef, const LinSources& src, Store F,
                         hipStream_t st) {
    if (nslot <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_batch_lincomb, dim3(nslot, kSlotBlocks), dim3(256), 0, st, slots, coef, src, F);
    return hipGetLastError();
}

}  // namespace uno
