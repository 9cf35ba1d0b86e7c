// Dense FP64 kernels: MFMA GEMM, Householder tridiagonalisation with reflector
// accumulation, row-parallel application of QL rotation sweeps, and the small
// element-wise / reduction kernels of the SCF loop.
#include <hip/hip_runtime.h>
#include "kernels.hpp"

#define UNO_LAUNCH_FILL(len, ptr, st) \
    do { hipError_t e_ = k_fill((len), 0.0, (ptr), (st)); if (e_ != hipSuccess) return e_; } while (0)

namespace uno {

typedef double double4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// element-wise
// ---------------------------------------------------------------------------
__global__ void k_unpack_(int n, const double* __restrict__ pk, double* __restrict__ D) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)n * n) return;
    const int i = (int)(t / n), j = (int)(t % n);
    D[t] = i >= j ? pk[(long)i * (i + 1) / 2 + j] : pk[(long)j * (j + 1) / 2 + i];
}
hipError_t k_unpack(int n, const double* packed, double* dense, hipStream_t st) {
    const long len = (long)n * n;
    hipLaunchKernelGGL(k_unpack_, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, n, packed, dense);
    return hipGetLastError();
}

__global__ void k_pack_(int n, const double* __restrict__ D, double* __restrict__ pk, int mode) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n2 = (long)n * (n + 1) / 2;
    if (t >= n2) return;
    // invert t = i(i+1)/2 + j
    int i = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((long)i * (i + 1) / 2 > t) --i;
    while ((long)(i + 1) * (i + 2) / 2 <= t) ++i;
    const int j = (int)(t - (long)i * (i + 1) / 2);
    if (mode == 0) pk[t] = D[(long)i * n + j];
    else pk[t] += D[(long)i * n + j] + D[(long)j * n + i];
}
hipError_t k_pack(int n, const double* dense, double* packed, hipStream_t st) {
    const long n2 = (long)n * (n + 1) / 2;
    hipLaunchKernelGGL(k_pack_, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, n, dense, packed, 0);
    return hipGetLastError();
}
hipError_t k_pack_sym_add(int n, const double* W, double* packed, hipStream_t st) {
    const long n2 = (long)n * (n + 1) / 2;
    hipLaunchKernelGGL(k_pack_, dim3((unsigned)((n2 + 255) / 256)), dim3(256), 0, st, n, W, packed, 1);
    return hipGetLastError();
}

__global__ void k_sym_w_(int n, const double* __restrict__ W, double* __restrict__ G, int acc) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)n * n) return;
    const int i = (int)(t / n), j = (int)(t % n);
    const double v = W[t] + W[(long)j * n + i];
    G[t] = acc ? G[t] + v : v;
}
hipError_t k_sym_w(int n, const double* W, double* G, hipStream_t st, bool accumulate) {
    const long len = (long)n * n;
    hipLaunchKernelGGL(k_sym_w_, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, n, W, G,
                       accumulate ? 1 : 0);
    return hipGetLastError();
}

__global__ void k_axpby_(long len, double a, const double* x, double b, const double* y, double* z) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < len) z[t] = a * x[t] + b * y[t];
}
hipError_t k_axpby(long len, double a, const double* x, double b, const double* y, double* z, hipStream_t st) {
    hipLaunchKernelGGL(k_axpby_, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, len, a, x, b, y, z);
    return hipGetLastError();
}

__global__ void k_fill_(long len, double v, double* x) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < len) x[t] = v;
}
hipError_t k_fill(long len, double v, double* x, hipStream_t st) {
    if (len <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill_, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, len, v, x);
    return hipGetLastError();
}

__global__ void k_scale_cols_(int n, const double* __restrict__ Z, const double* __restrict__ f, double* __restrict__ X) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < (long)n * n) X[t] = Z[t] * f[t % n];
}
hipError_t k_scale_cols(int n, const double* Z, const double* f, double* X, hipStream_t st) {
    const long nn = (long)n * n;
    if (nn <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_scale_cols_, dim3((unsigned)((nn + 255) / 256)), dim3(256), 0, st, n, Z, f, X);
    return hipGetLastError();
}

// deterministic block reduction (fixed order; blockDim.x a power of two)
__device__ double block_sum(double v, double* sh) {
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] += sh[t + s];
        __syncthreads();
    }
    return sh[0];
}

// two-pass reductions over long vectors, deterministic: kRedBlocks blocks each sum a
// contiguous chunk in a fixed order into ws[block], then one block adds ws in order
__global__ __launch_bounds__(256) void k_red_part(long len, const double* A, const double* B, int diff, double* ws) {
    __shared__ double sh[256];
    const long chunk = (len + gridDim.x - 1) / gridDim.x;
    const long lo = (long)blockIdx.x * chunk, hi = lo + chunk < len ? lo + chunk : len;
    double s = 0.0;
    for (long i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        if (diff) {
            const double d = A[i] - B[i];
            s = fma(d, d, s);
        } else {
            s = fma(A[i], B[i], s);
        }
    }
    s = block_sum(s, sh);
    if (threadIdx.x == 0) ws[blockIdx.x] = s;
}
// mode 0: out += sum; mode 1: out = sqrt(sum) / n
__global__ __launch_bounds__(256) void k_red_final(int nb, const double* ws, int mode, int n, double* out) {
    __shared__ double sh[256];
    double s = (int)threadIdx.x < nb ? ws[threadIdx.x] : 0.0;
    s = block_sum(s, sh);
    if (threadIdx.x == 0) {
        if (mode == 0) out[0] += s;
        else out[0] = sqrt(s) / n;
    }
}
hipError_t k_dot(long len, const double* A, const double* B, double* out, double* ws, hipStream_t st) {
    hipLaunchKernelGGL(k_red_part, dim3(kRedBlocks), dim3(256), 0, st, len, A, B, 0, ws);
    hipLaunchKernelGGL(k_red_final, dim3(1), dim3(256), 0, st, kRedBlocks, (const double*)ws, 0, 0, out);
    return hipGetLastError();
}
hipError_t k_diffnorm(long len, int n, const double* A, const double* B, double* out, double* ws, hipStream_t st) {
    hipLaunchKernelGGL(k_red_part, dim3(kRedBlocks), dim3(256), 0, st, len, A, B, 1, ws);
    hipLaunchKernelGGL(k_red_final, dim3(1), dim3(256), 0, st, kRedBlocks, (const double*)ws, 1, n, out);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Density-matrix purification (SCF densities without an eigensolve): Gershgorin bounds
// of F', the initial X = (hi I - F') / (hi - lo) with the bounds read on the device, and
// the traces tr(X) and tr(X^2) = sum X_ij^2 (symmetric X) per step.
// ---------------------------------------------------------------------------
// one block per row: lohi[2i] = F_ii - sum_{j != i} |F_ij|, lohi[2i+1] = F_ii + the same
__global__ __launch_bounds__(256) void k_gersh_rows(int n, const double* __restrict__ F, double* __restrict__ lohi) {
    __shared__ double sh[256];
    const int i = blockIdx.x;
    const double* row = F + (long)i * n;
    double r = 0.0;
    for (int j = threadIdx.x; j < n; j += 256)
        if (j != i) r += fabs(row[j]);
    r = block_sum(r, sh);
    if (threadIdx.x == 0) {
        lohi[2 * i] = row[i] - r;
        lohi[2 * i + 1] = row[i] + r;
    }
}
// bounds[0] = min lo, bounds[1] = max hi over the rows (one block)
__global__ __launch_bounds__(1024) void k_gersh_final(int n, const double* __restrict__ lohi, double* bounds) {
    __shared__ double slo[1024], shi[1024];
    double lo = 1e300, hi = -1e300;
    for (int i = threadIdx.x; i < n; i += 1024) {
        lo = fmin(lo, lohi[2 * i]);
        hi = fmax(hi, lohi[2 * i + 1]);
    }
    slo[threadIdx.x] = lo;
    shi[threadIdx.x] = hi;
    __syncthreads();
    for (int s = 512; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            slo[threadIdx.x] = fmin(slo[threadIdx.x], slo[threadIdx.x + s]);
            shi[threadIdx.x] = fmax(shi[threadIdx.x], shi[threadIdx.x + s]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        bounds[0] = slo[0];
        bounds[1] = shi[0];
    }
}
__global__ void k_sp2_init_(int n, const double* __restrict__ F, const double* __restrict__ bounds,
                            double* __restrict__ X) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)n * n) return;
    const double lo = bounds[0], hi = bounds[1];
    const double inv = 1.0 / (hi - lo);
    const long i = t / n, j = t - i * n;
    X[t] = ((i == j ? hi : 0.0) - F[t]) * inv;
}
hipError_t sp2_init(int n, const double* F, double* X, double* lohi, double* bounds, hipStream_t st) {
    hipLaunchKernelGGL(k_gersh_rows, dim3((unsigned)n), dim3(256), 0, st, n, F, lohi);
    hipLaunchKernelGGL(k_gersh_final, dim3(1), dim3(1024), 0, st, n, (const double*)lohi, bounds);
    const long len = (long)n * n;
    hipLaunchKernelGGL(k_sp2_init_, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, n, F,
                       (const double*)bounds, X);
    return hipGetLastError();
}
// out[0] = tr(A)
__global__ __launch_bounds__(1024) void k_trace_(int n, const double* __restrict__ A, double* out) {
    __shared__ double sh[1024];
    double s = 0.0;
    for (int i = threadIdx.x; i < n; i += 1024) s += A[(long)i * n + i];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int k = 512; k > 0; k >>= 1) {
        if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = sh[0];
}
hipError_t k_trace(int n, const double* A, double* out, hipStream_t st) {
    hipLaunchKernelGGL(k_trace_, dim3(1), dim3(1024), 0, st, n, A, out);
    return hipGetLastError();
}

// one thread per shell pair (s, t): max |D| over its function block of up to three matrices,
// and the largest of all (|x| orders as its bit pattern)
__global__ __launch_bounds__(256) void k_shell_max_(int n, int nsh, const int* __restrict__ off, const int* __restrict__ nf,
                                                    const double* __restrict__ D, const double* __restrict__ D1,
                                                    const double* __restrict__ D2, double* __restrict__ Dsh,
                                                    unsigned long long* dmax) {
    const long st = (long)blockIdx.x * 256 + threadIdx.x;
    double m = 0.0;
    if (st < (long)nsh * nsh) {
        const int s = (int)(st / nsh), t = (int)(st - (long)s * nsh);
        const int ns = nf[s], nt = nf[t];
        const long o = (long)off[s] * n + off[t];
        for (int a = 0; a < ns; ++a)
            for (int b = 0; b < nt; ++b) {
                const long ij = o + (long)a * n + b;
                m = fmax(m, fabs(D[ij]));
                if (D1) m = fmax(m, fabs(D1[ij]));
                if (D2) m = fmax(m, fabs(D2[ij]));
            }
        Dsh[st] = m;
    }
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if ((threadIdx.x & 63) == 0 && m > 0.0) atomicMax(dmax, (unsigned long long)__double_as_longlong(m));
}
hipError_t k_shell_max(int n, int nsh, const int* sh_off, const int* sh_n, const double* D, const double* D1,
                       const double* D2, double* Dsh, double* dmax, hipStream_t st) {
    const long len = (long)nsh * nsh;
    hipLaunchKernelGGL(k_shell_max_, dim3((unsigned)((len + 255) / 256)), dim3(256), 0, st, n, nsh, sh_off, sh_n, D, D1,
                       D2, Dsh, reinterpret_cast<unsigned long long*>(dmax));
    return hipGetLastError();
}

// max |x_i| over a long vector: |x_i| >= 0 orders as its bit pattern (a NaN above
// everything, so it propagates), so each block's maximum pattern goes to out with an
// integer atomicMax after a fill kernel zeroes out (no memset node under graph capture)
__global__ __launch_bounds__(256) void k_absmax_part(long len, const double* __restrict__ x,
                                                     unsigned long long* out) {
    __shared__ unsigned long long sh[256];
    unsigned long long m = 0;
    for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < len; i += (long)gridDim.x * 256) {
        const unsigned long long b = (unsigned long long)__double_as_longlong(x[i]) & 0x7fffffffffffffffull;
        m = b > m ? b : m;
    }
    sh[threadIdx.x] = m;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sh[threadIdx.x] = sh[threadIdx.x] > sh[threadIdx.x + s] ? sh[threadIdx.x] : sh[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0 && sh[0]) atomicMax(out, sh[0]);
}
hipError_t k_absmax(long len, const double* x, double* out, hipStream_t st) {
    if (hipError_t e = k_fill(1, 0.0, out, st)) return e;
    if (len <= 0) return hipSuccess;
    const long blocks = std::min<long>((len + 255) / 256, 1024);
    hipLaunchKernelGGL(k_absmax_part, dim3((unsigned)blocks), dim3(256), 0, st, len, x,
                       reinterpret_cast<unsigned long long*>(out));
    return hipGetLastError();
}

// A_ii += alpha (n x n)
__global__ void k_shift_diag_(int n, double alpha, double* A) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) A[(long)i * n + i] += alpha;
}
hipError_t k_shift_diag(int n, double alpha, double* A, hipStream_t st) {
    hipLaunchKernelGGL(k_shift_diag_, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, n, alpha, A);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// FP64 MFMA GEMM: 64x64 block tile, 4 waves each owning a 32x32 quarter made of
// 2x2 tiles of v_mfma_f64_16x16x4_f64.  Operand layout of that instruction:
// A(16x4): lane l holds A[l%16][l/16]; B(4x16): lane l holds B[l/16][l%16];
// D(16x16): lane l holds D[4*r + l/16][l%16] in register r (pinned by an on-device probe).
// ---------------------------------------------------------------------------
// Split K (gridDim.z > 1): block z covers k in [z kchunk, (z+1) kchunk) and adds
// alpha * its partial product into C, which the launcher has already scaled by beta.
// One 64 x 64 output tile of C = op(A) op(B) over k in [kb, ke), accumulated in acc (four
// waves, each a 32 x 32 quarter of 2 x 2 MFMA tiles).  K advances in chunks of 32: the next
// chunk's operands are loaded from global memory into registers while the current chunk's
// MFMAs run on LDS, then stored into the other LDS buffer (one barrier per chunk).
constexpr int kGemmKc = 32;
template <bool TA, bool TB>
__device__ __forceinline__ void gemm_tile(int M, int N, int kb, int ke, const double* __restrict__ A, int lda,
                                          const double* __restrict__ B, int ldb, int bi, int bj,
                                          double (*sA)[kGemmKc][64 + 2], double (*sB)[kGemmKc][64 + 2],
                                          double4_t acc[2][2]) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    for (int a = 0; a < 2; ++a)
        for (int b = 0; b < 2; ++b) acc[a][b] = (double4_t){0.0, 0.0, 0.0, 0.0};
    double ra[8], rb[8];
    // element e = tid + 256 m of a chunk: A as (i, kk), B as (kk, j); the fastest index runs
    // along the operand's contiguous dimension
    auto load = [&](int k0) {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int e = tid + 256 * m;
            int i, kk;
            if (TA) { kk = e / 64; i = e % 64; } else { i = e / kGemmKc; kk = e % kGemmKc; }
            const int gi = bi + i, gk = k0 + kk;
            ra[m] = (gi < M && gk < ke) ? (TA ? A[(long)gk * lda + gi] : A[(long)gi * lda + gk]) : 0.0;
            int j, kj;
            if (TB) { j = e / kGemmKc; kj = e % kGemmKc; } else { kj = e / 64; j = e % 64; }
            const int gj = bj + j, gk2 = k0 + kj;
            rb[m] = (gj < N && gk2 < ke) ? (TB ? B[(long)gj * ldb + gk2] : B[(long)gk2 * ldb + gj]) : 0.0;
        }
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int e = tid + 256 * m;
            int i, kk;
            if (TA) { kk = e / 64; i = e % 64; } else { i = e / kGemmKc; kk = e % kGemmKc; }
            sA[buf][kk][i] = ra[m];
            int j, kj;
            if (TB) { j = e / kGemmKc; kj = e % kGemmKc; } else { kj = e / 64; j = e % 64; }
            sB[buf][kj][j] = rb[m];
        }
    };
    if (kb >= ke) return;
    load(kb);
    store(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = kb; k0 < ke; k0 += kGemmKc) {
        const bool more = k0 + kGemmKc < ke;
        if (more) load(k0 + kGemmKc);
#pragma unroll
        for (int kk = 0; kk < kGemmKc; kk += 4) {
            double av[2], bv[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                av[t] = sA[buf][kk + (lane >> 4)][wi + t * 16 + (lane & 15)];
                bv[t] = sB[buf][kk + (lane >> 4)][wj + t * 16 + (lane & 15)];
            }
#pragma unroll
            for (int ta = 0; ta < 2; ++ta)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb)
                    acc[ta][tb] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[ta], bv[tb], acc[ta][tb], 0, 0, 0);
        }
        if (more) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
    }
}

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_gemm(int M, int N, int K, double alpha, const double* __restrict__ A,
                                              int lda, const double* __restrict__ B, int ldb, double beta,
                                              double* __restrict__ C, int ldc, int kchunk) {
    __shared__ double sA[2][kGemmKc][64 + 2];
    __shared__ double sB[2][kGemmKc][64 + 2];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int bi = blockIdx.y * 64, bj = blockIdx.x * 64;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    const int kb = blockIdx.z * kchunk, ke = kb + kchunk < K ? kb + kchunk : K;
    double4_t acc[2][2];
    gemm_tile<TA, TB>(M, N, kb, ke, A, lda, B, ldb, bi, bj, sA, sB, acc);
#pragma unroll
    for (int ta = 0; ta < 2; ++ta)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gi = bi + wi + ta * 16 + 4 * r + (lane >> 4);
                const int gj = bj + wj + tb * 16 + (lane & 15);
                if (gi < M && gj < N) {
                    double* c = C + (long)gi * ldc + gj;
                    if (gridDim.z > 1) unsafeAtomicAdd(c, alpha * acc[ta][tb][r]);
                    else *c = (beta == 0.0 ? 0.0 : beta * *c) + alpha * acc[ta][tb][r];
                }
            }
}

// C <- beta C on an M x N region (beta = 0 writes zeros)
__global__ void k_scale_c(int M, int N, double beta, double* C, int ldc) {
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (long)M * N) return;
    double* c = C + (t / N) * ldc + t % N;
    *c = beta == 0.0 ? 0.0 : beta * *c;
}

// split K adds the chunks' products with FP64 atomics, in whatever order the blocks
// finish; a thread that asks for deterministic products runs one block per tile instead
static thread_local int t_gemm_det = 0;
int gemm_deterministic(int on) {
    const int prev = t_gemm_det;
    t_gemm_det = on;
    return prev;
}

hipError_t gemm_f64(bool ta, bool tb, int m, int n, int k, double alpha, const double* A, int lda, const double* B,
                    int ldb, double beta, double* C, int ldc, hipStream_t st) {
    // few output tiles and a long K (the WY back-transform's 32-row products): split K so
    // that the launch has about 512 blocks, each chunk at least 64 long
    const long tiles = (long)((n + 63) / 64) * ((m + 63) / 64);
    int ksplit = 1, kchunk = k;
    if (tiles < 128 && k >= 256 && !t_gemm_det) {
        ksplit = (int)std::min<long>(512 / tiles, k / 64);
        if (ksplit > 1) {
            kchunk = ((k + ksplit - 1) / ksplit + kGemmKc - 1) / kGemmKc * kGemmKc;
            ksplit = (k + kchunk - 1) / kchunk;
        } else {
            ksplit = 1;
        }
    }
    if (ksplit > 1) {
        const long mn = (long)m * n;
        hipLaunchKernelGGL(k_scale_c, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, st, m, n, beta, C, ldc);
    }
    const dim3 grid((unsigned)((n + 63) / 64), (unsigned)((m + 63) / 64), (unsigned)ksplit), blk(256);
    if (!ta && !tb) hipLaunchKernelGGL((k_gemm<false, false>), grid, blk, 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, kchunk);
    else if (ta && !tb) hipLaunchKernelGGL((k_gemm<true, false>), grid, blk, 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, kchunk);
    else if (!ta && tb) hipLaunchKernelGGL((k_gemm<false, true>), grid, blk, 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, kchunk);
    else hipLaunchKernelGGL((k_gemm<true, true>), grid, blk, 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, kchunk);
    return hipGetLastError();
}

// One purification step per launch, the host never waiting in between.  The step's state
// (which buffer holds X, the countdown after idempotency, done) passes from launch k to
// launch k+1 through st[k] -> st[k+1]; every block derives the same decision from the
// same data in the same order.  Per step: tr(X) and tr(X^2) = sum X_ij^2 from the per-tile
// partial sums the previous step left (fixed-order sum), the choice X^2 or 2X - X^2
// (whichever trace lies nearer nocc), then X^2 on the upper-triangle 64 x 64 tiles only
// (FP64 MFMA, X symmetric) with the choice applied in the epilogue, each tile also
// written mirrored, and the new X's partial sums per tile.  Once tr(X) - tr(X^2) is below
// thr, two more steps run and the rest of the launches return at once.
struct Sp2State {
    int cur, extra, done, steps;
    double t1, t2;
};

__device__ __forceinline__ void sp2_tile_of(int t, int nb, int& ti, int& tj) {
    // upper-triangle tiles in row order: row ti holds tiles tj = ti .. nb-1
    int r = 0, base = 0;
    while (base + (nb - r) <= t) {
        base += nb - r;
        ++r;
    }
    ti = r;
    tj = r + (t - base);
}

// partial sums of X over tile t: [0] = sum X_ij^2 (mirror counted), [1] = sum of the diagonal
__device__ __forceinline__ void sp2_tile_sums(double s2, double s1, double* sh, double* out) {
    const int tid = threadIdx.x;
    sh[tid] = s2;
    sh[256 + tid] = s1;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) {
            sh[tid] += sh[tid + k];
            sh[256 + tid] += sh[256 + tid + k];
        }
        __syncthreads();
    }
    if (tid == 0) {
        out[0] = sh[0];
        out[1] = sh[256];
    }
}

__global__ __launch_bounds__(256) void k_sp2_stats0(int n, int nb, const double* __restrict__ X, double* part,
                                                     Sp2State* st0) {
    __shared__ double sh[512];
    int ti, tj;
    sp2_tile_of(blockIdx.x, nb, ti, tj);
    const int bi = ti * 64, bj = tj * 64;
    const double w = tj > ti ? 2.0 : 1.0;
    double s2 = 0.0, s1 = 0.0;
    for (int e = threadIdx.x; e < 4096; e += 256) {
        const int gi = bi + e / 64, gj = bj + e % 64;
        if (gi < n && gj < n) {
            const double v = X[(long)gi * n + gj];
            s2 += w * v * v;
            if (gi == gj) s1 += v;
        }
    }
    sp2_tile_sums(s2, s1, sh, part + 2 * blockIdx.x);
    if (blockIdx.x == 0 && threadIdx.x == 0) *st0 = Sp2State{0, -1, 0, 0, 0.0, 0.0};
}

__global__ __launch_bounds__(256) void k_sp2_step(int n, int nb, int nocc, double thr, const Sp2State* __restrict__ sin,
                                                  Sp2State* __restrict__ sout, double* buf0, double* buf1,
                                                  double* part0, double* part1) {
    __shared__ double sA[2][kGemmKc][64 + 2];
    __shared__ double sB[2][kGemmKc][64 + 2];
    __shared__ double sh[512];
    const int tid = threadIdx.x;
    const Sp2State s = *sin;
    if (s.done) {
        if (blockIdx.x == 0 && tid == 0) *sout = s;
        return;
    }
    // traces of the current X from the previous step's tile sums, in a fixed order
    const int ntile = nb * (nb + 1) / 2;
    const double* pin = s.cur ? part1 : part0;
    double a2 = 0.0, a1 = 0.0;
    for (int t = tid; t < ntile; t += 256) {
        a2 += pin[2 * t];
        a1 += pin[2 * t + 1];
    }
    sh[tid] = a2;
    sh[256 + tid] = a1;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) {
            sh[tid] += sh[tid + k];
            sh[256 + tid] += sh[256 + tid + k];
        }
        __syncthreads();
    }
    const double t2 = sh[0], t1 = sh[256];
    __syncthreads();
    const double idem = t1 - t2;
    int extra = s.extra, done = 0;
    if (!isfinite(idem)) done = 2;
    else {
        if (extra < 0 && fabs(idem) < thr) extra = 2;
        if (extra == 0) done = 1;
    }
    if (done) {
        if (blockIdx.x == 0 && tid == 0) *sout = Sp2State{s.cur, extra, done, s.steps, t1, t2};
        return;
    }
    if (extra > 0) --extra;
    const bool square = fabs(t2 - nocc) < fabs(2.0 * t1 - t2 - nocc);
    const double* X = s.cur ? buf1 : buf0;
    double* Y = s.cur ? buf0 : buf1;
    double* pout = s.cur ? part0 : part1;
    int ti, tj;
    sp2_tile_of(blockIdx.x, nb, ti, tj);
    const int wave = tid >> 6, lane = tid & 63;
    const int bi = ti * 64, bj = tj * 64;
    const int wi = (wave >> 1) * 32, wj = (wave & 1) * 32;
    double4_t acc[2][2];
    gemm_tile<false, false>(n, n, 0, n, X, n, X, n, bi, bj, sA, sB, acc);
    const double w = tj > ti ? 2.0 : 1.0;
    double s2 = 0.0, s1 = 0.0;
#pragma unroll
    for (int ta = 0; ta < 2; ++ta)
#pragma unroll
        for (int tb = 0; tb < 2; ++tb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int gi = bi + wi + ta * 16 + 4 * r + (lane >> 4);
                const int gj = bj + wj + tb * 16 + (lane & 15);
                if (gi < n && gj < n) {
                    const double x2 = acc[ta][tb][r];
                    const double v = square ? x2 : 2.0 * X[(long)gi * n + gj] - x2;
                    Y[(long)gi * n + gj] = v;
                    if (tj > ti) Y[(long)gj * n + gi] = v;
                    s2 += w * v * v;
                    if (gi == gj) s1 += v;
                }
            }
    sp2_tile_sums(s2, s1, sh, pout + 2 * blockIdx.x);
    if (blockIdx.x == 0 && tid == 0) *sout = Sp2State{1 - s.cur, extra, 0, s.steps + 1, t1, t2};
}

size_t sp2_state_bytes() { return sizeof(Sp2State); }

hipError_t sp2_start(int n, const double* X0, double* part0, void* st0, hipStream_t st) {
    const int nb = (n + 63) / 64, ntile = nb * (nb + 1) / 2;
    hipLaunchKernelGGL(k_sp2_stats0, dim3((unsigned)ntile), dim3(256), 0, st, n, nb, X0, part0,
                       reinterpret_cast<Sp2State*>(st0));
    return hipGetLastError();
}

hipError_t sp2_steps(int n, int nocc, double thr, void* states, int k0, int count, double* buf0, double* buf1,
                     double* part0, double* part1, hipStream_t st) {
    const int nb = (n + 63) / 64, ntile = nb * (nb + 1) / 2;
    Sp2State* S = reinterpret_cast<Sp2State*>(states);
    for (int k = k0; k < k0 + count; ++k)
        hipLaunchKernelGGL(k_sp2_step, dim3((unsigned)ntile), dim3(256), 0, st, n, nb, nocc, thr,
                           (const Sp2State*)(S + k), S + k + 1, buf0, buf1, part0, part1);
    return hipGetLastError();
}

hipError_t sp2_state_read(const void* states, int k, int* cur, int* done, int* steps, double* t1, hipStream_t st) {
    Sp2State h;
    hipError_t e = hipMemcpyAsync(&h, reinterpret_cast<const Sp2State*>(states) + k, sizeof(h),
                                  hipMemcpyDeviceToHost, st);
    if (e != hipSuccess) return e;
    if ((e = hipStreamSynchronize(st)) != hipSuccess) return e;
    *cur = h.cur;
    *done = h.done;
    *steps = h.steps;
    *t1 = h.t1;
    return hipSuccess;
}

// ---------------------------------------------------------------------------
// Householder tridiagonalisation A = Q T Q^T (one reflector per column k):
//   x = A[k+1:,k], alpha = -sign(x0)|x|, v = x - alpha e1, tau = 2/|v|^2
//   p = tau A22 v, K = tau/2 p.v, w = p - K v, A22 -= v w^T + w v^T
// d[k] = A[k][k], e[k] = alpha.  Reflector k is stored in row k of V (absolute column
// indices).  One launch per column k: every block first finishes step k-1 for itself
// (K and w of step k-1 from the previous launch's p and its terms of p.v, row k updated on the
// fly, reflector k from it: the same arithmetic in the same order in every block, so every
// block holds the same reflector; block 0 stores it), then applies the rank-2 update of
// step k-1 to its trailing rows and forms their p of step k.  The trailing matrix stays
// symmetric (full rows are updated), so row k is column k.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void hh_reflector(double nx2, double x0, double& alpha, double& v0, double& t) {
    const double nx = sqrt(nx2);
    alpha = x0 > 0.0 ? -nx : nx;
    v0 = x0 - alpha;
    const double vn2 = nx2 - x0 * x0 + v0 * v0;
    t = (nx2 == 0.0 || vn2 == 0.0) ? 0.0 : 2.0 / vn2;
}

// rows of the tridiagonal's chains, in chunks whose operands are read together; d and e carry zeros
// up to the next whole chunk
constexpr int kEigChunk = 16;
__host__ __device__ constexpr int eig_pad(int n) { return (n + kEigChunk - 1) / kEigChunk * kEigChunk; }

// sum over the wave in every lane, by DPP moves inside the vector unit (six LDS-crossbar shuffles
// cost four times their latency): quads, halves and rows of 16 by swaps, then rows 0 -> 1 and
// 2 -> 3 and halves 0 -> 1 by broadcasts, which leaves the total in lane 63
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
    return v + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// sum over the 16 lanes of a row, in every lane of it
__device__ __forceinline__ double row_total(double v) {
    v = dpp_add<0xb1, 0xf>(v);    // quad_perm 1,0,3,2
    v = dpp_add<0x4e, 0xf>(v);    // quad_perm 2,3,0,1
    v = dpp_add<0x141, 0xf>(v);   // row_half_mirror
    return dpp_add<0x140, 0xf>(v);   // row_mirror
}
__device__ __forceinline__ double lane_value(double v, int lane) {   // lane: the same in the whole wave
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, lane), hi = __builtin_amdgcn_readlane((int)(b >> 32), lane);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ double wave_total(double v) {
    v = row_total(v);
    v = dpp_add<0x142, 0xa>(v);   // row_bcast:15 into rows 1 and 3
    v = dpp_add<0x143, 0xc>(v);   // row_bcast:31 into rows 2 and 3
    return lane_value(v, 63);
}

// launch of column k (four rows per block, one wave per row; b0: the first block of the launch, a
// multiple of the XCD count, so that a row stays on one XCD and in its L2 from launch to launch).  Pp/partp: p and the rows'
// terms of p.v of step k-1 (read), Pc/partc: those of step k (written).  Dynamic LDS: 3 n
// doubles (v of step k, v and w of step k-1).  What a launch costs is its chain of latencies, not
// the matrix (9.7 MB at n = 1216, cache-resident): every global load that does not depend on
// another is issued first, and the two sums the reflector needs are shuffles and one barrier
// each (with tree reductions over the block, the partial sums read in a loop and rows that changed
// their XCD from column to column: 9.8 us a column at n = 1216; now 6.4).
constexpr int kHhVec = 6, kHhRow = 20;   // prefetched per thread: vector entries, row entries
__global__ __launch_bounds__(256) void k_hh_col(int n, int k, int b0, double* A, double* V, double* tau, double* d, double* e,
                                                const double* Pp, const double* partp, double* Pc, double* partc) {
    extern __shared__ double lds[];
    double* sv = lds;            // x of step k (absolute indices k+1..n-1)
    double* svp = lds + n;       // v_{k-1} (k..n-1)
    double* swp = lds + 2 * n;   // w_{k-1} (k..n-1)
    __shared__ double sh[8];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int m = n - k - 1;
    const int r = (blockIdx.x + b0) * 4 + wave, row = r - k - 1;
    const bool on = row >= 0 && row < m;
    const double* vp = V + (long)(k - 1) * n;
    const double* ak = A + (long)k * n;
    double* a = A + (long)r * n;
    double pa[kHhRow], pv[kHhVec], pw[kHhVec], px[kHhVec], ps[kHhVec];
#pragma unroll
    for (int c = 0; c < kHhVec; ++c) {
        const int j = k + 1 + tid + 256 * c;
        pv[c] = (k > 0 && j < n) ? vp[j] : 0.0;
        pw[c] = (k > 0 && j < n) ? Pp[j] : 0.0;
        px[c] = j < n ? ak[j] : 0.0;
        ps[c] = (k > 0 && j <= n) ? partp[j - k - 1] : 0.0;   // step k-1 had n - k rows
    }
#pragma unroll
    for (int c = 0; c < kHhRow; ++c) {
        const int j = k + 1 + lane + 64 * c;
        pa[c] = (on && j < n) ? a[j] : 0.0;
    }
    double K = 0.0, vk = 0.0, wk = 0.0;
    if (k > 0) {
        double s = 0.0;
#pragma unroll
        for (int c = 0; c < kHhVec; ++c) s += ps[c];
        for (int j = tid + 256 * kHhVec; j <= m; j += 256) s += partp[j];
        vk = vp[k];
        wk = Pp[k];
        s = wave_total(s);
        if (lane == 0) sh[wave] = s;
        __syncthreads();
        K = 0.5 * tau[k - 1] * ((sh[0] + sh[1]) + (sh[2] + sh[3]));
        wk -= K * vk;
    }
    // row k of the matrix after step k-1, and reflector k from it
    double s2 = 0.0;
    auto entry = [&](int j, double v, double p, double x) {
        const double w = p - K * v;
        x = k > 0 ? x - (vk * w + wk * v) : x;
        svp[j] = v;
        swp[j] = w;
        sv[j] = x;
        s2 = fma(x, x, s2);
    };
#pragma unroll
    for (int c = 0; c < kHhVec; ++c) {
        const int j = k + 1 + tid + 256 * c;
        if (j < n) entry(j, pv[c], pw[c], px[c]);
    }
    for (int j = k + 1 + tid + 256 * kHhVec; j < n; j += 256) entry(j, k > 0 ? vp[j] : 0.0, k > 0 ? Pp[j] : 0.0, ak[j]);
    s2 = wave_total(s2);
    if (lane == 0) sh[4 + wave] = s2;
    __syncthreads();
    const double x0 = sv[k + 1];
    double alpha, v0, t;
    hh_reflector((sh[4] + sh[5]) + (sh[6] + sh[7]), x0, alpha, v0, t);
    if (blockIdx.x == 0) {
        double* vrow = V + (long)k * n;
        for (int j = k + 1 + tid; j < n; j += 256) vrow[j] = j == k + 1 ? v0 : sv[j];
        if (tid == 0) {
            tau[k] = t;
            d[k] = k > 0 ? ak[k] - (vk * wk + wk * vk) : ak[k];
            e[k] = t == 0.0 ? x0 : alpha;
        }
    }
    // the block's trailing rows: update of step k-1, then p of step k
    if (!on) return;   // whole wave
    double acc = 0.0;
    const double vr = svp[r], wr = swp[r];
    auto step = [&](int j, double x) {
        if (k > 0) {
            x -= vr * swp[j] + wr * svp[j];
            a[j] = x;
        }
        acc = fma(x, j == k + 1 ? v0 : sv[j], acc);
    };
#pragma unroll
    for (int c = 0; c < kHhRow; ++c) {
        const int j = k + 1 + lane + 64 * c;
        if (j < n) step(j, pa[c]);
    }
    for (int j = k + 1 + lane + 64 * kHhRow; j < n; j += 64) step(j, a[j]);
    acc = wave_total(acc);
    if (lane == 0) {
        const double pr = t * acc;
        Pc[r] = pr;
        partc[row] = pr * (row == 0 ? v0 : sv[r]);
    }
}

// The reduction of the trailing m = n - k0 <= kHhOneN rows (all of a small matrix) in one block, the
// matrix in the registers of its 8 waves: a column takes two barriers and two vectors through LDS
// instead of a launch, and every wave does the vector work (reflector, K, w) for itself.  After
// k0 > 0 column launches the update of step k0-1 is still to be applied (Pp, partp: its p and
// terms of p.v).  Row r lies in slot r / 32 of the 16 lanes (r / 4 % 8, r % 4) = (wave, row of
// lanes), column j in lane j % 16 of them: a sum over the columns is four DPP moves for four
// rows at once.  n = 133: 313 us (one row per wave, six moves each: 408 us; a launch per
// column: 0.77 ms).
constexpr int kHhOneN = 192, kHhSlots = kHhOneN / 32, kHhCols = kHhOneN / 16;
__global__ __launch_bounds__(512) void k_hh_one(int n, int k0, const double* __restrict__ A0, double* V, double* tau, double* d,
                                                double* e, const double* __restrict__ Pp, const double* __restrict__ partp) {
    __shared__ double sx[kHhOneN], sp[kHhOneN];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, m = n - k0;
    const int row0 = __builtin_amdgcn_readfirstlane(tid >> 6) * 4, row = row0 + (lane >> 4);
    double a[kHhSlots][kHhCols];
#pragma unroll
    for (int s = 0; s < kHhSlots; ++s)
#pragma unroll
        for (int c = 0; c < kHhCols; ++c) {
            const int r = 32 * s + row, j = col + 16 * c;
            a[s][c] = (r < m && j < m) ? A0[(long)(k0 + r) * n + k0 + j] : 0.0;
        }
    if (k0 > 0) {   // the update of step k0 - 1: its v into sx, its w into sp
        double t = 0.0;
        for (int j = lane; j < m; j += 64) t += partp[j];
        const double K = 0.5 * tau[k0 - 1] * wave_total(t);
        for (int j = tid; j < kHhOneN; j += 512) {
            const double v = j < m ? V[(long)(k0 - 1) * n + k0 + j] : 0.0;
            sx[j] = v;
            sp[j] = j < m ? Pp[k0 + j] - K * v : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < kHhSlots; ++s) {
            const double vr = sx[32 * s + row], wr = sp[32 * s + row];
#pragma unroll
            for (int c = 0; c < kHhCols; ++c) a[s][c] -= vr * sp[col + 16 * c] + wr * sx[col + 16 * c];
        }
        __syncthreads();
    }
    for (int j = tid; j < kHhOneN; j += 512) sp[j] = 0.0;
    V += (long)k0 * n + k0;
    tau += k0;
    d += k0;
    e += k0;
    for (int k = 0; k + 2 < m; ++k) {
#pragma unroll
        for (int s = 0; s < kHhSlots; ++s)
            if (32 * s + row == k) {
#pragma unroll
                for (int c = 0; c < kHhCols; ++c) sx[col + 16 * c] = a[s][c];
            }
        __syncthreads();
        // the entries up to k of v are zero: those columns and rows keep what they have
        double v[kHhCols], w[kHhCols], s2 = 0.0;
#pragma unroll
        for (int c = 0; c < kHhCols; ++c) {
            v[c] = col + 16 * c > k ? sx[col + 16 * c] : 0.0;
            s2 = fma(v[c], v[c], s2);
        }
        const double x0 = sx[k + 1], dk = sx[k];
        double alpha, v0, t;
        hh_reflector(row_total(s2), x0, alpha, v0, t);
#pragma unroll
        for (int c = 0; c < kHhCols; ++c)
            if (col + 16 * c == k + 1) v[c] = v0;
        if (tid < 16) {
#pragma unroll
            for (int c = 0; c < kHhCols; ++c)
                if (col + 16 * c > k && col + 16 * c < m) V[(long)k * n + col + 16 * c] = v[c];
            if (tid == 0) {
                tau[k] = t;
                d[k] = dk;
                e[k] = t == 0.0 ? x0 : alpha;
            }
        }
#pragma unroll
        for (int s = 0; s < kHhSlots; ++s) {
            if (32 * s + row0 + 3 > k && 32 * s + row0 < m) {   // the same in the wave
                double acc = 0.0;
#pragma unroll
                for (int c = 0; c < kHhCols; ++c) acc = fma(a[s][c], v[c], acc);
                acc = t * row_total(acc);
                if (col == 0) sp[32 * s + row] = acc;
            }
        }
        double vr[kHhSlots];
#pragma unroll
        for (int s = 0; s < kHhSlots; ++s) {
            const int r = 32 * s + row;
            vr[s] = r == k + 1 ? v0 : r > k ? sx[r] : 0.0;
        }
        __syncthreads();
        double pv = 0.0;
#pragma unroll
        for (int c = 0; c < kHhCols; ++c) {
            w[c] = col + 16 * c > k ? sp[col + 16 * c] : 0.0;
            pv = fma(w[c], v[c], pv);
        }
        const double K = 0.5 * t * row_total(pv);
#pragma unroll
        for (int c = 0; c < kHhCols; ++c) w[c] -= K * v[c];
#pragma unroll
        for (int s = 0; s < kHhSlots; ++s)
            if (32 * s + row0 + 3 > k && 32 * s + row0 < m) {
                const int r = 32 * s + row;
                const double wr = r > k ? sp[r] - K * vr[s] : 0.0;
#pragma unroll
                for (int c = 0; c < kHhCols; ++c) a[s][c] -= vr[s] * w[c] + wr * v[c];
            }
    }
#pragma unroll
    for (int s = 0; s < kHhSlots; ++s) {
        const int r = 32 * s + row;
#pragma unroll
        for (int c = 0; c < kHhCols; ++c) {
            const int j = col + 16 * c;
            if (r < m && r == j && r >= m - 2) d[r] = a[s][c];
            if (r == m - 1 && j == m - 2) e[j] = a[s][c];
        }
    }
    if (tid == 0) e[m - 1] = 0.0;
    for (int j = n + tid; j < eig_pad(n); j += 512) d[j - k0] = e[j - k0] = 0.0;
}

// dynamic LDS above 64 KB has to be allowed; always the same `top`, so that threads with different
// sizes do not lower it for each other
constexpr size_t kLdsMax = 160 * 1024;   // of a block
static hipError_t lds_limit(const void* kernel, size_t bytes, size_t top) {
    if (bytes <= 64 * 1024) return hipSuccess;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)std::max(bytes, top));
}

static constexpr size_t hh_col_bytes(int n) { return 3 * (size_t)n * sizeof(double); }

hipError_t householder_tridiag(int n, EigWork& w, hipStream_t st) {
    if (n < 3 || n > kEigMaxN) return hipErrorInvalidValue;   // the callers solve n <= 2 in closed form
    // reflector rows must be zero outside their support for the blocked back-transform
    UNO_LAUNCH_FILL((long)n * n, w.V, st);
    // column launches down to the size that one block's registers hold: a whole solve of 192 takes
    // 0.90 ms; of 193, 1.12, and 1.54 by column launches to the end
    const int k1 = std::max(0, n - kHhOneN);
    // the inverse-iteration work space is unused until the tridiagonal is done: p and the
    // rows' terms of p.v of the steps of even and odd k live there
    double* P[2] = {w.wk, w.wk + n};
    double* part[2] = {w.wk + 2L * n, w.wk + 3L * n};
    const size_t lds = hh_col_bytes(n);
    if (k1 > 0)
        if (hipError_t er = lds_limit(reinterpret_cast<const void*>(&k_hh_col), lds, hh_col_bytes(kEigMaxN))) return er;
    for (int k = 0; k < k1; ++k) {
        const int b0 = (k + 1) / 32 * 8;
        hipLaunchKernelGGL(k_hh_col, dim3((unsigned)((n + 3) / 4 - b0)), dim3(256), lds, st, n, k, b0, w.A, w.V, w.tau, w.d, w.e,
                           P[(k + 1) & 1], part[(k + 1) & 1], P[k & 1], part[k & 1]);
    }
    hipLaunchKernelGGL(k_hh_one, dim3(1), dim3(512), 0, st, n, k1, (const double*)w.A, w.V, w.tau, w.d, w.e,
                       (const double*)P[(k1 + 1) & 1], (const double*)part[(k1 + 1) & 1]);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Back-transform Z <- H_0 H_1 ... H_{n-3} Z by blocks of kWy reflectors in compact WY form
// (H_k0 ... H_k1-1 = I - Vb^T T Vb with the reflectors as the rows of Vb and T upper
// triangular), the last block first: Z <- Z - Vb^T (M Z) with M = T Vb.  One launch forms
// every block's M (S = Vb Vb^T, the T recurrence and T Vb, one workgroup per block); then
// two MFMA GEMMs per block.
// ---------------------------------------------------------------------------
constexpr int kWy = 32;

// T[j][j] = tau_j, T[0:j][j] = -tau_j T[0:j][0:j] S[0:j][j], S = Vb Vb^T; M = T Vb
__global__ __launch_bounds__(256) void k_wy_m(int n, int nref, const double* __restrict__ V,
                                              const double* __restrict__ tau, double* __restrict__ M) {
    __shared__ double sS[kWy][kWy + 1];
    __shared__ double sT[kWy][kWy + 1];
    __shared__ double sV[kWy][65];
    const int k0 = blockIdx.x * kWy, nb = min(kWy, nref - k0);
    const double* Vb = V + (long)k0 * n;
    const int t = threadIdx.x;
    // S, in column chunks of 64 staged in LDS; thread t owns entries (l, j) = t / 32 + 8 q, t % 32
    double acc[4] = {0.0, 0.0, 0.0, 0.0};
    for (int c0 = 0; c0 < n; c0 += 64) {
        for (int q = t; q < kWy * 64; q += 256) {
            const int l = q / 64, c = q % 64;
            sV[l][c] = (l < nb && c0 + c < n) ? Vb[(long)l * n + c0 + c] : 0.0;
        }
        __syncthreads();
        const int j = t % kWy;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int l = t / kWy + 8 * q;
            double s = acc[q];
            for (int c = 0; c < 64; ++c) s = fma(sV[l][c], sV[j][c], s);
            acc[q] = s;
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) sS[t / kWy + 8 * q][t % kWy] = acc[q];
    for (int q = t; q < kWy * (kWy + 1); q += 256) sT[q / (kWy + 1)][q % (kWy + 1)] = 0.0;
    __syncthreads();
    for (int j = 0; j < nb; ++j) {
        if (t < j) {
            double s = 0.0;
            for (int l = t; l < j; ++l) s = fma(sT[t][l], sS[l][j], s);
            sT[t][j] = -tau[k0 + j] * s;
        }
        if (t == j) sT[j][j] = tau[k0 + j];
        __syncthreads();
    }
    // M = T Vb (nb x n), thread per column
    double* Mb = M + (long)k0 * n;
    for (int c = t; c < n; c += 256) {
        double v[kWy];
#pragma unroll
        for (int j2 = 0; j2 < kWy; ++j2) v[j2] = j2 < nb ? Vb[(long)j2 * n + c] : 0.0;
#pragma unroll 4
        for (int l = 0; l < nb; ++l) {
            double s = 0.0;
#pragma unroll
            for (int j2 = 0; j2 < kWy; ++j2) s = fma(sT[l][j2], v[j2], s);
            Mb[(long)l * n + c] = s;
        }
    }
}

// The reflectors applied one by one, a wave per column of Z with the column in registers and the
// next reflectors' rows read ahead: for n <= kHhOneN the whole back-transform is one launch of
// n - 2 steps of a few hundred cycles.  n = 133: 33 us (57 us for the blocks' T and 11 us for each of
// their ten GEMMs before).
__global__ __launch_bounds__(64) void k_apply_q_one(int n, const double* __restrict__ V, const double* __restrict__ tau,
                                                    double* __restrict__ Z) {
    constexpr int C = kHhOneN / 64, kAhead = 4;
    const int i = blockIdx.x, lane = threadIdx.x;
    double z[C], v[kAhead][C];
#pragma unroll
    for (int c = 0; c < C; ++c) z[c] = lane + 64 * c < n ? Z[(long)(lane + 64 * c) * n + i] : 0.0;
    auto read = [&](int k, double* r) {
#pragma unroll
        for (int c = 0; c < C; ++c) r[c] = (k >= 0 && lane + 64 * c < n) ? V[(long)k * n + lane + 64 * c] : 0.0;
    };
    const int k1 = n - 3;
#pragma unroll
    for (int q = 0; q < kAhead; ++q) read(k1 - q, v[q]);
    for (int k = k1; k >= 0; k -= kAhead) {
#pragma unroll
        for (int q = 0; q < kAhead; ++q) {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < C; ++c) s = fma(v[q][c], z[c], s);
            s = wave_total(s) * (k >= q ? tau[max(k - q, 0)] : 0.0);
#pragma unroll
            for (int c = 0; c < C; ++c) z[c] = fma(-s, v[q][c], z[c]);
            read(k - q - kAhead, v[q]);
        }
    }
#pragma unroll
    for (int c = 0; c < C; ++c)
        if (lane + 64 * c < n) Z[(long)(lane + 64 * c) * n + i] = z[c];
}

hipError_t apply_q(int n, EigWork& w, double* Z, hipStream_t st) {
    const int nref = n - 2;
    if (nref <= 0) return hipSuccess;
    if (n <= kHhOneN) {
        hipLaunchKernelGGL(k_apply_q_one, dim3((unsigned)n), dim3(64), 0, st, n, (const double*)w.V, (const double*)w.tau, Z);
        return hipGetLastError();
    }
    const int nblk = (nref + kWy - 1) / kWy;
    double* M = w.wk;                      // nref x n
    double* wy = w.wk + (long)nref * n;    // at most kWy x n
    hipLaunchKernelGGL(k_wy_m, dim3((unsigned)nblk), dim3(256), 0, st, n, nref, w.V, w.tau, M);
    for (int b = nblk - 1; b >= 0; --b) {
        const int k0 = b * kWy, nb = std::min(kWy, nref - k0);
        const double* Vb = w.V + (long)k0 * n;
        hipError_t e;
        if ((e = gemm_f64(false, false, nb, n, n, 1.0, M + (long)k0 * n, n, Z, n, 0.0, wy, n, st))) return e;
        if ((e = gemm_f64(true, false, n, n, nb, -1.0, Vb, n, wy, n, 1.0, Z, n, st))) return e;
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Tridiagonal eigenvalues by multisection on Sturm counts: one wave per eigenvalue.  The
// 64 lanes count at 64 interior points of the current interval at once, so each round
// narrows it 65-fold (about 9 rounds to full precision instead of 55 bisection steps);
// the search starts from the Gershgorin interval and stops at the same width as plain
// bisection would (2 eps max|end| + 4 pivmin).
// ---------------------------------------------------------------------------
// 1/a to rounding from the hardware estimate and two Newton steps; 1e-300 <= |a|, finite (0 where 1/a is subnormal)
__device__ __forceinline__ double recip(double a) {
    double r = __builtin_amdgcn_rcp(a);
    r = fma(fma(-a, r, 1.0), r, r);
    return fma(fma(-a, r, 1.0), r, r);
}

// (the loop is one chain of dependent operations: the quotient is a reciprocal and a product, half
// the length of a divide: 0.83 ms instead of 1.19 at n = 1216.  |q| stays between pivmin >= 1e-300 and 1 / 2.2e-308, which recip takes)
__device__ __forceinline__ int sturm_count(int n, const double* d, const double* e2, double x, double pivmin) {
    int c = 0;
    double q = d[0] - x;
    if (fabs(q) < pivmin) q = -pivmin;
    if (q < 0.0) ++c;
#pragma unroll 8
    for (int k = 1; k < n; ++k) {
        q = fma(-e2[k - 1], recip(q), d[k] - x);
        if (fabs(q) < pivmin) q = -pivmin;
        if (q < 0.0) ++c;
    }
    return c;
}

__device__ __forceinline__ double wave_min(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmin(v, __shfl_xor(v, o, 64));
    return v;
}
__device__ __forceinline__ double wave_max(double v) {
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
    return v;
}

// four eigenvalues per block (one per wave); d and e^2 staged in LDS
__global__ __launch_bounds__(256) void k_bisect(int n, const double* __restrict__ dg, const double* __restrict__ eg,
                                                double* __restrict__ evals) {
    extern __shared__ double sm[];
    double* d = sm;
    double* e2 = sm + n;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        d[k] = dg[k];
        e2[k] = (k + 1 < n) ? eg[k] * eg[k] : 0.0;
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int i = blockIdx.x * 4 + (threadIdx.x >> 6);   // eigenvalue of this wave
    if (i >= n) return;                                  // whole wave
    double lo = 1e300, hi = -1e300, emax = 0.0;
    for (int k = lane; k < n; k += 64) {
        const double r = (k > 0 ? sqrt(e2[k - 1]) : 0.0) + (k + 1 < n ? sqrt(e2[k]) : 0.0);
        lo = fmin(lo, d[k] - r);
        hi = fmax(hi, d[k] + r);
        emax = fmax(emax, e2[k]);
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    emax = wave_max(emax);
    const double tnorm = fmax(fabs(lo), fabs(hi));
    const double pivmin = 1e-300 + 2.2250738585072014e-308 * fmax(1.0, emax);
    lo -= 2.2e-16 * tnorm * n + pivmin;
    hi += 2.2e-16 * tnorm * n + pivmin;
    for (int it = 0; it < 64; ++it) {
        if (hi - lo <= 2.0 * 2.2204460492503131e-16 * fmax(fabs(lo), fabs(hi)) + 4.0 * pivmin) break;
        const double h = (hi - lo) / 65.0;
        double x = lo + h * (lane + 1);
        if (lane == 63 || x >= hi) x = fmin(x, hi);
        // points past rounding collapse onto hi count like hi: the count there is > i
        const bool above = x >= hi || sturm_count(n, d, e2, x, pivmin) > i;
        const unsigned long long m = __ballot(above);
        // counts are monotone in x: the first lane above brackets the eigenvalue
        const int f = m ? __builtin_ctzll(m) : 64;
        const double nlo = f == 0 ? lo : __shfl(x, f - 1, 64);
        const double nhi = f == 64 ? hi : __shfl(x, f, 64);
        if (!(nlo > lo || nhi < hi)) break;   // no progress left in double precision
        lo = nlo;
        hi = nhi;
    }
    if (lane == 0) evals[i] = 0.5 * (lo + hi);
}

// ---------------------------------------------------------------------------
// Inverse iteration: a thread solves (T - lambda_i I) x = b three times with a partially pivoted
// LU of the tridiagonal (tiny pivots replaced by eps*|T|), from a pseudo-random start vector
// seeded by i; the output Yt holds eigenvector i in column i (Yt[k n + i]).  Every work array is in
// LDS, `lanes` eigenvectors per one-wave block: the factors'
// reciprocal pivots and multipliers and the vector itself.  A row interchange is one bit; the
// superdiagonals of U follow from d, e, the bits and the multipliers.  The solves are chains of
// dependent operations, so rows go in
// chunks of 16, padded with rows that do nothing (d and e are padded with zeros), whose operands
// are read ahead of the chain, without branches; the scaling of one solve is done by the next
// one's loads.  T - lam is scaled by a power of two to norm 1, which keeps every pivot
// within the range of recip.  n = 1216: 0.63 ms, n = 133: 79 us (with the arrays in global memory and
// divides: 2.07 ms and 237 us).
constexpr size_t kInvLds = 156 * 1024;
static constexpr size_t inviter_bytes(int n) {   // LDS of one eigenvector
    const size_t np = eig_pad(n);
    return (3 * np + 1) * sizeof(double) + (np / kEigChunk + 1) / 2 * sizeof(double);
}
__global__ __launch_bounds__(64) void k_inviter_lds(int n, int lanes, const double* __restrict__ d,
                                                    const double* __restrict__ e, const double* __restrict__ evals,
                                                    double* __restrict__ Yt) {
    extern __shared__ double lds[];
    constexpr int kCh = kEigChunk;
    const int S = lanes, t = threadIdx.x, i = blockIdx.x * lanes + t, np = eig_pad(n);
    double tnorm = 0.0;
    for (int k = t; k < n; k += 64)
        tnorm = fmax(tnorm, fabs(d[k]) + (k + 1 < n ? fabs(e[k]) : 0.0) + (k > 0 ? fabs(e[k - 1]) : 0.0));
    tnorm = wave_max(tnorm);
    if (t >= lanes || i >= n) return;
    double* U1 = lds + t;                      // [k S]: reciprocal of the diagonal of U
    double* L = U1 + (long)np * S;             // multipliers
    double* x = L + (long)np * S;              // np + 1 entries
    unsigned* piv = reinterpret_cast<unsigned*>(lds + (3L * np + 1) * S) + t;   // [chunk S]
    const double sc = tnorm > 0.0 ? ldexp(1.0, -max(ilogb(tnorm), -1000)) : 1.0;
    const double lam = evals[i] * sc;
    const double tiny = tnorm > 0.0 ? 2.2204460492503131e-16 * (tnorm * sc) : 2.2204460492503131e-16;
    // factor T - lam I = P L U, row by row
    double a = d[0] * sc - lam, b = e[0] * sc;
    for (int k0 = 0; k0 < np; k0 += kCh) {
        double ds[kCh], es[kCh + 1];
        const bool last = k0 + kCh >= np;
#pragma unroll
        for (int c = 0; c < kCh; ++c) es[c] = e[k0 + c] * sc;
#pragma unroll
        for (int c = 0; c + 1 < kCh; ++c) ds[c] = d[k0 + c + 1] * sc - lam;
        es[kCh] = last ? 0.0 : e[last ? 0 : k0 + kCh] * sc;
        ds[kCh - 1] = last ? 0.0 : d[last ? 0 : k0 + kCh] * sc - lam;
        unsigned bits = 0;
        double u1[kCh], ls[kCh];
#pragma unroll
        for (int c = 0; c < kCh; ++c) {
            const double sub = es[c];
            const bool swap = !(fabs(a) >= fabs(sub));
            const double num = swap ? a : sub, u = swap ? sub : a;
            const double p = fabs(u) < tiny ? copysign(tiny, u) : u;
            const double rp = recip(p);
            double l = num * rp;
            l = fma(fma(-l, p, num), rp, l);
            const double up = swap ? ds[c] : b, dn = swap ? b : ds[c], en = es[c + 1];
            a = dn - l * up;
            b = swap ? -l * en : en;
            u1[c] = rp;
            ls[c] = l;
            bits |= swap ? 1u << c : 0u;
        }
        if (last) {   // the rows from n on do nothing, and row n - 1 has no successor
#pragma unroll
            for (int c = 0; c < kCh; ++c) {
                if (k0 + c >= n) u1[c] = 0.0;
                if (k0 + c >= n - 1) ls[c] = 0.0;
            }
            bits &= (1u << (n - 1 - k0)) - 1;
        }
#pragma unroll
        for (int c = 0; c < kCh; ++c) {
            U1[(k0 + c) * S] = u1[c];
            L[(k0 + c) * S] = ls[c];
        }
        piv[k0 / kCh * S] = bits;
    }
    // start vector
    unsigned int h = 2654435761u * (unsigned)(i + 1);
    for (int k = 0; k < n; ++k) {
        h ^= h << 13; h ^= h >> 17; h ^= h << 5;
        x[k * S] = ((double)(h & 0xffffff) / 16777216.0) - 0.5 + 1e-3;
    }
    for (int k = n; k <= np; ++k) x[k * S] = 0.0;
    double nrm = 1.0;
    for (int it = 0; it < 3; ++it) {
        // forward: apply the row interchanges and multipliers
        double xk = x[0] * nrm;
        for (int k0 = 0; k0 < np; k0 += kCh) {
            double xs[kCh], ls[kCh];
            const unsigned bits = piv[k0 / kCh * S];
#pragma unroll
            for (int c = 0; c < kCh; ++c) {
                xs[c] = x[(k0 + c + 1) * S] * nrm;
                ls[c] = L[(k0 + c) * S];
            }
#pragma unroll
            for (int c = 0; c < kCh; ++c) {
                const bool swap = bits >> c & 1;
                const double xn = xs[c], hi = swap ? xk : xn, lo = swap ? xn : xk;
                xs[c] = lo;
                xk = hi - ls[c] * lo;
            }
#pragma unroll
            for (int c = 0; c < kCh; ++c) x[(k0 + c) * S] = xs[c];
        }
        // back substitution with the banded U, then the norm
        double x1 = 0.0, x2 = 0.0, s2 = 0.0;
        for (int k0 = np - kCh; k0 >= 0; k0 -= kCh) {
            double xs[kCh], u1[kCh], u2[kCh], u3[kCh];
            // bit c + 1: row k0 + c was interchanged; bit 0: the row before the chunk
            const int before = k0 ? 1 : 0;
            const unsigned bits = piv[k0 / kCh * S] << 1 | before * (piv[(k0 / kCh - before) * S] >> (kCh - 1));
            double lp = L[(k0 - before) * S];
            const bool last = k0 + kCh >= np;
#pragma unroll
            for (int c = 0; c < kCh; ++c) {
                xs[c] = x[(k0 + c) * S];
                u1[c] = U1[(k0 + c) * S];
                const int k1 = last && c + 1 == kCh ? 0 : k0 + c + 1;   // past the end: not used
                const double dn = d[k1] * sc - lam, ec = e[k0 + c] * sc, en = last && c + 1 == kCh ? 0.0 : e[k1] * sc;
                const double ub = (bits >> c & 1) ? -lp * ec : ec;
                const bool swap = bits >> (c + 1) & 1;
                u2[c] = swap ? dn : ub;
                u3[c] = swap ? en : 0.0;
                lp = L[(k0 + c) * S];
            }
#pragma unroll
            for (int c = kCh - 1; c >= 0; --c) {
                const double v = ((xs[c] - u2[c] * x1) - u3[c] * x2) * u1[c];
                xs[c] = v;
                s2 = fma(v, v, s2);
                x2 = x1;
                x1 = v;
            }
#pragma unroll
            for (int c = 0; c < kCh; ++c) x[(k0 + c) * S] = xs[c];
        }
        nrm = 1.0 / sqrt(s2);
    }
#pragma unroll 8
    for (int k = 0; k < n; ++k) Yt[(long)k * n + i] = x[k * S] * nrm;
}

// modified Gram-Schmidt (two passes) inside each cluster of close eigenvalues (columns
// of Yt): clusters[2c], clusters[2c+1] = first and one-past-last index; one block per
// cluster
__global__ __launch_bounds__(256) void k_cluster_mgs(int n, const int* __restrict__ clusters, double* __restrict__ Yt) {
    __shared__ double red[256];
    const int c0 = clusters[2 * blockIdx.x], c1 = clusters[2 * blockIdx.x + 1];
    for (int j = c0; j < c1; ++j) {
        double* yj = Yt + j;
        for (int pass = 0; pass < 2; ++pass) {
            for (int p = c0; p < j; ++p) {
                const double* yp = Yt + p;
                double s = 0.0;
                for (int k = threadIdx.x; k < n; k += blockDim.x) s = fma(yj[(long)k * n], yp[(long)k * n], s);
                red[threadIdx.x] = s;
                __syncthreads();
                for (int o = 128; o > 0; o >>= 1) {
                    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
                    __syncthreads();
                }
                const double dot = red[0];
                __syncthreads();
                for (int k = threadIdx.x; k < n; k += blockDim.x) yj[(long)k * n] -= dot * yp[(long)k * n];
                __syncthreads();
            }
        }
        double s = 0.0;
        for (int k = threadIdx.x; k < n; k += blockDim.x) s = fma(yj[(long)k * n], yj[(long)k * n], s);
        red[threadIdx.x] = s;
        __syncthreads();
        for (int o = 128; o > 0; o >>= 1) {
            if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
            __syncthreads();
        }
        const double inv = 1.0 / sqrt(red[0]);
        __syncthreads();
        for (int k = threadIdx.x; k < n; k += blockDim.x) yj[(long)k * n] *= inv;
        __syncthreads();
    }
}

// the largest matrix: one eigenvector's solves, and the column launches' three vectors, in a block's LDS
static_assert(inviter_bytes(kEigMaxN) <= kLdsMax && inviter_bytes(kEigMaxN + 1) > kLdsMax, "one eigenvector per block");
static_assert(kEigMaxN == eig_pad(kEigMaxN) && hh_col_bytes(kEigMaxN) + 64 <= kLdsMax, "a column launch's vectors");

// doubles of EigWork::wk that a solve of this size uses: p and p.v of the column launches, and the
// blocked back-transform's rows (at most 5 n^2 for every n >= 3)
size_t eig_work_doubles(int n) {
    return std::max((size_t)n * n + (size_t)std::min(kWy, n) * n, 4 * (size_t)n);
}

hipError_t tridiag_eigen(int n, EigWork& w, int nclusters, const int* clusters, hipStream_t st) {
    if (n > kEigMaxN) return hipErrorInvalidValue;
    if (nclusters < 0) {
        const size_t lds = 2 * (size_t)n * sizeof(double);
        if (hipError_t er = lds_limit(reinterpret_cast<const void*>(&k_bisect), lds, 2 * kEigMaxN * sizeof(double))) return er;
        hipLaunchKernelGGL(k_bisect, dim3((unsigned)((n + 3) / 4)), dim3(256), lds, st, n, w.d, w.e, w.evals);
        return hipGetLastError();
    }
    // as many eigenvectors per block as LDS holds, but no fewer blocks than compute units
    const int fit = (int)std::min<size_t>(64, std::max<size_t>(1, kInvLds / inviter_bytes(n)));
    const int lanes = std::max(1, std::min(fit, (n + 255) / 256));
    const size_t lds = (size_t)lanes * inviter_bytes(n);
    if (hipError_t er = lds_limit(reinterpret_cast<const void*>(&k_inviter_lds), lds, kLdsMax)) return er;
    hipLaunchKernelGGL(k_inviter_lds, dim3((unsigned)((n + lanes - 1) / lanes)), dim3(64), lds, st, n, lanes,
                       (const double*)w.d, (const double*)w.e, (const double*)w.evals, w.Y);
    if (nclusters > 0) hipLaunchKernelGGL(k_cluster_mgs, dim3((unsigned)nclusters), dim3(256), 0, st, n, clusters, w.Y);
    return hipGetLastError();
}

}  // namespace uno

namespace uno {
// plain streaming copy of known size: calibrates the HBM traffic counters
__global__ __launch_bounds__(256) void k_copy_probe(long n, const double4* __restrict__ a, double4* __restrict__ b) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) b[i] = a[i];
}
hipError_t copy_probe(size_t bytes, int reps, float* ms, hipStream_t st) {
    const long n = (long)(bytes / sizeof(double4));
    double4 *a = nullptr, *b = nullptr;
    hipError_t e;
    if ((e = hipMalloc(&a, n * sizeof(double4))) != hipSuccess) return e;
    if ((e = hipMalloc(&b, n * sizeof(double4))) != hipSuccess) { (void)hipFree(a); return e; }
    (void)hipMemsetAsync(a, 0, n * sizeof(double4), st);
    hipEvent_t e0, e1;
    (void)hipEventCreate(&e0);
    (void)hipEventCreate(&e1);
    (void)hipEventRecord(e0, st);
    for (int r = 0; r < reps; ++r) hipLaunchKernelGGL(k_copy_probe, dim3(2048), dim3(256), 0, st, n, a, b);
    (void)hipEventRecord(e1, st);
    e = hipEventSynchronize(e1);
    (void)hipEventElapsedTime(ms, e0, e1);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    return e;
}
}  // namespace uno
