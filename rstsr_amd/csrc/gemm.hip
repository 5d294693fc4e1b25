// GEMM on gfx950: the matmul entry point with rstsr's batch-broadcast rules, the dispatch to the
// matrix-core tile kernel (gemm_tile.hpp: f32, f64, c64, c128) or the split GEMM (ozaki.hip), and
// a SIMT kernel for integers and for short products.
//
// Replaces DeviceMatMulAPI for DeviceFaer (rstsr-core/src/device_faer/matmul.rs:
// 19-239 -> faer) and the naive kernels of rstsr-native-impl/src/cpu_serial/
// matmul_naive.rs:78-122 (non-float types). Operand layouts map to (row stride,
// column stride) pairs directly, so no packing copy is made for any strided
// operand (the OpenBLAS device packs non-BLAS layouts, crates-device/
// rstsr-openblas/src/matmul_impl.rs:92-113; here the LDS tile load absorbs it).
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "registry.hpp"
#include "gemm.hpp"

#include <algorithm>
#include <functional>

namespace rstsr {
namespace hip {

template <class T>
struct GemmArgs {
    int64_t M, N, K;
    const T* a;
    int64_t rsa, csa;
    const T* b;
    int64_t rsb, csb;
    T* c;
    int64_t rsc, csc;
    T alpha, beta;
    int beta_zero;
    uint32_t tiles_m, tiles_n;
    uint32_t batch0;  // first batch index of this launch
    BatchDesc bd;
};

/* ---------------- SIMT kernel: i32, i64, short products ---------------- */

template <class T>
__device__ __forceinline__ T g_mul(T a, T b) {
    if constexpr (std::is_integral<T>::value) {
        using U = typename std::make_unsigned<T>::type;
        return (T)((U)a * (U)b);
    } else {
        return a * b;
    }
}
template <class T>
__device__ __forceinline__ T g_add(T a, T b) {
    if constexpr (std::is_integral<T>::value) {
        using U = typename std::make_unsigned<T>::type;
        return (T)((U)a + (U)b);
    } else {
        return a + b;
    }
}
__device__ __forceinline__ c64 g_mul(c64 a, c64 b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ c64 g_add(c64 a, c64 b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ c128 g_mul(c128 a, c128 b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ c128 g_add(c128 a, c128 b) { return {a.re + b.re, a.im + b.im}; }

template <class T>
__global__ void __launch_bounds__(256) k_gemm_simt(GemmArgs<T> g) {
    constexpr int TS = 16;
    __shared__ T As[TS][TS + 1];
    __shared__ T Bs[TS][TS + 1];
    const uint32_t tile = blockIdx.x;
    const uint32_t tm = tile / g.tiles_n, tn = tile % g.tiles_n;
    int64_t boa, bob, boc;
    batch_offsets(g.bd, g.batch0 + blockIdx.y, boa, bob, boc);
    const T* A = g.a + boa;
    const T* B = g.b + bob;
    T* C = g.c + boc;
    const int tx = threadIdx.x % TS, ty = threadIdx.x / TS;
    const int64_t gm = (int64_t)tm * TS + ty, gn = (int64_t)tn * TS + tx;
    T acc{};
    for (int64_t k0 = 0; k0 < g.K; k0 += TS) {
        int64_t ka = k0 + tx, kb = k0 + ty;
        As[ty][tx] = (gm < g.M && ka < g.K) ? A[gm * g.rsa + ka * g.csa] : T{};
        Bs[ty][tx] = (kb < g.K && gn < g.N) ? B[kb * g.rsb + gn * g.csb] : T{};
        __syncthreads();
#pragma unroll
        for (int k = 0; k < TS; ++k) acc = g_add(acc, g_mul(As[ty][k], Bs[k][tx]));
        __syncthreads();
    }
    if (gm < g.M && gn < g.N) {
        T* cp = C + gm * g.rsc + gn * g.csc;
        T v = g_mul(g.alpha, acc);
        if (!g.beta_zero) v = g_add(v, g_mul(g.beta, *cp));
        *cp = v;
    }
}

/* ---------------- host side ---------------- */

// The SIMT kernel: one output per thread, in pieces along the rows where a launch would hold more
// than 2^32 threads.
template <class T>
static void simt_gemm(rstsr_hip_ctx* ctx, const GemmProblem& P, T alpha, T beta, bool beta_zero) {
    GemmArgs<T> g;
    g.N = P.N;
    g.K = P.K;
    g.rsa = P.rsa;
    g.csa = P.csa;
    g.b = (const T*)P.b;
    g.rsb = P.rsb;
    g.csb = P.csb;
    g.rsc = P.rsc;
    g.csc = P.csc;
    g.alpha = alpha;
    g.beta = beta;
    g.beta_zero = beta_zero ? 1 : 0;
    g.bd = P.bd;
    g.tiles_n = ceil_div_u32(P.N, 16);
    const uint64_t YMAX = 65535, TMAX = (1ull << 24) - 1;
    if (g.tiles_n > TMAX) RSTSR_RAISE(UnImplemented, "GEMM grid too large");
    const int64_t step = (int64_t)(TMAX / g.tiles_n) * 16;
    for (int64_t m0 = 0; m0 < P.M; m0 += step) {
        g.M = std::min(step, P.M - m0);
        g.a = (const T*)P.a + m0 * P.rsa;
        g.c = (T*)P.c + m0 * P.rsc;
        g.tiles_m = ceil_div_u32(g.M, 16);
        for (uint64_t b0 = 0; b0 < P.nbatch; b0 += YMAX) {
            g.batch0 = (uint32_t)b0;
            const uint32_t nb = (uint32_t)std::min<uint64_t>(YMAX, P.nbatch - b0);
            hipLaunchKernelGGL(k_gemm_simt<T>, dim3(g.tiles_m * g.tiles_n, nb), dim3(256), 0, ctx->stream, g);
            check_launch("gemm");
        }
    }
}

// Short products with few rows or columns leave most of a matrix-core tile and of its 128-byte K
// slice empty. By sizes only, like the tile kernel's own choices (us, tile against SIMT: 10000 products of 4 x 4
// x 4 f32 31, 9, f64 29, 12, c128 34, 15, of 16 x 16 x 16 f64 33, 16; 200000 x 5 x 5 f32 23, 10, f64 23, 15; f32
// 5000 x 200 x 2 7.2, 5.4; but 200000 x 20 x 20 f32 18, 33, f64 24, 52; f32 1500 x 1500 x 4 8.0, 9.4). Complex
// symmetric products stay with the tile kernel, which makes them exactly symmetric.
template <class T>
static bool simt_pays(const GemmProblem& P) {
    constexpr bool CX = std::is_same<T, c64>::value || std::is_same<T, c128>::value;
    return P.K <= 16 && std::min(P.M, P.N) <= (sizeof(T) == 4 ? 256 : 16) && !(CX && P.a == P.b);
}

template <class T>
static void launch_gemm_t(rstsr_hip_ctx* ctx, const GemmProblem& P, T alpha, T beta, bool beta_zero,
                          const int* run_if = nullptr) {
    if constexpr (!std::is_integral<T>::value) {
        if (!run_if && simt_pays<T>(P)) {
            simt_gemm(ctx, P, alpha, beta, beta_zero);
            return;
        }
        // SYRK shortcut (device_faer/matmul.rs:38-48): beta = 0 and A is B's transpose
        // in the same buffer, so C is symmetric. Only the tiles on and below the
        // diagonal are multiplied, and stored twice. For real types C[i][j] and
        // C[j][i] sum the same products in the same K order, so the mirror equals the
        // full product bit for bit; for complex the imaginary part's two products
        // swap order, and the mirror makes the result exactly symmetric.
        if constexpr (std::is_same<T, float>::value) tile_gemm_f32(ctx, P, alpha, beta, beta_zero);
        else if constexpr (std::is_same<T, c64>::value) tile_gemm_c64(ctx, P, alpha, beta, beta_zero);
        else if constexpr (std::is_same<T, double>::value) tile_gemm_f64(ctx, P, alpha, beta, beta_zero, run_if);
        else tile_gemm_c128(ctx, P, alpha, beta, beta_zero, run_if);
    } else {
        simt_gemm(ctx, P, alpha, beta, beta_zero);
    }
}

void plain_dgemm(rstsr_hip_ctx* ctx, const GemmProblem& P, double alpha, double beta, bool beta_zero,
                 const int* run_if) {
    launch_gemm_t<double>(ctx, P, alpha, beta, beta_zero, run_if);
}


// Zero-fill C (k == 0 with beta == 0: crates-device/rstsr-openblas/src/matmul_impl.rs:78-81).
template <class T>
__global__ void k_scale_c(GemmArgs<T> g) {
    uint64_t idx = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    uint64_t mn = (uint64_t)g.M * g.N;
    if (idx >= mn) return;
    int64_t oa, ob, oc;
    batch_offsets(g.bd, g.batch0 + blockIdx.y, oa, ob, oc);
    int64_t m = idx / g.N, n = idx - (idx / g.N) * g.N;
    T* cp = g.c + oc + m * g.rsc + n * g.csc;
    *cp = g.beta_zero ? T{} : g_mul(g.beta, *cp);
}

template <class T>
static void scale_c(rstsr_hip_ctx* ctx, const GemmProblem& P, T beta, bool beta_zero) {
    GemmArgs<T> g{};
    g.M = P.M;
    g.N = P.N;
    g.c = (T*)P.c;
    g.rsc = P.rsc;
    g.csc = P.csc;
    g.beta = beta;
    g.beta_zero = beta_zero;
    g.bd = P.bd;
    uint64_t mn = (uint64_t)P.M * P.N;
    for (uint64_t b0 = 0; b0 < P.nbatch; b0 += 65535) {
        g.batch0 = (uint32_t)b0;
        uint32_t nb = (uint32_t)std::min<uint64_t>(65535, P.nbatch - b0);
        hipLaunchKernelGGL(k_scale_c<T>, dim3(ceil_div_u32(mn, 256), nb), dim3(256), 0, ctx->stream, g);
        check_launch("gemm scale");
    }
}

static bool is_zero_scalar(rstsr_dtype_t t, const void* v) {
    switch (t) {
        case RSTSR_F32: return *(const float*)v == 0.0f;
        case RSTSR_F64: return *(const double*)v == 0.0;
        case RSTSR_I32: return *(const int32_t*)v == 0;
        case RSTSR_I64: return *(const int64_t*)v == 0;
        case RSTSR_C64: return ((const float*)v)[0] == 0.0f && ((const float*)v)[1] == 0.0f;
        case RSTSR_C128: return ((const double*)v)[0] == 0.0 && ((const double*)v)[1] == 0.0;
        default: return false;
    }
}

// S (rows x cols, dense row-major) = Re X + Im X for a strided complex matrix X. run_if as for
// plain_dgemm.
__global__ void __launch_bounds__(256) k_zsum_parts(double* __restrict__ S, double* __restrict__ Xr,
                                                    double* __restrict__ Xi, const c128* __restrict__ X, int64_t rows,
                                                    int64_t cols, int64_t rs, int64_t cs,
                                                    const int* __restrict__ run_if) {
    if (run_if && *run_if == 0) return;
    // row blockIdx.y (grid-strided), columns along the block: S = re + im, and the real and
    // imaginary planes as contiguous rows (the split then reads them once, at unit stride)
    for (int64_t i = blockIdx.y; i < rows; i += gridDim.y) {
        const c128* xr = X + i * rs;
        const int64_t o = i * cols;
        for (int64_t j = (int64_t)blockIdx.x * 256 + threadIdx.x; j < cols; j += (int64_t)gridDim.x * 256) {
            const c128 x = xr[j * cs];
            S[o + j] = x.re + x.im;
            Xr[o + j] = x.re;
            Xi[o + j] = x.im;
        }
    }
}

// C holds (a T1, a T3) with T1 = Ar Br, T3 = (Ar + Ai)(Br + Bi); T2 = a Ai Bi (dense M x N).
// C = (a T1 - a T2, a T3 - a T1 - a T2).
__global__ void __launch_bounds__(256) k_z3m_combine(c128* __restrict__ C, int64_t rsc, int64_t csc,
                                                     const double* __restrict__ T2, int64_t M, int64_t N,
                                                     const int* __restrict__ run_if) {
    if (run_if && *run_if == 0) return;
    const int64_t n = M * N;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const int64_t i = e / N, j = e - i * N;
        c128* p = C + i * rsc + j * csc;
        const c128 c = *p;
        const double t2 = T2[e];
        *p = c128{c.re - t2, (c.im - c.re) - t2};
    }
}

// The three-product form of a complex product (ozaki_zgemm3) by real products of the parts, which
// lie in `z` (Zgemm3Parts): split products, or with run_if plain ones that run if *run_if != 0.
struct Zgemm3Parts {
    size_t nA, nB, nT;  // doubles, each a multiple of 256 bytes
    explicit Zgemm3Parts(const GemmProblem& P) {
        auto al = [](int64_t x) { return ((size_t)x + 31) & ~(size_t)31; };
        nA = al(P.M * P.K);
        nB = al(P.K * P.N);
        nT = al(P.M * P.N);
    }
    size_t bytes() const { return (3 * nA + 3 * nB + nT) * sizeof(double); }
};

static void zgemm3_products(rstsr_hip_ctx* ctx, const GemmProblem& P, double a, char* z, const int* run_if) {
    const int64_t M = P.M, N = P.N, K = P.K;
    // the sums Ar + Ai and Br + Bi, T2, and the four parts as contiguous planes
    const Zgemm3Parts s(P);
    double* SA = (double*)z;
    double* SB = SA + s.nA;
    double* T2 = SB + s.nB;
    double* Ar = T2 + s.nT;
    double* Ai = Ar + s.nA;
    double* Br = Ai + s.nA;
    double* Bi = Br + s.nB;
    // launches that may not run stay small
    const int64_t ymax = run_if ? 64 : 65535;
    auto grid = [&](int64_t rows, int64_t cols) {
        return dim3((uint32_t)std::min<int64_t>((cols + 255) / 256, 64), (uint32_t)std::min<int64_t>(rows, ymax));
    };
    hipLaunchKernelGGL(k_zsum_parts, grid(M, K), dim3(256), 0, ctx->stream, SA, Ar, Ai, (const c128*)P.a, M, K,
                       P.rsa, P.csa, run_if);
    hipLaunchKernelGGL(k_zsum_parts, grid(K, N), dim3(256), 0, ctx->stream, SB, Br, Bi, (const c128*)P.b, K, N,
                       P.rsb, P.csb, run_if);
    check_launch("complex split sums");
    GemmProblem Q = P;
    Q.bd.nbd = 0;
    Q.nbatch = 1;
    Q.rsa = K;
    Q.csa = 1;
    Q.rsb = N;
    Q.csb = 1;
    auto prod = [&](const double* x, const double* y, double* c, int64_t rsc, int64_t csc) {
        Q.a = x;
        Q.b = y;
        Q.c = c;
        Q.rsc = rsc;
        Q.csc = csc;
        if (run_if) plain_dgemm(ctx, Q, a, 0.0, true, run_if);
        else ozaki_gemm_f64(ctx, Q, a, 0.0, true);
    };
    prod(Ar, Br, (double*)P.c, 2 * P.rsc, 2 * P.csc);      // T1 into Re C
    prod(SA, SB, (double*)P.c + 1, 2 * P.rsc, 2 * P.csc);  // T3 into Im C
    prod(Ai, Bi, T2, N, 1);
    const size_t nT = (size_t)M * N;
    hipLaunchKernelGGL(k_z3m_combine, dim3((uint32_t)std::min<size_t>((nT + 255) / 256, run_if ? 4096 : 65536)),
                       dim3(256), 0, ctx->stream, (c128*)P.c, P.rsc, P.csc, T2, M, N, run_if);
    check_launch("complex split combine");
}

// Complex split GEMM from real split products. With beta = 0 and one matrix: the three-product form,
// in one run of the split kernels (ozaki_zgemm3) or, for the forms that does not take, one by one;
// otherwise four on the real/imaginary planes (stride-2 double views): Cr = a ArBr - a AiBi + b Cr,
// Ci = a ArBi + a AiBr + b Ci.
static void ozaki_zgemm(rstsr_hip_ctx* ctx, const GemmProblem& P, c128 alpha, c128 beta, bool beta_zero) {
    if (alpha.im != 0.0 || beta.im != 0.0)
        RSTSR_RAISE(UnImplemented, "the complex split GEMM takes real alpha and beta");
    if (beta_zero && P.nbatch == 1 && P.bd.nbd == 0 && P.K > 0) {
        const size_t bytes = Zgemm3Parts(P).bytes();
        if (!ozaki_zgemm3(ctx, P, alpha.re, bytes,
                          [&](const int* flag, char* ws) { zgemm3_products(ctx, P, alpha.re, ws, flag); }))
            zgemm3_products(ctx, P, alpha.re, (char*)zbuf_buffer(ctx, bytes), nullptr);
        return;
    }
    auto part = [&](const void* base, int im) { return (const void*)((const double*)base + im); };
    GemmProblem R = P;
    R.rsa *= 2;
    R.csa *= 2;
    R.rsb *= 2;
    R.csb *= 2;
    R.rsc *= 2;
    R.csc *= 2;
    for (int d = 0; d < R.bd.nbd; ++d) {
        R.bd.sa[d] *= 2;
        R.bd.sb[d] *= 2;
        R.bd.sc[d] *= 2;
    }
    const double a = alpha.re, b = beta.re;
    auto prod = [&](int ai, int bi, int ci, double al, double be, bool bz) {
        GemmProblem Q = R;
        Q.a = part(P.a, ai);
        Q.b = part(P.b, bi);
        Q.c = (void*)((double*)P.c + ci);
        ozaki_gemm_f64(ctx, Q, al, be, bz);
    };
    prod(0, 0, 0, a, b, beta_zero);   // Cr  = a Ar Br + b Cr
    prod(1, 1, 0, -a, 1.0, false);    // Cr -= a Ai Bi
    prod(0, 1, 1, a, b, beta_zero);   // Ci  = a Ar Bi + b Ci
    prod(1, 0, 1, a, 1.0, false);     // Ci += a Ai Br
}

// Merge batch axes into the matrix: the innermost batch axis folds into M when
// B is the same for every batch and A's and C's batch strides continue their
// row strides (sa = M rsa, sc = M rsc), so batch b row m is row b M + m of one
// taller product; likewise into N when A is shared and B and C chain along
// columns. One large GEMM instead of many, and no per-batch tile padding: the
// 60 x (400 x 24000 x 1600) RI contraction becomes one 24000 x 24000 x 1600
// product, the broadcast 64 x 1024^3 batch one 65536 x 1024 x 1024.
static GemmProblem fold_batches(const GemmProblem& P0) {
    GemmProblem P = P0;
    while (P.bd.nbd > 0) {
        const int64_t s = P.bd.shape[0];
        if (P.bd.sb[0] == 0 && P.bd.sa[0] == P.M * P.rsa && P.bd.sc[0] == P.M * P.rsc &&
            (uint64_t)(P.M * s) < (1ull << 40)) {
            P.M *= s;
        } else if (P.bd.sa[0] == 0 && P.bd.sb[0] == P.N * P.csb && P.bd.sc[0] == P.N * P.csc &&
                   (uint64_t)(P.N * s) < (1ull << 40)) {
            P.N *= s;
        } else {
            break;
        }
        for (int d = 1; d < P.bd.nbd; ++d) {
            P.bd.shape[d - 1] = P.bd.shape[d];
            P.bd.fd[d - 1] = P.bd.fd[d];
            P.bd.sa[d - 1] = P.bd.sa[d];
            P.bd.sb[d - 1] = P.bd.sb[d];
            P.bd.sc[d - 1] = P.bd.sc[d];
        }
        P.bd.nbd -= 1;
        P.nbatch /= (uint64_t)s;
    }
    return P;
}

void run_gemm(rstsr_hip_ctx* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, const GemmProblem& P0, const void* alpha,
              const void* beta) {
    if (!alpha || !beta) RSTSR_RAISE(InvalidValue, "null alpha/beta");
    if (P0.M == 0 || P0.N == 0 || P0.nbatch == 0) return;
    const GemmProblem P = fold_batches(P0);
    bool bz = is_zero_scalar(t, beta);
    if (mode != RSTSR_GEMM_PLAIN && mode != RSTSR_GEMM_OZAKI_INT8) RSTSR_RAISE(InvalidValue, "unknown GEMM mode");
    if (mode == RSTSR_GEMM_OZAKI_INT8 && t != RSTSR_F64 && t != RSTSR_C128)
        RSTSR_RAISE(UnImplemented, "the Ozaki split GEMM is provided for f64 and c128");
    auto body = [&](auto tag) {
        using T = decltype(tag);
        T al, be;
        std::memcpy(&al, alpha, sizeof(T));
        std::memcpy(&be, beta, sizeof(T));
        if (P.K == 0) {
            scale_c<T>(ctx, P, be, bz);
            return;
        }
        if constexpr (std::is_same<T, double>::value) {
            if (mode == RSTSR_GEMM_OZAKI_INT8) {
                ozaki_gemm_f64(ctx, P, al, be, bz);
                return;
            }
        }
        if constexpr (std::is_same<T, c128>::value) {
            if (mode == RSTSR_GEMM_OZAKI_INT8) {
                ozaki_zgemm(ctx, P, al, be, bz);
                return;
            }
        }
        if (gemv(ctx, t, P, alpha, beta, bz)) return;
        launch_gemm_t<T>(ctx, P, al, be, bz);
    };
    switch (t) {
        case RSTSR_F32: body(float{}); break;
        case RSTSR_F64: body(double{}); break;
        case RSTSR_I32: body(int32_t{}); break;
        case RSTSR_I64: body(int64_t{}); break;
        case RSTSR_C64: body(c64{}); break;
        case RSTSR_C128: body(c128{}); break;
        default: RSTSR_RAISE(UnImplemented, "matmul dtype");
    }
}

// Check that each operand's matrices of every batch stay inside its buffer.
static void check_gemm_extent(const GemmProblem& P, size_t es) {
    auto mk = [&](const void* p, int64_t r, int64_t cdim, int64_t rs, int64_t cs, const int64_t* bs, const char* nm) {
        size_t s[MAXD + 2];
        int64_t t[MAXD + 2];
        int nd = 0;
        for (int d = 0; d < P.bd.nbd; ++d, ++nd) {
            s[nd] = P.bd.shape[d];
            t[nd] = bs[d];
        }
        s[nd] = (size_t)r;
        t[nd++] = rs;
        s[nd] = (size_t)cdim;
        t[nd++] = cs;
        check_extent_rel(p, (size_t)nd, s, t, es, nm);
    };
    mk(P.a, P.M, P.K, P.rsa, P.csa, P.bd.sa, "a");
    mk(P.b, P.K, P.N, P.rsb, P.csb, P.bd.sb, "b");
    mk(P.c, P.M, P.N, P.rsc, P.csc, P.bd.sc, "c");
}

}  // namespace hip
}  // namespace rstsr

using namespace rstsr;
using namespace rstsr::hip;

extern "C" {

int rstsr_hip_gemm(rstsr_hip_ctx_t* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, size_t m, size_t n, size_t k,
                   const void* alpha, const void* a, ptrdiff_t rsa, ptrdiff_t csa, const void* b, ptrdiff_t rsb,
                   ptrdiff_t csb, const void* beta, void* c, ptrdiff_t rsc, ptrdiff_t csc) {
    return guarded([&] {
        bind(ctx);
        GemmProblem P{};
        P.M = (int64_t)m;
        P.N = (int64_t)n;
        P.K = (int64_t)k;
        P.a = a;
        P.rsa = rsa;
        P.csa = csa;
        P.b = b;
        P.rsb = rsb;
        P.csb = csb;
        P.c = c;
        P.rsc = rsc;
        P.csc = csc;
        P.bd.nbd = 0;
        P.nbatch = 1;
        check_gemm_extent(P, dtype_size(t));
        std::lock_guard<std::mutex> g(ctx->mu);
        run_gemm(ctx, t, mode, P, alpha, beta);
    });
}

// rstsr-common/src/layout/matmul.rs:287-421 (layout_matmul_dyn_row_major_with_lc):
// split each operand into (batch rest, matrix) and broadcast the batch rests
// of A and B to C's; vectors become 1 x K / K x 1 matrices.
int rstsr_hip_matmul(rstsr_hip_ctx_t* ctx, rstsr_dtype_t t, void* c, const rstsr_layout_t* lc_, const void* a,
                     const rstsr_layout_t* la_, const void* b, const rstsr_layout_t* lb_, const void* alpha,
                     const void* beta, rstsr_gemm_mode_t mode) {
    return guarded([&] {
        bind(ctx);
        Layout lc = from_abi(lc_), la = from_abi(la_), lb = from_abi(lb_);
        size_t na = la.ndim(), nb = lb.ndim(), nc = lc.ndim();
        if (na == 0 || nb == 0) RSTSR_RAISE(InvalidValue, "In matmul, 0-dim is not allowed.");
        // matrices as (shape, stride) pairs
        int64_t M, N, K, rsa, csa, rsb, csb, rsc, csc;
        Layout ra, rb, rc;  // batch rests
        auto split = [](const Layout& l, size_t nm, Layout& rest) {
            Shape s(l.shape.begin(), l.shape.end() - nm);
            Stride st(l.stride.begin(), l.stride.end() - nm);
            rest = Layout(s, st, 0);
        };
        if (na == 1 && nb == 1) {  // rule 1: inner dot -> 1 x 1
            if (la.shape != lb.shape || nc != 0) RSTSR_RAISE(InvalidLayout, "matmul rule 1 shape mismatch");
            M = 1;
            N = 1;
            K = la.shape[0];
            rsa = 0;
            csa = la.stride[0];
            rsb = lb.stride[0];
            csb = 0;
            rsc = 0;
            csc = 0;
            ra = rb = rc = Layout({}, {}, 0);
        } else if (na == 1) {  // rule 3: K @ (..., K, N) -> (..., N)
            if (nb != nc + 1 || la.shape[0] != lb.shape[nb - 2] || lc.shape[nc - 1] != lb.shape[nb - 1])
                RSTSR_RAISE(InvalidLayout, "matmul rule 3 shape mismatch");
            M = 1;
            K = la.shape[0];
            N = lb.shape[nb - 1];
            rsa = 0;
            csa = la.stride[0];
            rsb = lb.stride[nb - 2];
            csb = lb.stride[nb - 1];
            rsc = 0;
            csc = lc.stride[nc - 1];
            split(lb, 2, rb);
            split(lc, 1, rc);
            ra = Layout(rc.shape, Stride(rc.ndim(), 0), 0);
        } else if (nb == 1) {  // rule 4: (..., M, K) @ K -> (..., M)
            if (na != nc + 1 || lb.shape[0] != la.shape[na - 1] || lc.shape[nc - 1] != la.shape[na - 2])
                RSTSR_RAISE(InvalidLayout, "matmul rule 4 shape mismatch");
            M = la.shape[na - 2];
            K = la.shape[na - 1];
            N = 1;
            rsa = la.stride[na - 2];
            csa = la.stride[na - 1];
            rsb = lb.stride[0];
            csb = 0;
            rsc = lc.stride[nc - 1];
            csc = 0;
            split(la, 2, ra);
            split(lc, 1, rc);
            rb = Layout(rc.shape, Stride(rc.ndim(), 0), 0);
        } else {  // rules 2, 5, 6, 7
            if (nc < 2) RSTSR_RAISE(InvalidLayout, "matmul output rank");
            M = la.shape[na - 2];
            K = la.shape[na - 1];
            N = lb.shape[nb - 1];
            if (lb.shape[nb - 2] != (size_t)K || lc.shape[nc - 2] != (size_t)M || lc.shape[nc - 1] != (size_t)N)
                RSTSR_RAISE(InvalidLayout, "matmul shape mismatch");
            rsa = la.stride[na - 2];
            csa = la.stride[na - 1];
            rsb = lb.stride[nb - 2];
            csb = lb.stride[nb - 1];
            rsc = lc.stride[nc - 2];
            csc = lc.stride[nc - 1];
            split(la, 2, ra);
            split(lb, 2, rb);
            split(lc, 2, rc);
        }
        // broadcast batch rests of A and B to C's (broadcast_layout_to_first)
        ra = broadcast_layout_to_shape(ra, rc.shape, FlagOrder::RowMajor);
        rb = broadcast_layout_to_shape(rb, rc.shape, FlagOrder::RowMajor);
        GemmProblem P{};
        P.M = M;
        P.N = N;
        P.K = K;
        P.a = (const char*)a + la.offset * dtype_size(t);
        P.b = (const char*)b + lb.offset * dtype_size(t);
        P.c = (char*)c + lc.offset * dtype_size(t);
        P.rsa = rsa;
        P.csa = csa;
        P.rsb = rsb;
        P.csb = csb;
        P.rsc = rsc;
        P.csc = csc;
        // batch dims: drop size 1, innermost first for the unravel
        std::vector<size_t> bd;
        for (size_t i = 0; i < rc.ndim(); ++i)
            if (rc.shape[i] != 1) bd.push_back(i);
        if ((int)bd.size() > MAXD) RSTSR_RAISE(UnImplemented, "too many batch axes");
        P.bd.nbd = (int)bd.size();
        uint64_t nbat = 1;
        for (int d = 0; d < MAXD; ++d) {
            P.bd.shape[d] = 1;
            P.bd.fd[d] = FastDiv(1);
            P.bd.sa[d] = P.bd.sb[d] = P.bd.sc[d] = 0;
        }
        for (int d = 0; d < P.bd.nbd; ++d) {
            size_t ax = bd[bd.size() - 1 - d];
            if (rc.shape[ax] >= (1ull << 31)) RSTSR_RAISE(UnImplemented, "batch extent too large");
            P.bd.shape[d] = (uint32_t)rc.shape[ax];
            P.bd.fd[d] = FastDiv((uint32_t)rc.shape[ax]);
            P.bd.sa[d] = ra.stride[ax];
            P.bd.sb[d] = rb.stride[ax];
            P.bd.sc[d] = rc.stride[ax];
            nbat *= rc.shape[ax];
        }
        if (nbat >= (1ull << 32)) RSTSR_RAISE(UnImplemented, "too many batches");
        P.nbatch = nbat;
        if (lc.size() == 0) return;
        // extents (relative to the operand base pointers, offsets folded in)
        {
            size_t es = dtype_size(t);
            check_extent(a, la, es, "a");
            check_extent(b, lb, es, "b");
            check_extent(c, lc, es, "c");
        }
        std::lock_guard<std::mutex> g(ctx->mu);
        run_gemm(ctx, t, mode, P, alpha, beta);
    });
}

int rstsr_hip_gemm_grouped(rstsr_hip_ctx_t* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, size_t count,
                           const rstsr_gemm_desc_t* descs, const void* alpha, const void* beta) {
    return guarded([&] {
        bind(ctx);
        if (count && !descs) RSTSR_RAISE(InvalidValue, "null descriptors");
        if (!alpha || !beta) RSTSR_RAISE(InvalidValue, "null alpha/beta");
        size_t es = dtype_size(t);
        std::vector<GemmProblem> probs;
        for (size_t i = 0; i < count; ++i) {
            const auto& d = descs[i];
            GemmProblem P{};
            P.M = (int64_t)d.m;
            P.N = (int64_t)d.n;
            P.K = (int64_t)d.k;
            P.a = d.a;
            P.rsa = d.rsa;
            P.csa = d.csa;
            P.b = d.b;
            P.rsb = d.rsb;
            P.csb = d.csb;
            P.c = d.c;
            P.rsc = d.rsc;
            P.csc = d.csc;
            P.bd.nbd = 0;
            P.nbatch = 1;
            check_gemm_extent(P, es);
            if (P.M && P.N) probs.push_back(P);
        }
        std::lock_guard<std::mutex> g(ctx->mu);
        bool plain_mfma = mode == RSTSR_GEMM_PLAIN && (t == RSTSR_F64 || t == RSTSR_C128);
        std::vector<GemmProblem> rest;
        if (plain_mfma) {
            auto go = [&](auto tag) {
                using T = decltype(tag);
                T al, be;
                std::memcpy(&al, alpha, sizeof(T));
                std::memcpy(&be, beta, sizeof(T));
                std::vector<GemmProblem> gp;
                for (auto& P : probs) (P.K == 0 ? rest : gp).push_back(P);
                if constexpr (std::is_same<T, double>::value) tile_grouped_f64(ctx, gp, al, be, is_zero_scalar(t, beta), nullptr);
                else tile_grouped_c128(ctx, gp, al, be, is_zero_scalar(t, beta), nullptr);
            };
            if (t == RSTSR_F64) go(double{});
            else go(c128{});
        } else if (mode == RSTSR_GEMM_OZAKI_INT8 && t == RSTSR_F64) {
            double al, be;
            std::memcpy(&al, alpha, sizeof(double));
            std::memcpy(&be, beta, sizeof(double));
            std::vector<GemmProblem> oz;
            for (auto& P : probs) (P.K == 0 ? rest : oz).push_back(P);
            ozaki_grouped_f64(ctx, oz, al, be, is_zero_scalar(t, beta));
        } else {
            rest = probs;
        }
        // complex split mode and non-MFMA dtypes: one call per problem, in order
        for (auto& P : rest) run_gemm(ctx, t, mode, P, alpha, beta);
    });
}

}  // extern "C"
