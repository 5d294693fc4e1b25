// BLAS-style driver entry points over the MFMA GEMM: GEMMDriverAPI::driver_gemm
// (rstsr-blas-traits/src/blas3/gemm.rs:4-20), SYHEMMDriverAPI::driver_syhemm
// (blas3/syhemm.rs:4-19) and TRSMDriverAPI::driver_trsm (blas3/trsm.rs:4-19), with
// cblas flag values (FlagOrder C = 101 / F = 102, FlagTrans N = 111 / T = 112 /
// C = 113 / CN = 114, FlagUpLo U = 121 / L = 122, FlagDiag N = 131 / U = 132,
// FlagSide L = 141 / R = 142; rstsr-common/src/flags.rs:62-213).
//
// Storage order and transposition become (row stride, column stride) pairs of
// op(A), op(B) and C for the strided GEMM, so no operand is copied, except:
//  - a conjugated complex operand (trans C or CN), copied conjugated into a
//    dense scratch matrix first (the GEMM tiles have no conjugate path);
//  - the symmetric / Hermitian matrix of syhemm, expanded from its stored
//    triangle into a dense scratch matrix (BLAS reads only that triangle, and
//    only the real part of a Hermitian diagonal).
// Scratch lives in the context's auxiliary buffer, which a single GEMM does not
// use.
#include "common.hpp"
#include "registry.hpp"
#include "gemm_tile.hpp"

#include <cstring>
#include <type_traits>

namespace rstsr {
namespace hip {

void run_gemm(rstsr_hip_ctx* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, const GemmProblem& P0, const void* alpha,
              const void* beta);

namespace {

enum : int { ORD_C = 101, ORD_F = 102, TR_N = 111, TR_T = 112, TR_C = 113, TR_CN = 114 };
enum : int { UPLO_U = 121, UPLO_L = 122, DIAG_N = 131, DIAG_U = 132, SIDE_L = 141, SIDE_R = 142 };

template <class T>
__device__ __forceinline__ T conj_v(T x) {
    if constexpr (std::is_same<T, c128>::value || std::is_same<T, c64>::value) return T{x.re, -x.im};
    else return x;
}

// dst (rows x cols, row-major, dense) = conj(src) read with strides (rs, cs)
template <class T>
__global__ void __launch_bounds__(256) k_conj_copy(T* __restrict__ dst, const T* __restrict__ src, uint32_t rows,
                                                   uint32_t cols, int64_t rs, int64_t cs) {
    const uint64_t n = (uint64_t)rows * cols;
    for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (uint64_t)gridDim.x * 256) {
        const uint32_t i = (uint32_t)(e / cols), j = (uint32_t)(e - (uint64_t)i * cols);
        dst[e] = conj_v(src[(int64_t)i * rs + (int64_t)j * cs]);
    }
}

// dst (n x n, row-major) = the full symmetric / Hermitian matrix whose `lower`
// (else upper) triangle is stored at src with strides (rs, cs); a Hermitian
// diagonal keeps its real part only.
template <class T, bool HERMI>
__global__ void __launch_bounds__(256) k_sym_expand(T* __restrict__ dst, const T* __restrict__ src, uint32_t n,
                                                    int64_t rs, int64_t cs, int lower) {
    const uint64_t total = (uint64_t)n * n;
    for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (uint64_t)gridDim.x * 256) {
        const uint32_t i = (uint32_t)(e / n), j = (uint32_t)(e - (uint64_t)i * n);
        const bool stored = lower ? (i >= j) : (i <= j);
        T v = stored ? src[(int64_t)i * rs + (int64_t)j * cs] : src[(int64_t)j * rs + (int64_t)i * cs];
        if constexpr (HERMI) {
            if (!stored) v = conj_v(v);
            if (i == j) {
                if constexpr (std::is_same<T, c128>::value || std::is_same<T, c64>::value) v.im = 0;
            }
        }
        dst[e] = v;
    }
}

template <class T>
__device__ __forceinline__ T t_mul(T a, T b) {
    if constexpr (std::is_same<T, c128>::value || std::is_same<T, c64>::value)
        return T{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
    else return a * b;
}

// Quotients by one divisor, as accurate as divisions and without their setup per quotient, by a
// reciprocal of twice the precision. exact() (f64) divides.
template <class R>
struct Recip;
// f32: the f64 product with the f64 reciprocal has an error below 2^-28 f32 ulp, and no quotient of two
// f32 lies within 2^-25 ulp of the middle of two: rounded as the division, subnormal results too.
template <>
struct Recip<float> {
    double r;
    __device__ static Recip of(float d) { return {1.0 / d}; }
    __device__ __forceinline__ float quot(float a) const { return (float)(a * r); }
};
// f64: a (r + rl), r + rl = 1 / d to 2^-105, both parts scaled to [1/2, 1): half an ulp and 2^-50 ulp,
// that is rounded as the division but for quotients that close to the middle of two numbers. The
// exponents are put back, and v_div_fixup gives zeros, infinities and NaN their IEEE results.
// Subnormal results are rounded a second time there.
template <>
struct Recip<double> {
    double d, r, rl;
    int e;
    __device__ static Recip of(double d) {
        const double m = __builtin_amdgcn_frexp_mant(d), r = 1 / m;
        return {d, r, fma(-m, r, 1.0) * r, __builtin_amdgcn_frexp_exp(d)};
    }
    __device__ __forceinline__ double quot(double a) const {
        const double m = __builtin_amdgcn_frexp_mant(a);
        const double q = fma(m, r, m * rl);
        return __builtin_amdgcn_div_fixup(ldexp(q, __builtin_amdgcn_frexp_exp(a) - e), d, a);
    }
    __device__ double exact(double a) const { return a / d; }
};
__device__ __forceinline__ bool subnormal(double x) { return __builtin_amdgcn_class(x, 0x90); }
__device__ __forceinline__ bool subnormal(c128 x) { return subnormal(x.re) || subnormal(x.im); }

// Complex quotients: a conj(b) / |b|^2, b scaled by a power of two 2^k so that its larger part lies in
// [1/2, 1) (exact; no overflow of |b|^2), and the quotient scaled back.
template <class T, class R>
struct Scaled {
    R br, bi, d;
    int k;
    __device__ static Scaled of(T b) {
        const int k = ilogb2(fmax(fabs(b.re), fabs(b.im)));
        const R br = ldexp(b.re, -k), bi = ldexp(b.im, -k);
        return {br, bi, br * br + bi * bi, k};
    }
    __device__ static int ilogb2(double m) { return __builtin_amdgcn_frexp_exp(m); }
    __device__ static int ilogb2(float m) { return __builtin_amdgcn_frexp_expf(m); }
    __device__ __forceinline__ R re(T a) const { return a.re * br + a.im * bi; }
    __device__ __forceinline__ R im(T a) const { return a.im * br - a.re * bi; }
};
// a / b
template <class T>
__device__ __forceinline__ T t_div(T a, T b) {
    if constexpr (ElemOf<T>::CX) {
        const auto s = Scaled<T, typename ElemOf<T>::R>::of(b);
        return T{ldexp(s.re(a) / s.d, -s.k), ldexp(s.im(a) / s.d, -s.k)};
    } else {
        return a / b;
    }
}
// The divisor of one row of the solve.
template <class T>
struct Divisor {
    Recip<T> s;
    __device__ static Divisor of(T b) { return {Recip<T>::of(b)}; }
    __device__ __forceinline__ T quot(T a) const { return s.quot(a); }
    __device__ T exact(T a) const { return s.exact(a); }
};
template <class T, class R>
struct DivisorC {
    Scaled<T, R> b;
    Recip<R> d;
    __device__ static DivisorC of(T x) {
        const auto b = Scaled<T, R>::of(x);
        return {b, Recip<R>::of(b.d)};
    }
    __device__ __forceinline__ T quot(T a) const {
        return T{ldexp(d.quot(b.re(a)), -b.k), ldexp(d.quot(b.im(a)), -b.k)};
    }
    __device__ T exact(T a) const { return T{ldexp(d.exact(b.re(a)), -b.k), ldexp(d.exact(b.im(a)), -b.k)}; }
};
template <>
struct Divisor<c64> : DivisorC<c64, float> {
    __device__ static Divisor of(c64 b) { return {DivisorC<c64, float>::of(b)}; }
};
template <>
struct Divisor<c128> : DivisorC<c128, double> {
    __device__ static Divisor of(c128 b) { return {DivisorC<c128, double>::of(b)}; }
};

// v of lanes 16 g .. 16 g + 15 in every group of 16 lanes
__device__ __forceinline__ uint32_t bcast_row(uint32_t v, int g) {
    const auto h = __builtin_amdgcn_permlane32_swap(v, v, false, false);  // lower halves, upper halves
    const uint32_t w = g < 2 ? h[0] : h[1];
    const auto r = __builtin_amdgcn_permlane16_swap(w, w, false, false);  // even rows, odd rows
    return g % 2 == 0 ? r[0] : r[1];
}
template <class T>
__device__ __forceinline__ T bcast_rows(T v, int g) {
    uint32_t w[sizeof(T) / 4];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 4; ++i) w[i] = bcast_row(w[i], g);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Barrier for data that waves exchange through LDS: unlike __syncthreads it leaves global loads and
// stores in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

constexpr int TRSM_CB = 32;  // rows the column kernel takes at most

// Triangular solve of few rows, arguments as for k_trsm_block: one thread per column of X, 64 per
// block, T and the columns staged in LDS. Bound by reading and writing X where columns are many; for
// few columns by its chain, longer per row than k_trsm_block's. That one, eight waves per 16 columns,
// takes 5 us (f32) to 12 us (c128) per round of blocks however few the rows. So: up to 8 rows always
// here (no slower at one column), up to 32 from 16 rows CUs bytes of a row of X on, where the others
// need several rounds (us, f64, k_trsm_block against this: 2 rows x 1000000 382, 7; 8 x 300000 230, 16; 16
// x 10000 16, 8; 32 x 30000 42, 21; the other way round 16 x 3000 6.3, 8.5; 32 x 10000 16, 19).
template <class T>
__global__ void __launch_bounds__(64) k_trsm_cols(const T* __restrict__ Tm, int64_t trs, int64_t tcs, int unit, int kb,
                                                  T* __restrict__ X, int64_t xrs, int64_t xcs, int64_t r) {
    __shared__ T ts[TRSM_CB][TRSM_CB + 1];
    __shared__ T xs[TRSM_CB][64];
    const int j = threadIdx.x;
    const int64_t col = (int64_t)blockIdx.x * 64 + j;
    for (int e = j; e < kb * kb; e += 64) {
        const int i = e / kb, k = e - i * kb;
        // only the triangle is read, and a unit diagonal not at all
        if (k < i || (k == i && !unit)) ts[i][k] = Tm[(int64_t)i * trs + (int64_t)k * tcs];
    }
    if (col < r)
        for (int i = 0; i < kb; ++i) xs[i][j] = X[(int64_t)i * xrs + col * xcs];
    __syncthreads();
    if (col >= r) return;
    for (int i = 0; i < kb; ++i) {
        T acc = xs[i][j];
        for (int k = 0; k < i; ++k) {
            const T p = t_mul(ts[i][k], xs[k][j]);
            if constexpr (ElemOf<T>::CX) acc = T{acc.re - p.re, acc.im - p.im};
            else acc = acc - p;
        }
        xs[i][j] = unit ? acc : t_div(acc, ts[i][i]);
    }
    for (int i = 0; i < kb; ++i) X[(int64_t)i * xrs + col * xcs] = xs[i][j];
}

constexpr int TRSM_NB = 256;                 // rows solved by one launch
constexpr int TRSM_F = TRSM_NB / 16;         // 16-row fragments of them
constexpr int TRSM_NW = 8;                   // waves per block
constexpr int TRSM_FPW = TRSM_F / TRSM_NW;   // fragments per wave

// Triangular solve of up to 256 rows, in place: X (kb x r, strides xrs / xcs) := T^-1 X for the
// lower triangle T (kb x kb, strides trs / tcs; an upper one comes with its rows, columns and X's
// rows reversed, that is negative strides; unit: diagonal taken as one and not read).
//
// What bounds it: the chain over the rows (a column's x[i] needs every x before it), so all of it
// runs in one launch and each step is kept short. A block owns 16 columns of X, which are
// independent of all others: r / 16 blocks without any exchange. X stays in registers, its updates in
// the matrix cores' accumulators, fragment f (rows 16 f ..) in wave f % 8. Step j: the wave that owns
// fragment j subtracts block j - 1's share from it (four MFMAs), solves its 16 rows by substitution in
// the accumulators' own layout and publishes x through LDS; after one barrier the waves subtract
// T(f, j) x from their fragments below, with the blocks of T loaded a step ahead.
// Measured: 256 rows x 1600 columns f64 37 us; 2000 rows 0.51 ms in all, eight such launches and
// the updates between them by the GEMM (3.5 ms with 64-row blocks, one thread per column).
// TRSM_OCC waves per SIMD: three blocks per CU (f32), two (f64, c64), one (c128: its LDS).
template <class T>
constexpr int TRSM_OCC = sizeof(T) == 16 ? 2 : sizeof(T) == 4 ? 6 : 4;

template <class T>
__global__ void __launch_bounds__(64 * TRSM_NW, TRSM_OCC<T>)
    k_trsm_block(const T* __restrict__ Tm, int64_t trs, int64_t tcs, int unit, int kb, T* __restrict__ X, int64_t xrs,
                 int64_t xcs, int64_t r) {
    using R = typename ElemOf<T>::R;
    using MM = Mma<R>;
    constexpr bool CX = ElemOf<T>::CX;
    constexpr int NP = CX ? 2 : 1;
    __shared__ T diag[TRSM_F][16][16];  // [block][column c][row r > c]
    __shared__ Divisor<T> divs[TRSM_NB];
    __shared__ T xs[2][16][16];         // x of the current block: [parity][row][column]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = lane & 15, q = lane >> 4;
    const int64_t col = (int64_t)blockIdx.x * 16 + n;
    const int nf = (kb + 15) / 16;
    // rows past kb: x = 0, divisor one
    constexpr int DL = TRSM_F * 256 / (64 * TRSM_NW);  // diagonal elements per thread, all in flight at once
    T dl[DL];
#pragma unroll
    for (int u = 0; u < DL; ++u) {
        const int e = u * 64 * TRSM_NW + threadIdx.x, f = e >> 8, i = e >> 4 & 15, c = e & 15, row = 16 * f + i;
        dl[u] = i > c && row < kb ? Tm[(int64_t)row * trs + (int64_t)(16 * f + c) * tcs] : T{};
    }
    for (int i = threadIdx.x; i < nf * 16; i += 64 * TRSM_NW) {
        T d{};
        if constexpr (CX) d.re = 1;
        else d = 1;
        if (!unit && i < kb) d = Tm[(int64_t)i * (trs + tcs)];
        divs[i] = Divisor<T>::of(d);
    }
    // The right-hand sides of the wave's next fragment to solve and, apart from them, the sums of the
    // updates: terms below the rounding of a right-hand side still count together. The sums start at
    // -0, which leaves every value as it is.
    constexpr bool LATE = sizeof(T) == 16;  // c128: a fragment's right-hand sides come when the one before is solved
    T rhs[LATE ? 1 : TRSM_FPW][4];
    auto load_rhs = [&](int i) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int row = 16 * (i * TRSM_NW + wave) + MM::row(k, lane);
            rhs[LATE ? 0 : i][k] = row < kb && col < r ? X[(int64_t)row * xrs + col * xcs] : T{};
        }
    };
    load_rhs(0);
    if (!LATE) load_rhs(1);
    typename MM::Acc acc[TRSM_FPW][NP];
#pragma unroll
    for (int i = 0; i < TRSM_FPW; ++i)
#pragma unroll
        for (int p = 0; p < NP; ++p)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc[i][p][k] = -(R)0;
    // T(f, j) of this lane: row n of the fragment, positions 4 q + e of block j
    auto load_t = [&](T (&t)[4], int f, int j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 16 * f + n;
            t[e] = f > j && row < kb ? Tm[(int64_t)row * trs + (int64_t)(16 * j + 4 * q + e) * tcs] : T{};
        }
    };
    auto subtract = [&](typename MM::Acc (&a)[NP], const T (&t)[4], const T (&x)[4]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if constexpr (CX) {
                a[0] = MM::mma(-t[e].re, x[e].re, a[0]);
                a[0] = MM::mma(t[e].im, x[e].im, a[0]);
                a[NP - 1] = MM::mma(-t[e].re, x[e].im, a[NP - 1]);
                a[NP - 1] = MM::mma(-t[e].im, x[e].re, a[NP - 1]);
            } else {
                a[0] = MM::mma(-t[e], x[e], a[0]);
            }
        }
    };
    // substitution of fragment f (this wave's right-hand sides and update sums a): x goes to xs[f & 1],
    // which nothing else reads any more. Lane (n, q) holds rows MM::row(k, lane) of column n; each quotient
    // is formed in the lanes that hold its row and handed to the column's other lanes by two lane swaps.
    // The divisors and columns of the diagonal block do not depend on x: they are read a step ahead.
    constexpr bool F64 = sizeof(R) == 8;
    // the same by divisions, a lane per column, for results below the normal range: xf holds the
    // right-hand sides less the updates
    auto divide = [&](auto& xf, int f) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (q != 0) return;
#pragma unroll 1
        for (int i = 0; i < 16; ++i) {
            T v = xf[i][n];
#pragma unroll 1
            for (int c = 0; c < i; ++c) {
                const T e = diag[f][c][i], x = xf[c][n];
                if constexpr (CX) {
                    v.re = fma(e.im, x.im, fma(-e.re, x.re, v.re));
                    v.im = fma(-e.im, x.re, fma(-e.re, x.im, v.im));
                } else {
                    v = fma(-e, x, v);
                }
            }
            xf[i][n] = divs[16 * f + i].exact(v);
        }
    };
    auto solve = [&](const T (&rf)[4], const typename MM::Acc (&a)[NP], int f) __attribute__((always_inline)) {
        T(&xf)[16][16] = xs[f & 1];
        constexpr bool NARROW = CX;  // not a step ahead: their registers are scarce
        T b[4], d[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if constexpr (CX) b[k] = T{rf[k].re + a[0][k], rf[k].im + a[NP - 1][k]};
            else b[k] = rf[k] + a[0][k];
            if constexpr (F64) xf[MM::row(k, lane)][n] = b[k];
            d[k] = diag[f][0][MM::row(k, lane)];
        }
        Divisor<T> dv = divs[16 * f];
#pragma unroll
        for (int c = 0; c < 16; ++c) {
            constexpr bool RS = sizeof(R) == 8;  // row 4 k + q (else 4 q + k) is in lanes q, register k
            const int k0 = RS ? c / 4 : c % 4, g = RS ? c % 4 : c / 4;
            const Divisor<T> dc = dv;
            T e[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) e[k] = NARROW ? diag[f][c][MM::row(k, lane)] : d[k];
            if (c < 15) {
                dv = divs[16 * f + c + 1];
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (!NARROW) d[k] = diag[f][c + 1][MM::row(k, lane)];
            }
            // no quotient by one: (inf + i nan) / 1 would spread the NaN
            const T xc = unit ? b[k0] : dc.quot(b[k0]);
            if (q == g) b[k0] = xc;
            const T xb = bcast_rows(xc, g);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (RS && k < k0) continue;  // rows above c only
                T v = b[k];
                if constexpr (CX) {
                    v.re = fma(e[k].im, xb.im, fma(-e[k].re, xb.re, v.re));
                    v.im = fma(-e[k].im, xb.re, fma(-e[k].re, xb.im, v.im));
                } else {
                    v = fma(-e[k], xb, v);
                }
                if (MM::row(k, lane) > c) b[k] = v;
            }
        }
        if constexpr (F64) {
            bool low = false;
#pragma unroll
            for (int k = 0; k < 4; ++k) low = low || subnormal(b[k]);
            if (__any(low) && !unit) {
                divide(xf, f);
                return;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) xf[MM::row(k, lane)][n] = b[k];
    };
    T t[TRSM_FPW][4];
#pragma unroll
    for (int i = 0; i < TRSM_FPW; ++i) load_t(t[i], i * TRSM_NW + wave, 0);
#pragma unroll
    for (int u = 0; u < DL; ++u) {
        const int e = u * 64 * TRSM_NW + threadIdx.x;
        diag[e >> 8][e & 15][e >> 4 & 15] = dl[u];
    }
    __syncthreads();  // diagonal blocks and divisors staged
    if (wave == 0) {
        solve(rhs[0], acc[0], 0);
        if (LATE) load_rhs(1);
    }
    lds_barrier();
    for (int j = 0; j < nf; ++j) {
        // x of block j is in xs[j & 1], T(., j) in t
        T x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = xs[j & 1][4 * q + e][n];
        const int own = (j + 1) % TRSM_NW == wave && j + 1 < nf ? (j + 1) / TRSM_NW : -1;
#pragma unroll
        for (int i = 0; i < TRSM_FPW; ++i)
            if (i == own) {
                subtract(acc[i], t[i], x);
                solve(rhs[LATE ? 0 : i], acc[i], j + 1);
                if (LATE && i + 1 < TRSM_FPW) load_rhs(i + 1);
            }
#pragma unroll
        for (int i = 0; i < TRSM_FPW; ++i)
            if (i != own && i * TRSM_NW + wave > j && i * TRSM_NW + wave < nf) subtract(acc[i], t[i], x);
        // the wave that solves last from here on stores block j
        if (wave == j % TRSM_NW && col < r) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = 16 * j + 4 * q + e;
                if (row < kb) X[(int64_t)row * xrs + col * xcs] = x[e];
            }
        }
        // the next solver is another wave, whose loads run while this step's solver works
#pragma unroll
        for (int i = 0; i < TRSM_FPW; ++i) load_t(t[i], i * TRSM_NW + wave, j + 1);
        lds_barrier();
    }
}

// X (rows x cols, strides rs / cs) *= alpha, or := 0 when zero (BLAS: B is not read)
template <class T>
__global__ void __launch_bounds__(256) k_scale2d(T* __restrict__ X, uint32_t rows, uint32_t cols, int64_t rs,
                                                 int64_t cs, T alpha, int zero) {
    const uint64_t n = (uint64_t)rows * cols;
    for (uint64_t e = (uint64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (uint64_t)gridDim.x * 256) {
        const uint32_t i = (uint32_t)(e / cols), j = (uint32_t)(e - (uint64_t)i * cols);
        T* p = X + (int64_t)i * rs + (int64_t)j * cs;
        *p = zero ? T{} : t_mul(alpha, *p);
    }
}

uint32_t grid_for(uint64_t n) {
    uint64_t b = (n + 255) / 256;
    return (uint32_t)std::min<uint64_t>(std::max<uint64_t>(b, 1), 65536);
}

bool is_cplx(rstsr_dtype_t t) { return t == RSTSR_C64 || t == RSTSR_C128; }

template <class F>
void dispatch_gemm_dtype(rstsr_dtype_t t, F&& f) {
    switch (t) {
        case RSTSR_F32: f(float{}); break;
        case RSTSR_F64: f(double{}); break;
        case RSTSR_C64: f(c64{}); break;
        case RSTSR_C128: f(c128{}); break;
        default: RSTSR_RAISE(UnImplemented, "the BLAS drivers take f32, f64, c64 and c128");
    }
}

// Strides of a stored (rows x cols) matrix with leading dimension ld.
void stored_strides(int order, int64_t ld, int64_t& rs, int64_t& cs) {
    if (order == ORD_C) {
        rs = ld;
        cs = 1;
    } else {
        rs = 1;
        cs = ld;
    }
}

void check_ld(int order, size_t rows, size_t cols, size_t ld, const char* nm) {
    const size_t need = order == ORD_C ? cols : rows;
    if (ld < std::max<size_t>(need, 1))
        RSTSR_RAISE(InvalidValue, std::string("leading dimension of ") + nm + " is smaller than the stored extent");
}

void check_mat(const void* p, size_t rows, size_t cols, int64_t rs, int64_t cs, size_t es, const char* nm) {
    size_t s[2] = {rows, cols};
    int64_t t[2] = {rs, cs};
    check_extent_rel(p, 2, s, t, es, nm);
}

}  // namespace

// driver_gemm: C (m x n) = alpha op(A) op(B) + beta C.
static void driver_gemm(rstsr_hip_ctx* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, int order, int transa,
                        int transb, size_t m, size_t n, size_t k, const void* alpha, const void* a, size_t lda,
                        const void* b, size_t ldb, const void* beta, void* c, size_t ldc) {
    if (order != ORD_C && order != ORD_F) RSTSR_RAISE(InvalidValue, "order must be 101 (C) or 102 (F)");
    dispatch_gemm_dtype(t, [](auto) {});  // BLAS types only
    for (int tr : {transa, transb})
        if (tr < TR_N || tr > TR_CN) RSTSR_RAISE(InvalidValue, "trans must be 111 (N), 112 (T), 113 (C) or 114 (CN)");
    const size_t es = dtype_size(t);
    const bool ta = transa == TR_T || transa == TR_C, tb = transb == TR_T || transb == TR_C;
    const bool ca = is_cplx(t) && (transa == TR_C || transa == TR_CN);
    const bool cb = is_cplx(t) && (transb == TR_C || transb == TR_CN);
    // stored shapes: A is (m x k) or (k x m) when transposed; B (k x n) or (n x k)
    const size_t ar = ta ? k : m, ac = ta ? m : k, br = tb ? n : k, bc = tb ? k : n;
    check_ld(order, ar, ac, lda, "a");
    check_ld(order, br, bc, ldb, "b");
    check_ld(order, m, n, ldc, "c");
    int64_t srs, scs;
    GemmProblem P{};
    P.M = (int64_t)m;
    P.N = (int64_t)n;
    P.K = (int64_t)k;
    P.bd.nbd = 0;
    P.nbatch = 1;
    stored_strides(order, (int64_t)lda, srs, scs);
    P.a = a;
    P.rsa = ta ? scs : srs;
    P.csa = ta ? srs : scs;
    stored_strides(order, (int64_t)ldb, srs, scs);
    P.b = b;
    P.rsb = tb ? scs : srs;
    P.csb = tb ? srs : scs;
    stored_strides(order, (int64_t)ldc, srs, scs);
    P.c = c;
    P.rsc = srs;
    P.csc = scs;
    if (m == 0 || n == 0) return;
    if (k > 0) {
        check_mat(P.a, m, k, P.rsa, P.csa, es, "a");
        check_mat(P.b, k, n, P.rsb, P.csb, es, "b");
    }
    check_mat(P.c, m, n, P.rsc, P.csc, es, "c");
    std::lock_guard<std::mutex> g(ctx->mu);
    if ((ca || cb) && k > 0) {
        const size_t na = ca ? m * k : 0, nb = cb ? k * n : 0;
        char* buf = (char*)aux_buffer(ctx, (na + nb) * es + 256);
        dispatch_gemm_dtype(t, [&](auto tag) {
            using T = decltype(tag);
            if (ca) {
                T* d = (T*)buf;
                hipLaunchKernelGGL(k_conj_copy<T>, dim3(grid_for(na)), dim3(256), 0, ctx->stream, d, (const T*)P.a,
                                   (uint32_t)m, (uint32_t)k, P.rsa, P.csa);
                check_launch("conjugate copy");
                P.a = d;
                P.rsa = (int64_t)k;
                P.csa = 1;
            }
            if (cb) {
                T* d = (T*)(buf + ((na * es + 255) & ~(size_t)255));
                hipLaunchKernelGGL(k_conj_copy<T>, dim3(grid_for(nb)), dim3(256), 0, ctx->stream, d, (const T*)P.b,
                                   (uint32_t)k, (uint32_t)n, P.rsb, P.csb);
                check_launch("conjugate copy");
                P.b = d;
                P.rsb = (int64_t)n;
                P.csb = 1;
            }
        });
    }
    run_gemm(ctx, t, mode, P, alpha, beta);
}

// driver_syhemm: C (m x n) = alpha A B + beta C (side L, A m x m) or alpha B A + beta C
// (side R, A n x n); A symmetric (hermi 0) or Hermitian (hermi 1), its `uplo` triangle stored.
static void driver_syhemm(rstsr_hip_ctx* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, int hermi, int order, int side,
                          int uplo, size_t m, size_t n, const void* alpha, const void* a, size_t lda, const void* b,
                          size_t ldb, const void* beta, void* c, size_t ldc) {
    if (order != ORD_C && order != ORD_F) RSTSR_RAISE(InvalidValue, "order must be 101 (C) or 102 (F)");
    if (side != SIDE_L && side != SIDE_R) RSTSR_RAISE(InvalidValue, "side must be 141 (L) or 142 (R)");
    if (uplo != UPLO_U && uplo != UPLO_L) RSTSR_RAISE(InvalidValue, "uplo must be 121 (U) or 122 (L)");
    dispatch_gemm_dtype(t, [](auto) {});  // BLAS types only
    const size_t es = dtype_size(t);
    const size_t na = side == SIDE_L ? m : n;
    check_ld(order, na, na, lda, "a");
    check_ld(order, m, n, ldb, "b");
    check_ld(order, m, n, ldc, "c");
    if (m == 0 || n == 0) return;
    int64_t ars, acs, brs, bcs, crs, ccs;
    stored_strides(order, (int64_t)lda, ars, acs);
    stored_strides(order, (int64_t)ldb, brs, bcs);
    stored_strides(order, (int64_t)ldc, crs, ccs);
    check_mat(a, na, na, ars, acs, es, "a");
    check_mat(b, m, n, brs, bcs, es, "b");
    check_mat(c, m, n, crs, ccs, es, "c");
    std::lock_guard<std::mutex> g(ctx->mu);
    void* full = aux_buffer(ctx, na * na * es + 256);
    dispatch_gemm_dtype(t, [&](auto tag) {
        using T = decltype(tag);
        auto go = [&](auto h) {
            hipLaunchKernelGGL((k_sym_expand<T, decltype(h)::value>), dim3(grid_for((uint64_t)na * na)), dim3(256), 0,
                               ctx->stream, (T*)full, (const T*)a, (uint32_t)na, ars, acs, uplo == UPLO_L ? 1 : 0);
        };
        if (hermi && is_cplx(t)) go(std::true_type{});
        else go(std::false_type{});
        check_launch("symmetric expand");
    });
    GemmProblem P{};
    P.M = (int64_t)m;
    P.N = (int64_t)n;
    P.K = (int64_t)na;
    P.bd.nbd = 0;
    P.nbatch = 1;
    if (side == SIDE_L) {
        P.a = full;
        P.rsa = (int64_t)na;
        P.csa = 1;
        P.b = b;
        P.rsb = brs;
        P.csb = bcs;
    } else {
        P.a = b;
        P.rsa = brs;
        P.csa = bcs;
        P.b = full;
        P.rsb = (int64_t)na;
        P.csb = 1;
    }
    P.c = c;
    P.rsc = crs;
    P.csc = ccs;
    run_gemm(ctx, t, mode, P, alpha, beta);
}

// driver_trsm: op(A) X = alpha B (side L, A m x m) or X op(A) = alpha B (side R, A n x n), B (m x n)
// overwritten by X; A triangular (its `uplo` triangle read; diag U: unit diagonal, not read).
// Every case becomes T Y = alpha Z with T lower or upper: side R solves op(A)^T X^T = alpha B^T, and
// a transposition swaps T's strides and its triangle; a conjugated A (trans C or CN) is copied
// conjugated into scratch first. T Y = Z is solved recursively: halves of the rows, the
// trailing half updated by the GEMM (alpha -1, beta 1) with K the leading half's size, down to
// 256-row diagonal blocks solved in one launch each (k_trsm_block).
static void driver_trsm(rstsr_hip_ctx* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, int order, int side, int uplo,
                        int transa, int diag, size_t m, size_t n, const void* alpha, const void* a, size_t lda, void* b,
                        size_t ldb) {
    if (order != ORD_C && order != ORD_F) RSTSR_RAISE(InvalidValue, "order must be 101 (C) or 102 (F)");
    if (side != SIDE_L && side != SIDE_R) RSTSR_RAISE(InvalidValue, "side must be 141 (L) or 142 (R)");
    if (uplo != UPLO_U && uplo != UPLO_L) RSTSR_RAISE(InvalidValue, "uplo must be 121 (U) or 122 (L)");
    if (diag != DIAG_N && diag != DIAG_U) RSTSR_RAISE(InvalidValue, "diag must be 131 (N) or 132 (U)");
    if (transa < TR_N || transa > TR_CN) RSTSR_RAISE(InvalidValue, "trans must be 111 (N), 112 (T), 113 (C) or 114 (CN)");
    dispatch_gemm_dtype(t, [](auto) {});  // BLAS types only
    const size_t es = dtype_size(t);
    const size_t s = side == SIDE_L ? m : n;  // order of A
    check_ld(order, s, s, lda, "a");
    check_ld(order, m, n, ldb, "b");
    if (m == 0 || n == 0) return;
    int64_t ars, acs, brs, bcs;
    stored_strides(order, (int64_t)lda, ars, acs);
    stored_strides(order, (int64_t)ldb, brs, bcs);
    check_mat(a, s, s, ars, acs, es, "a");
    check_mat(b, m, n, brs, bcs, es, "b");
    // T = op(A) (side L) or op(A)^T (side R); Y = X (rows s = m) or X^T (rows s = n)
    const bool trans_op = transa == TR_T || transa == TR_C;
    const bool tr = trans_op != (side == SIDE_R);
    const bool conj = is_cplx(t) && (transa == TR_C || transa == TR_CN);
    int64_t trs = tr ? acs : ars, tcs = tr ? ars : acs;
    const bool lower = (uplo == UPLO_L) != tr;
    const int64_t yrs = side == SIDE_L ? brs : bcs, ycs = side == SIDE_L ? bcs : brs;
    const int64_t r = (int64_t)(side == SIDE_L ? n : m);  // columns of Y
    std::lock_guard<std::mutex> g(ctx->mu);
    dispatch_gemm_dtype(t, [&](auto tag) {
        using T = decltype(tag);
        const T* Tm = (const T*)a;
        if (conj) {
            T* d = (T*)aux_buffer(ctx, s * s * es + 256);
            hipLaunchKernelGGL(k_conj_copy<T>, dim3(grid_for((uint64_t)s * s)), dim3(256), 0, ctx->stream, d, Tm,
                               (uint32_t)s, (uint32_t)s, trs, tcs);
            check_launch("conjugate copy");
            Tm = d;
            trs = (int64_t)s;
            tcs = 1;
        }
        T* Y = (T*)b;
        T al;
        std::memcpy(&al, alpha, sizeof(T));
        T one{}, minus_one{};
        if constexpr (std::is_same<T, c128>::value || std::is_same<T, c64>::value) {
            one.re = 1;
            minus_one.re = -1;
        } else {
            one = 1;
            minus_one = -1;
        }
        const bool is_one = std::memcmp(&al, &one, sizeof(T)) == 0;
        const T zero{};
        const bool is_zero = std::memcmp(&al, &zero, sizeof(T)) == 0;
        if (!is_one) {
            hipLaunchKernelGGL(k_scale2d<T>, dim3(grid_for((uint64_t)s * r)), dim3(256), 0, ctx->stream, Y,
                               (uint32_t)s, (uint32_t)r, yrs, ycs, al, is_zero ? 1 : 0);
            check_launch("trsm scale");
            if (is_zero) return;
        }
        // rows [lo, hi) of the solve
        auto solve = [&](auto&& self, int64_t lo, int64_t hi) -> void {
            const int64_t len = hi - lo;
            if (len <= TRSM_NB) {
                // an upper triangle is a lower one with every row order reversed
                const int64_t at = lower ? lo : hi - 1, sg = lower ? 1 : -1;
                const int64_t cu = std::max(ctx->num_cu, 1);
                const bool cols = len <= TRSM_CB && (len <= 8 || r * (int64_t)sizeof(T) >= 16 * len * cu);
                // at most 2^32 - 1 threads per launch
                const int64_t step = (int64_t)1 << 26;
                for (int64_t c0 = 0; c0 < r; c0 += step) {
                    const int64_t rc = std::min(step, r - c0);
                    const dim3 grid((uint32_t)(cols ? (rc + 63) / 64 : (rc + 15) / 16)), blk(cols ? 64 : 64 * TRSM_NW);
                    hipLaunchKernelGGL(cols ? k_trsm_cols<T> : k_trsm_block<T>, grid, blk, 0, ctx->stream,
                                       Tm + at * (trs + tcs), sg * trs, sg * tcs, diag == DIAG_U ? 1 : 0, (int)len,
                                       Y + at * yrs + c0 * ycs, sg * yrs, ycs, rc);
                }
                check_launch("trsm diagonal block");
                return;
            }
            const int64_t mid = lo + ((len / 2 + TRSM_NB - 1) / TRSM_NB) * TRSM_NB;
            // first the half the other depends on, then its update of the other half, then that half
            const int64_t f0 = lower ? lo : mid, f1 = lower ? mid : hi;  // solved first
            const int64_t s0 = lower ? mid : lo, s1 = lower ? hi : mid;  // updated, solved second
            self(self, f0, f1);
            GemmProblem P{};
            P.M = s1 - s0;
            P.N = r;
            P.K = f1 - f0;
            P.bd.nbd = 0;
            P.nbatch = 1;
            P.a = Tm + s0 * trs + f0 * tcs;
            P.rsa = trs;
            P.csa = tcs;
            P.b = Y + f0 * yrs;
            P.rsb = yrs;
            P.csb = ycs;
            P.c = Y + s0 * yrs;
            P.rsc = yrs;
            P.csc = ycs;
            run_gemm(ctx, t, mode, P, &minus_one, &one);
            self(self, s0, s1);
        };
        solve(solve, 0, (int64_t)s);
    });
}

}  // namespace hip
}  // namespace rstsr

using namespace rstsr;
using namespace rstsr::hip;

extern "C" {

int rstsr_hip_driver_gemm(rstsr_hip_ctx_t* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, int order, int transa,
                          int transb, size_t m, size_t n, size_t k, const void* alpha, const void* a, size_t lda,
                          const void* b, size_t ldb, const void* beta, void* c, size_t ldc) {
    return guarded([&] {
        bind(ctx);
        driver_gemm(ctx, t, mode, order, transa, transb, m, n, k, alpha, a, lda, b, ldb, beta, c, ldc);
    });
}

int rstsr_hip_driver_syhemm(rstsr_hip_ctx_t* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, int hermi, int order,
                            int side, int uplo, size_t m, size_t n, const void* alpha, const void* a, size_t lda,
                            const void* b, size_t ldb, const void* beta, void* c, size_t ldc) {
    return guarded([&] {
        bind(ctx);
        driver_syhemm(ctx, t, mode, hermi, order, side, uplo, m, n, alpha, a, lda, b, ldb, beta, c, ldc);
    });
}

int rstsr_hip_driver_trsm(rstsr_hip_ctx_t* ctx, rstsr_dtype_t t, rstsr_gemm_mode_t mode, int order, int side,
                          int uplo, int transa, int diag, size_t m, size_t n, const void* alpha, const void* a,
                          size_t lda, void* b, size_t ldb) {
    return guarded([&] {
        bind(ctx);
        driver_trsm(ctx, t, mode, order, side, uplo, transa, diag, m, n, alpha, a, lda, b, ldb);
    });
}

}  // extern "C"
