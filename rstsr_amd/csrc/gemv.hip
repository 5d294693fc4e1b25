// Matrix-vector products: y[i] = alpha sum_k A(i, k) x(k) + beta y[i], for every matmul with one
// row or one column (rules 1, 3 and 4 of the matmul, and 2-d products with M or N = 1).
//
// What bounds them: A is read once (HBM), two operations per element, so the matrix cores have
// nothing to gain and a tile kernel wastes all but one row of its tile. The kernels stream A with
// 16-byte loads along its unit-stride axis, several rows or steps in flight per lane:
//   k_gemv_row: lanes along k, four rows per wave share each load of x;
//   k_gemv_col: lanes along i, four waves of a block take a quarter of the k range each.
// Where the outputs alone give too few waves, k is split over blocks and k_gemv_fin adds the
// partial sums in order. Kernel and splits follow from the sizes, A's layout and the number of CUs, so
// a product in another layout may round differently.
// Measured: f64 8000 x 8000 79 us row-major (6.5 TB/s), 86 us column-major; 528 us on a tile kernel.
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"

namespace rstsr {
namespace hip {

template <class T>
struct GemvArgs {
    int64_t M, K;
    const T* a;
    int64_t rs, cs;  // A(i, k) at a + i rs + k cs
    const T* x;
    int64_t xs;
    T* y;
    int64_t ys;
    T alpha, beta;
    int beta_zero;
    int64_t chunk;  // k positions per split (grid y)
    int nsplit;
    T* part;        // [batch][split][i] when nsplit > 1
    BatchDesc bd;   // sa: A, sb: x, sc: y
};

template <class T>
__device__ __forceinline__ T gv_zero() {
    return T{};
}
template <class T>
__device__ __forceinline__ T gv_add(T a, T b) {
    if constexpr (std::is_integral<T>::value) {
        using U = typename std::make_unsigned<T>::type;
        return (T)((U)a + (U)b);
    } else if constexpr (std::is_floating_point<T>::value) {
        return a + b;
    } else {
        return T{a.re + b.re, a.im + b.im};
    }
}
template <class T>
__device__ __forceinline__ T gv_fma(T a, T b, T c) {
    if constexpr (std::is_integral<T>::value) {
        using U = typename std::make_unsigned<T>::type;
        return (T)((U)a * (U)b + (U)c);
    } else if constexpr (std::is_same<T, double>::value) {
        return fma(a, b, c);
    } else if constexpr (std::is_same<T, float>::value) {
        return fmaf(a, b, c);
    } else if constexpr (std::is_same<T, c128>::value) {
        return T{fma(-a.im, b.im, fma(a.re, b.re, c.re)), fma(a.im, b.re, fma(a.re, b.im, c.im))};
    } else {
        return T{fmaf(-a.im, b.im, fmaf(a.re, b.re, c.re)), fmaf(a.im, b.re, fmaf(a.re, b.im, c.im))};
    }
}
template <class T>
__device__ __forceinline__ T gv_shfl(T v, int m) {
    constexpr int W = sizeof(T) / 4;
    int w[W];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int i = 0; i < W; ++i) w[i] = __shfl_xor(w[i], m, 64);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}
template <class T>
__device__ __forceinline__ T gv_wave_sum(T v) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) v = gv_add(v, gv_shfl(v, m));
    return v;
}

// VEC consecutive elements in one 16-byte load; the address needs the element's alignment only
template <class T, int VEC>
struct GvPack {
    T v[VEC];
};
template <class T, int VEC, bool NT>
__device__ __forceinline__ GvPack<T, VEC> gv_load(const T* p) {
    GvPack<T, VEC> r;
    if constexpr (VEC == 1) {
        r.v[0] = *p;
    } else {
        typedef uint32_t w4 __attribute__((ext_vector_type(4), aligned(4)));
        w4 w;
        if constexpr (NT) w = __builtin_nontemporal_load((const w4*)p);
        else w = *(const w4*)p;
        __builtin_memcpy(&r, &w, 16);
    }
    return r;
}

template <class T>
__device__ __forceinline__ T gv_out(const GemvArgs<T>& g, T s, const T* y) {
    if constexpr (std::is_integral<T>::value || std::is_floating_point<T>::value) {
        T v = gv_fma<T>(g.alpha, s, T{});
        if (!g.beta_zero) v = gv_fma<T>(g.beta, *y, v);
        return v;
    } else {
        T v{g.alpha.re * s.re - g.alpha.im * s.im, g.alpha.re * s.im + g.alpha.im * s.re};
        if (!g.beta_zero) v = gv_fma<T>(g.beta, *y, v);
        return v;
    }
}
// output i of batch b (split sp): the result, or a partial sum
template <class T>
__device__ __forceinline__ void gv_put(const GemvArgs<T>& g, int64_t oc, uint32_t b, int sp, int64_t i, T s) {
    if (g.nsplit > 1) {
        g.part[((int64_t)b * g.nsplit + sp) * g.M + i] = s;
    } else {
        T* y = g.y + oc + i * g.ys;
        *y = gv_out(g, s, y);
    }
}

constexpr int GV_RPW = 4;  // rows per wave: four rows' loads share one load of x

// WPR waves (of a block of four) share each group of four rows, k interleaved between them.
// XU: x has unit stride. VEC > 1: A has unit stride along k.
template <class T, int VEC, int WPR, bool XU, bool NT>
__global__ void __launch_bounds__(256) k_gemv_row(GemvArgs<T> g) {
    constexpr int G = 4 / WPR;  // row groups per block
    constexpr int64_t W = 64 * VEC * WPR;
    __shared__ T red[WPR > 1 ? 4 : 1][GV_RPW];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t i0 = ((int64_t)blockIdx.x * G + wave / WPR) * GV_RPW;
    int64_t oa, ox, oy;
    batch_offsets(g.bd, blockIdx.z, oa, ox, oy);
    const int64_t k0 = (int64_t)blockIdx.y * g.chunk, k1 = min(g.K, k0 + g.chunk);
    const T* x = g.x + ox;
    const T* row[GV_RPW];
    // rows past the last one repeat it and are not stored
#pragma unroll
    for (int r = 0; r < GV_RPW; ++r) row[r] = g.a + oa + min(i0 + r, g.M - 1) * g.rs;
    T acc[GV_RPW];
#pragma unroll
    for (int r = 0; r < GV_RPW; ++r) acc[r] = gv_zero<T>();
    auto load_x = [&](int64_t k) {
        if constexpr (XU) {
            return gv_load<T, VEC, false>(x + k);
        } else {
            GvPack<T, VEC> p;
#pragma unroll
            for (int v = 0; v < VEC; ++v) p.v[v] = x[(k + v) * g.xs];
            return p;
        }
    };
    int64_t k = k0 + (int64_t)((wave % WPR) * 64 + lane) * VEC;
    if (i0 < g.M) {
        for (; k + W + VEC <= k1; k += 2 * W) {
            GvPack<T, VEC> a0[GV_RPW], a1[GV_RPW];
#pragma unroll
            for (int r = 0; r < GV_RPW; ++r) {
                a0[r] = gv_load<T, VEC, NT>(row[r] + k * g.cs);
                a1[r] = gv_load<T, VEC, NT>(row[r] + (k + W) * g.cs);
            }
            const GvPack<T, VEC> x0 = load_x(k), x1 = load_x(k + W);
#pragma unroll
            for (int r = 0; r < GV_RPW; ++r)
#pragma unroll
                for (int v = 0; v < VEC; ++v) {
                    acc[r] = gv_fma(a0[r].v[v], x0.v[v], acc[r]);
                    acc[r] = gv_fma(a1[r].v[v], x1.v[v], acc[r]);
                }
        }
        for (; k + VEC <= k1; k += W) {
            GvPack<T, VEC> a0[GV_RPW];
#pragma unroll
            for (int r = 0; r < GV_RPW; ++r) a0[r] = gv_load<T, VEC, NT>(row[r] + k * g.cs);
            const GvPack<T, VEC> x0 = load_x(k);
#pragma unroll
            for (int r = 0; r < GV_RPW; ++r)
#pragma unroll
                for (int v = 0; v < VEC; ++v) acc[r] = gv_fma(a0[r].v[v], x0.v[v], acc[r]);
        }
        if (VEC > 1 && k < k1) {
#pragma unroll
            for (int v = 0; v < VEC; ++v)
                if (k + v < k1) {
                    const T xv = x[(k + v) * g.xs];
#pragma unroll
                    for (int r = 0; r < GV_RPW; ++r) acc[r] = gv_fma(row[r][(k + v) * g.cs], xv, acc[r]);
                }
        }
    }
#pragma unroll
    for (int r = 0; r < GV_RPW; ++r) acc[r] = gv_wave_sum(acc[r]);
    if constexpr (WPR > 1) {
        if (lane == 0)
#pragma unroll
            for (int r = 0; r < GV_RPW; ++r) red[wave][r] = acc[r];
        __syncthreads();
        if (threadIdx.x < GV_RPW && i0 + threadIdx.x < g.M) {
            T s = red[0][threadIdx.x];
#pragma unroll
            for (int w = 1; w < 4; ++w) s = gv_add(s, red[w][threadIdx.x]);
            gv_put(g, oy, blockIdx.z, blockIdx.y, i0 + threadIdx.x, s);
        }
    } else {
        if (lane == 0)
#pragma unroll
            for (int r = 0; r < GV_RPW; ++r)
                if (i0 + r < g.M) gv_put(g, oy, blockIdx.z, blockIdx.y, i0 + r, acc[r]);
    }
}

// Lane l of every wave owns outputs i0 + l VEC .. + VEC - 1; the block's four waves take a quarter of
// its k range each. VEC > 1: A has unit stride along i.
template <class T, int VEC, bool NT>
__global__ void __launch_bounds__(256) k_gemv_col(GemvArgs<T> g) {
    constexpr int U = 8;
    __shared__ T red[4][64 * VEC];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i = ((int64_t)blockIdx.x * 64 + lane) * VEC;
    int64_t oa, ox, oy;
    batch_offsets(g.bd, blockIdx.z, oa, ox, oy);
    const int64_t b0 = (int64_t)blockIdx.y * g.chunk, b1 = min(g.K, b0 + g.chunk), q = (b1 - b0 + 3) / 4;
    const int64_t k0 = min(b1, b0 + wave * q), k1 = min(b1, k0 + q);
    const T* x = g.x + ox;
    T acc[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) acc[v] = gv_zero<T>();
    if (i + VEC <= g.M) {
        const T* p = g.a + oa + i * g.rs;
        int64_t k = k0;
        for (; k + U <= k1; k += U) {
            GvPack<T, VEC> a[U];
            T xv[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                a[u] = gv_load<T, VEC, NT>(p + (k + u) * g.cs);
                xv[u] = x[(k + u) * g.xs];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int v = 0; v < VEC; ++v) acc[v] = gv_fma(a[u].v[v], xv[u], acc[v]);
        }
        for (; k < k1; ++k) {
            const GvPack<T, VEC> a = gv_load<T, VEC, NT>(p + k * g.cs);
            const T xv = x[k * g.xs];
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[v] = gv_fma(a.v[v], xv, acc[v]);
        }
    } else {
#pragma unroll
        for (int v = 0; v < VEC; ++v)
            if (i + v < g.M)
                for (int64_t k = k0; k < k1; ++k) acc[v] = gv_fma(g.a[oa + (i + v) * g.rs + k * g.cs], x[k * g.xs], acc[v]);
    }
#pragma unroll
    for (int v = 0; v < VEC; ++v) red[wave][lane * VEC + v] = acc[v];
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * VEC; e += 256) {
        const int64_t o = (int64_t)blockIdx.x * 64 * VEC + e;
        if (o >= g.M) break;
        T s = red[0][e];
#pragma unroll
        for (int w = 1; w < 4; ++w) s = gv_add(s, red[w][e]);
        gv_put(g, oy, blockIdx.z, blockIdx.y, o, s);
    }
}

// Few outputs with many splits (dot products): one wave per output, four per block.
template <class T>
__global__ void __launch_bounds__(256) k_gemv_fin_wave(GemvArgs<T> g) {
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= g.M) return;
    int64_t oa, ox, oy;
    batch_offsets(g.bd, blockIdx.z, oa, ox, oy);
    const T* p = g.part + (int64_t)blockIdx.z * g.nsplit * g.M + i;
    T s = gv_zero<T>();
    for (int z = lane; z < g.nsplit; z += 64) s = gv_add(s, p[(int64_t)z * g.M]);
    s = gv_wave_sum(s);
    T* y = g.y + oy + i * g.ys;
    if (lane == 0) *y = gv_out(g, s, y);
}

template <class T>
__global__ void __launch_bounds__(256) k_gemv_fin(GemvArgs<T> g) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= g.M) return;
    int64_t oa, ox, oy;
    batch_offsets(g.bd, blockIdx.z, oa, ox, oy);
    const T* p = g.part + (int64_t)blockIdx.z * g.nsplit * g.M + i;
    T s = p[0];
    for (int z = 1; z < g.nsplit; ++z) s = gv_add(s, p[(int64_t)z * g.M]);
    T* y = g.y + oy + i * g.ys;
    *y = gv_out(g, s, y);
}

template <class T>
static void gemv_run(rstsr_hip_ctx* ctx, const GemmProblem& P, T alpha, T beta, bool beta_zero) {
    GemvArgs<T> g;
    const bool t = P.N != 1;  // one row: y^T = x^T B is y = B^T x
    g.M = t ? P.N : P.M;
    g.K = P.K;
    g.a = (const T*)(t ? P.b : P.a);
    g.rs = t ? P.csb : P.rsa;
    g.cs = t ? P.rsb : P.csa;
    g.x = (const T*)(t ? P.a : P.b);
    g.xs = t ? P.csa : P.rsb;
    g.y = (T*)P.c;
    g.ys = t ? P.csc : P.rsc;
    g.alpha = alpha;
    g.beta = beta;
    g.beta_zero = beta_zero ? 1 : 0;
    g.bd = P.bd;
    if (t)
        for (int d = 0; d < P.bd.nbd; ++d) std::swap(g.bd.sa[d], g.bd.sb[d]);
    constexpr int V16 = sizeof(T) >= 16 ? 1 : 16 / (int)sizeof(T);
    const uint32_t nb = (uint32_t)P.nbatch;
    const int64_t cu = std::max(ctx->num_cu, 1);
    // one output (a dot product) leaves the column kernel one lane
    const bool row = g.M == 1 || std::llabs(g.cs) <= std::llabs(g.rs);
    // waves per row group, outputs per block, k positions a split should have at least
    int wpr = 1, vec = 1;
    int64_t per, least;
    if (row) {
        vec = g.cs == 1 ? V16 : 1;
        // four waves per row group until the rows alone give four waves per CU
        wpr = (g.M * nb + GV_RPW - 1) / GV_RPW >= 4 * cu ? 1 : 4;
        per = GV_RPW * (4 / wpr);
        least = (int64_t)64 * vec * wpr * 4;
    } else {
        vec = g.rs == 1 ? V16 : 1;
        per = 64 * vec;
        least = 64;
    }
    // eight (row) or sixteen (col: one step per lane in flight instead of four rows) waves per CU
    const int64_t want = (row ? 2 : 4) * cu, have = (g.M + per - 1) / per * nb;
    int64_t ns = have >= want ? 1 : std::min<int64_t>((want + have - 1) / have, std::max<int64_t>(1, g.K / least));
    ns = std::min<int64_t>(ns, 1024);
    g.chunk = ((g.K + ns - 1) / ns + vec - 1) / vec * vec;
    g.nsplit = (int)((g.K + g.chunk - 1) / g.chunk);
    g.part = g.nsplit > 1 ? (T*)workspace(ctx, (size_t)nb * g.nsplit * g.M * sizeof(T)) : nullptr;
    const dim3 blk(256);
    using One = std::integral_constant<int, 1>;
    using Four = std::integral_constant<int, 4>;
    using Vec = std::integral_constant<int, V16>;
    // Streaming loads of A, which leave nothing in the last-level cache, unless A is small or shared by
    // batches (us, with and without: the same 32 MB f32 matrix again 6.8, 5.1, many in turn 7.6, 8.0; 200
    // MB f64 37, 32 and 38, 41; 512 MB 80, 91).
    bool once = (uint64_t)g.M * g.K * nb * sizeof(T) >= (40ull << 20);
    for (int d = 0; d < g.bd.nbd; ++d) once = once && g.bd.sa[d] != 0;
    // a launch holds fewer than 2^32 threads (16 per output at most): more outputs in pieces
    constexpr int64_t PIECE = (int64_t)1 << 27;
    for (int64_t i = 0; i < g.M; i += PIECE) {
        GemvArgs<T> q = g;
        q.M = std::min(PIECE, g.M - i);  // all of them where k is split
        q.a += i * g.rs;
        q.y += i * g.ys;
        const dim3 grid((uint32_t)((q.M + per - 1) / per), (uint32_t)g.nsplit, nb);
        auto rows = [&](auto v, auto w, auto nt) {
            constexpr int V = decltype(v)::value, W = decltype(w)::value;
            constexpr bool H = decltype(nt)::value;
            if (g.xs == 1) hipLaunchKernelGGL((k_gemv_row<T, V, W, true, H>), grid, blk, 0, ctx->stream, q);
            else hipLaunchKernelGGL((k_gemv_row<T, V, W, false, H>), grid, blk, 0, ctx->stream, q);
        };
        auto wide = [&](auto nt) {
            if (!row) hipLaunchKernelGGL((k_gemv_col<T, V16, decltype(nt)::value>), grid, blk, 0, ctx->stream, q);
            else if (wpr == 1) rows(Vec{}, One{}, nt);
            else rows(Vec{}, Four{}, nt);
        };
        if (vec > 1) {
            if constexpr (V16 > 1) once ? wide(std::true_type{}) : wide(std::false_type{});
        } else if (row) {
            wpr == 1 ? rows(One{}, One{}, std::false_type{}) : rows(One{}, Four{}, std::false_type{});
        } else {
            hipLaunchKernelGGL((k_gemv_col<T, 1, false>), grid, blk, 0, ctx->stream, q);
        }
        check_launch("gemv");
    }
    if (g.nsplit > 1) {
        if (g.nsplit >= 16 && g.M * nb <= 4096)
            hipLaunchKernelGGL(k_gemv_fin_wave<T>, dim3(ceil_div_u32((uint64_t)g.M, 4), 1, nb), blk, 0, ctx->stream, g);
        else
            hipLaunchKernelGGL(k_gemv_fin<T>, dim3(ceil_div_u32((uint64_t)g.M, 256), 1, nb), blk, 0, ctx->stream, g);
        check_launch("gemv split");
    }
}

bool gemv(rstsr_hip_ctx* ctx, rstsr_dtype_t t, const GemmProblem& P, const void* alpha, const void* beta, bool beta_zero) {
    if ((P.M != 1 && P.N != 1) || P.nbatch > 65535 || std::max(P.M, P.N) >= (1ll << 31)) return false;
    auto go = [&](auto tag) {
        using T = decltype(tag);
        T al, be;
        std::memcpy(&al, alpha, sizeof(T));
        std::memcpy(&be, beta, sizeof(T));
        gemv_run<T>(ctx, P, al, be, beta_zero);
        return true;
    };
    switch (t) {
        case RSTSR_F32: return go(float{});
        case RSTSR_F64: return go(double{});
        case RSTSR_I32: return go(int32_t{});
        case RSTSR_I64: return go(int64_t{});
        case RSTSR_C64: return go(c64{});
        case RSTSR_C128: return go(c128{});
        default: return false;
    }
}

}  // namespace hip
}  // namespace rstsr
