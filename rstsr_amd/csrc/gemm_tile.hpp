// Matrix-core GEMM tile for f32, f64, c64 and c128: one BM x BN tile of C per block,
// operands loaded straight from global memory into a ring of LDS buffers.
//
// What bounds it: the FP matrix cores (v_mfma_f32_16x16x4_f32 issues every 32 cycles per SIMD,
// v_mfma_f64_16x16x4_f64 every 64), if the operands arrive in time. So nothing is staged through
// registers (global_load_lds writes LDS itself), slices are 128 bytes of K per row and ST - 1 of
// them are in flight, one barrier per slice, and every fragment read is 16 bytes wide and free
// of bank conflicts.
//
// LDS image of a slice, per operand, 16-byte chunks (EPC elements each):
//   KC (the operand's K axis is the one chunks run along): one 128-byte row per m (or n), chunk c
//      of row r at chunk c ^ (r % 8), so that 8 neighbouring rows' chunk c (one fragment read)
//      lie in 8 distinct bank groups; a lane's chunk holds EPC consecutive k.
//   NC (chunks run along m or n): one row per k, unswizzled; a fragment read is contiguous over
//      lanes, and a lane's chunk holds neighbouring m (or n).
// Either way the image is linear in (load, thread), which is what the direct loads write.
//
// Measured (MI355X, TFLOP/s; before: f64 and c128 a register-staged tile, f32 and c64 one output per
// thread without matrix cores): f64 8192 x 8192 x 2048 69 (62), c128 4096^2 x 2048 69 (63), c64 the
// same 135 (about 5), f32 4096^3 134, f32 2000 x 1511 x 3001 111 (13.7).
//
// K order: step s of a slice multiplies, for e in 0 .. EPC - 1, the four positions
// k = (4 s + q) EPC + e, q = 0 .. 3, in one MFMA. It is the same for every layout, load width
// and tile shape, so the sum of an output does not depend on them.
#pragma once

#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"

namespace rstsr {
namespace hip {

typedef double tg_d4 __attribute__((ext_vector_type(4)));
typedef float tg_f4 __attribute__((ext_vector_type(4)));

// The matrix core of a real type: register r of lane l holds row `row(r, l)`, column l % 16.
template <class R>
struct Mma;
template <>
struct Mma<double> {
    using Acc = tg_d4;
    __device__ static Acc mma(double a, double b, Acc c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    __device__ static int row(int r, int lane) { return 4 * r + (lane >> 4); }
};
template <>
struct Mma<float> {
    using Acc = tg_f4;
    __device__ static Acc mma(float a, float b, Acc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    __device__ static int row(int r, int lane) { return 4 * (lane >> 4) + r; }
};

template <class T>
struct ElemOf {
    using R = T;
    static constexpr bool CX = false;
};
template <>
struct ElemOf<c64> {
    using R = float;
    static constexpr bool CX = true;
};
template <>
struct ElemOf<c128> {
    using R = double;
    static constexpr bool CX = true;
};

// WVM x WVN waves of (16 FM) x (16 FN) outputs each; OCC waves per SIMD in the register budget;
// ST LDS buffers per operand; SG: the second step's fragment reads are scheduled between the
// first step's MFMAs.
template <int WVM_, int WVN_, int FM_, int FN_, int OCC_, int ST_, bool SG_>
struct TCfg {
    static constexpr int WVM = WVM_, WVN = WVN_, FM = FM_, FN = FN_, OCC = OCC_, ST = ST_;
    static constexpr bool SG = SG_;
    static constexpr int NT = 64 * WVM * WVN, BM = 16 * WVM * FM, BN = 16 * WVN * FN;
};

template <class T>
struct TileGemmArgs {
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
    uint32_t batch0;
    int tri;           // symmetric product: only tiles with tm >= tn
    int64_t ksl;       // K slices per split (grid z); the whole K when not split
    typename ElemOf<T>::R* part;  // split: partial sums [split][batch][m][n] (complex: re, im)
    BatchDesc bd;
};

// 16 zero bytes a lane reads in place of positions past K
static __device__ const uint4 tg_zero = {0u, 0u, 0u, 0u};

// One operand's loads of a K slice into its LDS image. V16: the chunk axis has stride 1 and, for
// NC, the rows run upwards at least EPC apart, so chunks come by 16-byte loads (global addresses
// need 4-byte alignment only). A chunk that starts inside a row but ends past it reads into the
// next row, whose positions are not stored (NC) or belong to the operand (KC: only the last
// slice has such chunks); the last slice, after which no row is left to read into, comes by
// 4-byte words then, and so does every slice of operands of other strides. mn0: first row; MN: rows in all;
// smn, sk: strides in elements.
template <class T, bool KC, int BMN, int NT, bool V16>
struct SliceLoad {
    static constexpr int ES = sizeof(T), EPC = 16 / ES, BK = 128 / ES, WPE = ES / 4;
    template <int UNIT>  // bytes per lane and load
    struct Map {
        static constexpr int LOADS = BMN * 128 / (NT * UNIT);  // loads per thread
        static constexpr int RPL = NT * UNIT / 128;            // KC: rows per load
        static constexpr int UPR = BMN * ES / UNIT;            // NC: lanes per k row
        static constexpr int REP = UPR > NT ? UPR / NT : 1;    // NC: loads per k row
        static constexpr int KPL = UPR > NT ? 1 : NT / UPR;    // NC: k rows per load
        static_assert(LOADS >= 1 && BMN * 128 % (NT * UNIT) == 0, "slice loads");
        static_assert(KC ? RPL % 8 == 0 : (NT % UPR == 0 || UPR % NT == 0), "slice load shape");
        int row, k, sub;  // this thread's row and k of load 0, byte inside the element
        __device__ __forceinline__ explicit Map(int tid) {
            sub = 0;
            if constexpr (KC) {
                constexpr int LPR = 128 / UNIT, LPC = 16 / UNIT;  // lanes per row, per chunk
                row = tid / LPR;
                k = ((tid % LPR / LPC) ^ (row & 7)) * EPC;
                if constexpr (UNIT == 4) {
                    k += tid % 4 / WPE;
                    sub = tid % 4 % WPE * 4;
                }
            } else {
                const int u = UPR > NT ? tid : tid % UPR;
                k = UPR > NT ? 0 : tid / UPR;
                row = UNIT == 16 ? u * EPC : u / WPE;
                if constexpr (UNIT == 4) sub = u % WPE * 4;
            }
        }
        __device__ int row_of(int i) const { return KC ? row + i * RPL : row + i % REP * (NT * UNIT / ES); }
        __device__ int k_of(int i) const { return KC ? k : k + i / REP * KPL; }
    };
    static constexpr int U = V16 ? 16 : 4;
    static constexpr int LOADS = Map<U>::LOADS;  // the fewest loads a slice takes

    // Addresses of this thread's loads of the next slice. Rows past the last one repeat it (their
    // outputs are not stored), so that edge tiles load as others do: a bounds test per load and
    // slice made them take half as long again, and the launch waits for its slowest tile.
    const char* p[LOADS];
    const char* base;       // element (mn0, 0) of the operand
    int64_t smn, sk, next;  // strides in bytes, bytes from a slice to the next
    int64_t lim;            // MN - mn0: rows from mn0 on that exist

    __device__ __forceinline__ SliceLoad(const T* op, int64_t mn0, int64_t MN, int64_t smn_, int64_t sk_, int64_t k0) {
        smn = smn_ * ES;
        sk = sk_ * ES;
        next = BK * sk;
        lim = MN - mn0;
        base = (const char*)op + mn0 * smn;
        const Map<U> m(threadIdx.x);
        const int last = (int)min((int64_t)BMN, KC || U == 4 ? lim : (lim + EPC - 1) / EPC * EPC) - (KC || U == 4 ? 1 : EPC);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) p[i] = base + min(m.row_of(i), last) * smn + (k0 + m.k_of(i)) * sk + m.sub;
    }
    // every lane's UNIT bytes at p to LDS, lane l of the wave at lds + l UNIT
    template <int UNIT>
    __device__ static void to_lds(const char* p, char* lds) {
        if constexpr (UNIT == 16) __builtin_amdgcn_global_load_lds(p, lds, 16, 0, 0);
        else __builtin_amdgcn_global_load_lds(p, lds, 4, 0, 0);
    }
    // the next slice, which starts at k0, into the image at `lds`; positions past K as zeros
    __device__ __forceinline__ void issue(char* lds, int64_t k0, int64_t K) {
        const int wave = threadIdx.x >> 6;
        if (k0 + BK < K) {
#pragma unroll
            for (int i = 0; i < LOADS; ++i) {
                to_lds<U>(p[i], lds + (wave * 64 + i * NT) * U);
                p[i] += next;
            }
            return;
        }
        // the last slice; opaque: its index math must not be hoisted into registers of the slice loop
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const bool cut = KC ? K % EPC != 0 : lim < BMN && lim % EPC != 0;  // chunks that end past the row
        if (!V16 || !cut) {
            const Map<U> m(tid);
#pragma unroll
            for (int i = 0; i < LOADS; ++i)
                to_lds<U>(k0 + m.k_of(i) < K ? p[i] : (const char*)&tg_zero, lds + (wave * 64 + i * NT) * U);
        } else {
            const Map<4> m(tid);
#pragma unroll
            for (int i = 0; i < Map<4>::LOADS; ++i) {
                const int64_t r = min((int64_t)m.row_of(i), lim - 1), k = k0 + m.k_of(i);
                to_lds<4>(k < K ? base + r * smn + k * sk + m.sub : (const char*)&tg_zero, lds + (wave * 64 + i * NT) * 4);
            }
        }
    }
};

// wait until at most N of this wave's vector memory operations are outstanding and its LDS reads
// are done, then the block barrier
template <int N>
__device__ __forceinline__ void tg_wait_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <class T, class CF>
struct TileSmem {
    char a[CF::ST][CF::BM * 128];
    char b[CF::ST][CF::BN * 128];
};

// Fragments of one operand for one K step: F reads of 16 bytes (NC with F < EPC: narrower).
// get(i, e): the value of fragment i at the lane's position (4 s + q) EPC + e.
template <class T, bool KC, int F>
struct Frags {
    using R = typename ElemOf<T>::R;
    static constexpr int ES = sizeof(T), EPC = 16 / ES;
    // NC: neighbouring rows per read
    static constexpr int VN = F % EPC == 0 ? EPC : (F % 2 == 0 && EPC > 1 ? 2 : 1);
    struct Ch {
        T v[KC ? EPC : VN];
    };
    // A read as one vector of words: a struct read makes the compiler wait for every direct load
    // in flight before it (it cannot tell their buffers apart), which the barriers already order.
    typedef uint32_t Words __attribute__((ext_vector_type(sizeof(Ch) / 4)));
    __device__ static Ch read(const char* p) {
        const Words w = *(const Words*)p;
        Ch c;
        __builtin_memcpy(&c, &w, sizeof(Ch));
        return c;
    }
    static constexpr int NEAR = KC ? 1 : VN;  // fragments i .. i + NEAR - 1 hold neighbouring rows
    static constexpr int READS = KC ? F : EPC * (F / VN);
    Ch ch[READS];

    // wrow: first row of this wave in the image of MN rows
    template <int MN>
    __device__ __forceinline__ void load(const char* lds, int wrow, int s, int lane) {
        const int fr = lane & 15, q = lane >> 4;
        if constexpr (KC) {
            const char* p = lds + (wrow + fr) * 128 + (((4 * s + q) ^ (fr & 7)) << 4);
#pragma unroll
            for (int i = 0; i < F; ++i) ch[i] = read(p + i * 16 * 128);
        } else {
            const char* p = lds + ((4 * s + q) * EPC * MN + wrow + fr * VN) * ES;
#pragma unroll
            for (int e = 0; e < EPC; ++e)
#pragma unroll
                for (int g = 0; g < F / VN; ++g) ch[e * (F / VN) + g] = read(p + (e * MN + g * 16 * VN) * ES);
        }
    }
    __device__ __forceinline__ T get(int i, int e) const {
        if constexpr (KC) return ch[i].v[e];
        else return ch[e * (F / VN) + i / VN].v[i % VN];
    }
    // row of the wave's tile that index x (0 .. 15) of fragment i stands for
    __device__ static int row(int i, int x) {
        if constexpr (KC) return i * 16 + x;
        else return i / VN * 16 * VN + x * VN + i % VN;
    }
};

template <class T>
__device__ __forceinline__ T tg_axpby(T alpha, T x, T beta, const T* c, bool beta_zero) {
    if constexpr (!ElemOf<T>::CX) {
        T v = alpha * x;
        if (!beta_zero) v += beta * *c;
        return v;
    } else {
        T v{alpha.re * x.re - alpha.im * x.im, alpha.re * x.im + alpha.im * x.re};
        if (!beta_zero) {
            const T o = *c;
            v.re += beta.re * o.re - beta.im * o.im;
            v.im += beta.re * o.im + beta.im * o.re;
        }
        return v;
    }
}

// Where a tile's outputs go: C = alpha x + beta C. Symmetric products (tri, beta 0): the outputs on
// and below the diagonal, each also onto its mirror, so that no further pass reads C (f64 24000^2 x
// 1600: 13.8 ms, with a mirror kernel 14.6). Neighbouring outputs leave in one store where they are
// neighbours in C too (f64: half the store instructions).
// SCALE false: C = x (the partial sums of a K split).
template <class T, bool SCALE = true>
struct TileStore {
    T* c;
    int64_t rsc, csc, M, N;
    T alpha, beta;
    bool beta_zero, tri;

    __device__ __forceinline__ T value(T x, const T* p, bool bz) const {
        if constexpr (SCALE) return tg_axpby(alpha, x, beta, p, bz);
        else return x;
    }
    template <int V>
    __device__ __forceinline__ void pack(T* p, const T (&x)[V]) const {
        typedef uint32_t Words __attribute__((ext_vector_type(V * sizeof(T) / 4), aligned(4)));
        T y[V];
#pragma unroll
        for (int v = 0; v < V; ++v) y[v] = value(x[v], p, true);
        Words w;
        __builtin_memcpy(&w, y, sizeof(y));
        *(Words*)p = w;
    }
    // x[v] is output (m, n + v)
    template <int V>
    __device__ __forceinline__ void put(int64_t m, int64_t n, const T (&x)[V]) const {
        if (m >= M || n >= N) return;
        T* p = c + m * rsc + n * csc;
        if (V > 1 && csc == 1 && beta_zero && n + V <= (tri ? min(N, m + 1) : N)) {
            pack(p, x);
            return;
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (n + v < N && (!tri || n + v <= m)) p[v * csc] = value(x[v], p + v * csc, beta_zero);
    }
    // x[v] is output (m + v, n): its mirror, output (n, m + v)
    template <int V>
    __device__ __forceinline__ void mirror(int64_t m, int64_t n, const T (&x)[V]) const {
        if (m >= M || n >= N) return;
        T* p = c + n * rsc + m * csc;
        if (V > 1 && csc == 1 && m > n && m + V <= M) {
            pack(p, x);
            return;
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (m + v < M && m + v > n) p[v * csc] = value(x[v], p, true);
    }
};

// One C tile. A(m, k) at a + m rsa + k csa, B(k, n) at b + k rsb + n csb. AK / BKC: the operand's
// image is KC. Slices [sl0, sl1) of K.
template <class T, class CF, bool AK, bool BKC, bool V16, class Store>
__device__ __forceinline__ void tile_gemm(const T* A, int64_t rsa, int64_t csa, const T* B, int64_t rsb, int64_t csb,
                                          int64_t M, int64_t N, int64_t K, uint32_t tm, uint32_t tn, int64_t sl0,
                                          int64_t sl1, TileSmem<T, CF>& sm, const Store& store) {
    using R = typename ElemOf<T>::R;
    using MM = Mma<R>;
    using Acc = typename MM::Acc;
    constexpr bool CX = ElemOf<T>::CX;
    constexpr int NP = CX ? 2 : 1, FM = CF::FM, FN = CF::FN, ST = CF::ST, NT = CF::NT;
    constexpr int ES = sizeof(T), EPC = 16 / ES, BK = 128 / ES;
    using LA = SliceLoad<T, AK, CF::BM, NT, V16>;
    using LB = SliceLoad<T, BKC, CF::BN, NT, V16>;
    constexpr int NI = LA::LOADS + LB::LOADS;
    static_assert(ST >= 2 && (ST - 2) * NI < 64, "loads in flight");
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave / CF::WVN, wn = wave % CF::WVN;
    const int64_t m0 = (int64_t)tm * CF::BM, n0 = (int64_t)tn * CF::BN;
    LA la(A, m0, M, rsa, csa, sl0 * BK);
    LB lb(B, n0, N, csb, rsb, sl0 * BK);

    Acc acc[NP][FM][FN];
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[p][i][j][r] = 0;

    // the buffers are written only by the direct loads, which the compiler does not count as
    // stores: their address escapes here, so no read of them can be folded away as undefined
    asm volatile("" ::"v"(&sm) : "memory");
    auto issue = [&](int64_t sl, int st) {
        la.issue(sm.a[st], sl * BK, K);
        lb.issue(sm.b[st], sl * BK, K);
    };
    // waves whose outputs all lie past the matrix only take part in the loads and barriers
    const bool active = m0 + wm * 16 * FM < M && n0 + wn * 16 * FN < N;
    auto compute = [&](int st) {
        if (!active) return;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Frags<T, AK, FM> fa;
            Frags<T, BKC, FN> fb;
            fa.template load<CF::BM>(sm.a[st], wm * 16 * FM, s, lane);
            fb.template load<CF::BN>(sm.b[st], wn * 16 * FN, s, lane);
#pragma unroll
            for (int e = 0; e < EPC; ++e)
#pragma unroll
                for (int i = 0; i < FM; ++i)
#pragma unroll
                    for (int j = 0; j < FN; ++j) {
                        const T x = fa.get(i, e), y = fb.get(j, e);
                        if constexpr (!CX) {
                            acc[0][i][j] = MM::mma(x, y, acc[0][i][j]);
                        } else {
                            acc[0][i][j] = MM::mma(x.re, y.re, acc[0][i][j]);
                            acc[0][i][j] = MM::mma(-x.im, y.im, acc[0][i][j]);
                            acc[1][i][j] = MM::mma(x.re, y.im, acc[1][i][j]);
                            acc[1][i][j] = MM::mma(x.im, y.re, acc[1][i][j]);
                        }
                    }
        }
        if constexpr (CF::SG) {
            // order for the scheduler: step 0's reads, step 1's two MFMAs apart, the other MFMAs
            constexpr int NR = Frags<T, AK, FM>::READS + Frags<T, BKC, FN>::READS, NMF = FM * FN * EPC * (CX ? 4 : 1);
            constexpr int Q = NMF >= 2 * NR ? 2 : 1;
            if constexpr (Q * NR <= NMF) {
                __builtin_amdgcn_sched_group_barrier(0x100, NR, 0);
#pragma unroll
                for (int r = 0; r < NR; ++r) {
                    __builtin_amdgcn_sched_group_barrier(0x008, Q, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
                __builtin_amdgcn_sched_group_barrier(0x008, 2 * NMF - Q * NR, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // slice v lives in buffer v % ST, issued ST - 1 slices ahead
    const int64_t ns = sl1 - sl0;
#pragma unroll
    for (int s = 0; s < ST - 1; ++s)
        if (s < ns) issue(sl0 + s, s);
    if (ns >= ST - 1) tg_wait_barrier<(ST - 2) * NI>();
    else tg_wait_barrier<0>();
    int st = 0, sn = ST - 1;
    for (int64_t v = 0; v < ns; ++v) {
        const bool more = v + ST - 1 < ns;
        if (more) issue(sl0 + v + ST - 1, sn);
        compute(st);
        // slice v + 1 has landed (a slice takes at least NI loads), no wave reads buffer st any more
        if (more) tg_wait_barrier<(ST - 2) * NI>();
        else tg_wait_barrier<0>();
        st = st + 1 == ST ? 0 : st + 1;
        sn = sn + 1 == ST ? 0 : sn + 1;
    }
    // neighbouring columns (rows, for the mirror) that a lane holds, NC images, in one store each
    constexpr int VB = Frags<T, BKC, FN>::NEAR, VA = Frags<T, AK, FM>::NEAR;
    auto value = [&](int i, int j, int r) {
        if constexpr (CX) return T{acc[0][i][j][r], acc[1][i][j][r]};
        else return (T)acc[0][i][j][r];
    };
    const int64_t mw = m0 + wm * 16 * FM, nw = n0 + wn * 16 * FN;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t gm = mw + Frags<T, AK, FM>::row(i, MM::row(r, lane));
#pragma unroll
            for (int j = 0; j < FN; j += VB) {
                T x[VB];
#pragma unroll
                for (int v = 0; v < VB; ++v) x[v] = value(i, j + v, r);
                store.put(gm, nw + Frags<T, BKC, FN>::row(j, lane & 15), x);
            }
        }
    if (store.tri) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int64_t gn = nw + Frags<T, BKC, FN>::row(j, lane & 15);
#pragma unroll
            for (int i = 0; i < FM; i += VA)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    T x[VA];
#pragma unroll
                    for (int v = 0; v < VA; ++v) x[v] = value(i + v, j, r);
                    store.mirror(mw + Frags<T, AK, FM>::row(i, MM::row(r, lane)), gn, x);
                }
        }
    }
}

// Grid: x tiles, y batches (from batch0), z splits of K.
template <class T, class CF, bool AK, bool BKC, bool V16, bool SPLIT>
__global__ void __launch_bounds__(CF::NT, CF::OCC) k_gemm_tile(TileGemmArgs<T> g, const int* run_if) {
    if (run_if && *run_if == 0) return;
    __shared__ __attribute__((aligned(16))) TileSmem<T, CF> sm;
    constexpr int BK = 128 / (int)sizeof(T);
    uint32_t tm, tn;
    if (g.tri) {
        tri_coords(xcd_remap8(blockIdx.x, g.tiles_m * (g.tiles_m + 1) / 2), tm, tn);
    } else {
        tile_coords<8>(blockIdx.x, g.tiles_m, g.tiles_n, tm, tn);
    }
    int64_t oa, ob, oc;
    batch_offsets(g.bd, g.batch0 + blockIdx.y, oa, ob, oc);
    const int64_t nsl = (g.K + BK - 1) / BK;
    const int64_t sl0 = SPLIT ? (int64_t)blockIdx.z * g.ksl : 0;
    const int64_t sl1 = SPLIT ? min(nsl, sl0 + g.ksl) : nsl;
    const TileStore<T, !SPLIT> st =
        SPLIT ? TileStore<T, !SPLIT>{(T*)g.part + ((int64_t)blockIdx.z * gridDim.y + blockIdx.y) * g.M * g.N,
                                     g.N, 1, g.M, g.N, T{}, T{}, true, false}
              : TileStore<T, !SPLIT>{g.c + oc, g.rsc, g.csc, g.M, g.N, g.alpha, g.beta, g.beta_zero != 0, g.tri != 0};
    tile_gemm<T, CF, AK, BKC, V16>(g.a + oa, g.rsa, g.csa, g.b + ob, g.rsb, g.csb, g.M, g.N, g.K, tm, tn, sl0, sl1, sm,
                                   st);
}

// One problem of a grouped launch.
template <class T>
struct TileProblem {
    int64_t M, N, K;
    const T* a;
    int64_t rsa, csa;
    const T* b;
    int64_t rsb, csb;
    T* c;
    int64_t rsc, csc;
    uint32_t tiles_n;
};

// Block id -> tile, so that each XCD (blocks go to them in turn) takes runs of RUN neighbouring tiles,
// whose operand panels its L2 then holds once, while the launch as a whole still walks the tiles
// in order. The last, incomplete round is not reordered. (512 uneven f64 GEMMs: runs of 1 tile
// 2.85 ms, of 8 2.83, of 16 2.80, of 32 2.82.)
template <uint32_t RUN>
__device__ __forceinline__ uint32_t xcd_runs(uint32_t b, uint32_t n) {
    constexpr uint32_t R = 8 * RUN;
    if (b >= n / R * R) return b;
    const uint32_t i = b % R;
    return b - i + i % 8 * RUN + i / 8;
}

// Uneven GEMMs of one form in one launch. Problem g owns tiles [prefix[g], prefix[g+1]); the blocks
// are dispatched in tile order, each as soon as a CU has room for it, which is the queue a
// persistent grid would keep by hand, without the registers its loop takes from the tile's.
template <class T, class CF, bool AK, bool BKC, bool V16>
__global__ void __launch_bounds__(CF::NT, CF::OCC) k_gemm_tile_grouped(const TileProblem<T>* __restrict__ probs, int count,
                                                                       const uint32_t* __restrict__ prefix, T alpha,
                                                                       T beta, int beta_zero,
                                                                       const int* __restrict__ run_if) {
    if (run_if && *run_if == 0) return;
    __shared__ __attribute__((aligned(16))) TileSmem<T, CF> sm;
    constexpr int BK = 128 / (int)sizeof(T);
    const uint32_t tile = xcd_runs<16>(blockIdx.x, gridDim.x);
    // problem of this tile: last g with prefix[g] <= tile
    int lo = 0, hi = count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (prefix[mid] <= tile) lo = mid;
        else hi = mid - 1;
    }
    const TileProblem<T> p = probs[lo];
    const uint32_t local = tile - prefix[lo], tm = local / p.tiles_n, tn = local - tm * p.tiles_n;
    tile_gemm<T, CF, AK, BKC, V16>(p.a, p.rsa, p.csa, p.b, p.rsb, p.csb, p.M, p.N, p.K, tm, tn, 0, (p.K + BK - 1) / BK,
                                   sm, TileStore<T>{p.c, p.rsc, p.csc, p.M, p.N, alpha, beta, beta_zero != 0, false});
}

// C = alpha (sum of the partials, in split order) + beta C; symmetric products (tri): of the
// outputs (m, n) and (n, m) both take the sums of the one on or below the diagonal
template <class T>
__global__ void __launch_bounds__(256) k_gemm_split_fin(TileGemmArgs<T> g, int nsplit, uint32_t nb, const int* run_if) {
    if (run_if && *run_if == 0) return;
    const int64_t mn = g.M * g.N, e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= mn) return;
    const int64_t m = e / g.N, n = e - m * g.N;
    const T* P = (const T*)g.part + (int64_t)blockIdx.y * mn + (g.tri && n > m ? n * g.N + m : e);
    T s = P[0];
    for (int z = 1; z < nsplit; ++z) {
        const T x = P[(int64_t)z * nb * mn];
        if constexpr (ElemOf<T>::CX) {
            s.re += x.re;
            s.im += x.im;
        } else {
            s += x;
        }
    }
    int64_t oa, ob, oc;
    batch_offsets(g.bd, g.batch0 + blockIdx.y, oa, ob, oc);
    T* cp = g.c + oc + m * g.rsc + n * g.csc;
    *cp = tg_axpby(g.alpha, s, g.beta, cp, g.beta_zero != 0);
}

}  // namespace hip
}  // namespace rstsr
