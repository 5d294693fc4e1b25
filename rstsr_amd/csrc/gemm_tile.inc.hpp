// Host side of the matrix-core tile GEMM (gemm_tile.hpp): layouts, load width, tile shape and
// K split of one call. Included by the files that instantiate it, one element type each.
#pragma once

#include <cstdio>
#include <functional>
#include <string>

#include "gemm_tile.hpp"

namespace rstsr {
namespace hip {

// 64 x 64 tiles: K splits, and operands read by words (whose loads leave the registers of larger
// tiles no room); 32 x 32 ones for the latter where 64 x 64 leave most of the chip idle
template <class T>
using TileMid = TCfg<2, 2, 2, 2, 4, 2, !std::is_same<T, double>::value>;
using TileLow = TCfg<2, 2, 1, 1, 2, 6, false>;

template <class T, class CF, bool V16, bool SPLIT>
static void tile_gemm_launch(rstsr_hip_ctx* ctx, TileGemmArgs<T> g, uint32_t nb, uint32_t nsplit, bool ak, bool bk,
                             const int* run_if) {
    g.tiles_m = ceil_div_u32(g.M, CF::BM);
    g.tiles_n = ceil_div_u32(g.N, CF::BN);
    uint64_t nt = (uint64_t)g.tiles_m * g.tiles_n;
    if (g.tri) nt = (uint64_t)g.tiles_m * (g.tiles_m + 1) / 2;
    if (nt >= (1ull << 31) || nt * CF::NT >= (1ull << 32)) RSTSR_RAISE(UnImplemented, "GEMM grid too large");
    auto go = [&](auto a, auto b) {
        hipLaunchKernelGGL((k_gemm_tile<T, CF, decltype(a)::value, decltype(b)::value, V16, SPLIT>),
                           dim3((uint32_t)nt, nb, nsplit), dim3(CF::NT), 0, ctx->stream, g, run_if);
    };
    using Y = std::true_type;
    using F = std::false_type;
    if (ak && bk) go(Y{}, Y{});
    else if (ak) go(Y{}, F{});
    else if (bk) go(F{}, Y{});
    else go(F{}, F{});
    check_launch("gemm");
}

// Whether an operand can be read by 16-byte chunks (SliceLoad's V16). kc: chunks along K (stride sk),
// else along m or n (stride smn).
template <class T>
static bool tile_chunks(bool kc, int64_t sk, int64_t smn) {
    return kc ? sk == 1 : smn == 1 && sk >= 16 / (int64_t)sizeof(T);
}

// Splits of K for a product whose 64 x 64 tiles leave most of the chip idle: enough blocks for
// two per CU, each at least eight slices long. Shorter K than the lines below goes to 32 x 32 tiles
// unsplit, which need no second launch (us, split against not; K of 24, 32 and 40 slices): f64
// 128^2 12.6, 13.0, 13.0 against 12.1, 15.1, 17.9; 512^2 15.4, 17.3, 20.9 against 12.7, 15.8, 18.7;
// 256 x 1600 21.3, 21.8, 22.2 against 16.4, 20.4, 24.2; f32 and c64 alike, c128 1000 x 400 at 40 and 48
// 38.7, 42.3 against 32.2, 37.6. By sizes only, so that a product rounds the same whatever its strides
// and load width.
template <class T>
static uint32_t tile_gemm_splits(const rstsr_hip_ctx* ctx, const GemmProblem& P) {
    const int64_t nsl = (P.K * (int64_t)sizeof(T) + 127) / 128;
    const int64_t t = ((P.M + 63) / 64) * ((P.N + 63) / 64) * (int64_t)P.nbatch;
    const int64_t cu = std::max(ctx->num_cu, 1);
    if (t >= cu || nsl < (4 * t < cu ? 28 : sizeof(T) == 16 ? 56 : 40)) return 1;
    return (uint32_t)std::max<int64_t>(1, std::min<int64_t>({(2 * cu + t - 1) / t, nsl / 8, 64}));
}

// Tile shapes of one element type, in the tuner's order. Measured (TFLOP/s of a large product, 16-byte
// loads): two or more blocks per CU are needed to cover the slice boundaries, so the register budget
// decides.
template <class T>
struct TileShapes;
template <>
struct TileShapes<float> {
    using S0 = TCfg<2, 2, 4, 4, 2, 2, true>;   // 128 x 128, 4 waves of 64 x 64: 130 TF
    using S1 = TCfg<2, 2, 2, 2, 4, 2, true>;   // 64 x 64: 122 TF
    using S2 = TCfg<2, 2, 1, 1, 2, 6, false>;  // 32 x 32
    using S3 = S1;
    static constexpr int COUNT = 3;
};
template <>
struct TileShapes<c64> {
    using S0 = TCfg<2, 2, 2, 2, 4, 2, true>;   // 64 x 64: 130 TF (128 x 128 of 64 x 64 waves: 99)
    using S1 = TCfg<2, 2, 1, 1, 2, 6, false>;  // 32 x 32
    using S2 = S0;
    using S3 = S0;
    static constexpr int COUNT = 2;
};
template <>
struct TileShapes<double> {
    using S0 = TCfg<4, 2, 2, 4, 4, 2, false>;  // 128 x 128, 8 waves of 32 x 64: 69 TF
    using S1 = TCfg<2, 2, 1, 1, 2, 6, false>;  // 32 x 32
    using S2 = TCfg<2, 2, 4, 4, 2, 2, true>;   // 128 x 128, 4 waves of 64 x 64: 68 TF
    using S3 = TCfg<2, 2, 2, 2, 4, 2, false>;  // 64 x 64: 65 TF
    static constexpr int COUNT = 4;
};
template <>
struct TileShapes<c128> {
    using S0 = TCfg<2, 2, 2, 2, 4, 2, true>;   // 64 x 64: 69 TF
    using S1 = TCfg<4, 2, 2, 4, 2, 2, true>;   // 128 x 128: 70 TF
    using S2 = TCfg<2, 2, 1, 1, 2, 6, false>;  // 32 x 32
    using S3 = S0;
    static constexpr int COUNT = 3;
};

// Tile shapes of grouped launches, in the tuner's order; MID is the untuned one.
template <class T>
struct TileGroupedShapes;
template <>
struct TileGroupedShapes<double> {
    using S0 = TCfg<4, 2, 2, 4, 4, 2, false>;  // 128 x 128
    using S1 = TCfg<2, 2, 2, 4, 3, 2, false>;  // 64 x 128
    using S2 = TCfg<2, 2, 2, 2, 4, 2, false>;  // 64 x 64
    using S3 = TCfg<2, 2, 4, 4, 2, 2, true>;
    static constexpr int COUNT = 4, MID = 2;
};
template <>
struct TileGroupedShapes<c128> {
    using S0 = TCfg<2, 2, 2, 2, 4, 2, true>;   // 64 x 64
    using S1 = TCfg<2, 2, 1, 1, 2, 6, false>;  // 32 x 32
    using S2 = S0;
    using S3 = S0;
    static constexpr int COUNT = 2, MID = 0;
};

// Index of the first shape of BM (the next smaller one the type has).
template <class T>
static int tile_shape_index(int bm) {
    using S = TileShapes<T>;
    const int b[4] = {S::S0::BM, S::S1::BM, S::S2::BM, S::S3::BM};
    for (int want = bm; want >= 32; want /= 2)
        for (int i = 0; i < S::COUNT; ++i)
            if (b[i] == want) return i;
    return 0;
}

template <class T>
static void tile_gemm_run(rstsr_hip_ctx* ctx, const char* tag, const GemmProblem& P, T alpha, T beta, bool beta_zero,
                          const int* run_if) {
    using S = TileShapes<T>;
    TileGemmArgs<T> g;
    g.M = P.M;
    g.N = P.N;
    g.K = P.K;
    g.a = (const T*)P.a;
    g.rsa = P.rsa;
    g.csa = P.csa;
    g.b = (const T*)P.b;
    g.rsb = P.rsb;
    g.csb = P.csb;
    g.c = (T*)P.c;
    g.rsc = P.rsc;
    g.csc = P.csc;
    g.alpha = alpha;
    g.beta = beta;
    g.beta_zero = beta_zero ? 1 : 0;
    g.part = nullptr;
    g.ksl = 0;
    g.bd = P.bd;
    // an operand's chunks run along its unit-stride axis (the smaller stride when neither is 1)
    const bool ak = std::llabs(P.csa) <= std::llabs(P.rsa), bk = std::llabs(P.rsb) <= std::llabs(P.csb);
    const bool v16 = tile_chunks<T>(ak, P.csa, P.rsa) && tile_chunks<T>(bk, P.rsb, P.csb);
    bool syrk = beta_zero && run_if == nullptr && P.a == P.b && P.M == P.N && P.rsa == P.csb && P.csa == P.rsb;
    for (int d = 0; d < P.bd.nbd && syrk; ++d) syrk = P.bd.sa[d] == P.bd.sb[d];
    const uint64_t YMAX = 65535;
    const uint32_t ns = run_if ? 1 : tile_gemm_splits<T>(ctx, P);
    if (ns > 1) {
        const int64_t nsl = (P.K * (int64_t)sizeof(T) + 127) / 128;
        g.ksl = (nsl + ns - 1) / ns;
        const uint32_t nsplit = ceil_div_u32((uint64_t)nsl, (uint64_t)g.ksl);
        const uint32_t nb = (uint32_t)P.nbatch;  // fewer than one block per CU in all
        g.tri = 0;
        g.batch0 = 0;
        g.part = (typename ElemOf<T>::R*)workspace(ctx, (size_t)nsplit * nb * P.M * P.N * sizeof(T));
        if (v16) tile_gemm_launch<T, TileMid<T>, true, true>(ctx, g, nb, nsplit, ak, bk, run_if);
        else tile_gemm_launch<T, TileMid<T>, false, true>(ctx, g, nb, nsplit, ak, bk, run_if);
        g.tri = syrk ? 1 : 0;
        hipLaunchKernelGGL(k_gemm_split_fin<T>, dim3(ceil_div_u32((uint64_t)P.M * P.N, 256), nb), dim3(256), 0,
                           ctx->stream, g, (int)nsplit, nb, run_if);
        check_launch("gemm split");
        return;
    }
    const int big = tile_shape_index<T>(128), mid = tile_shape_index<T>(64), small = tile_shape_index<T>(32);
    // a launch holds fewer than 2^32 threads: outputs of 2^34 elements and more only fit the larger tiles
    const int bms[4] = {S::S0::BM, S::S1::BM, S::S2::BM, S::S3::BM}, nts[4] = {S::S0::NT, S::S1::NT, S::S2::NT, S::S3::NT};
    auto fits = [&](int c) {
        const uint64_t bm = (uint64_t)bms[c], tm = (P.M + bm - 1) / bm, tn = (P.N + bm - 1) / bm;
        return tm * tn * (uint64_t)nts[c] < (1ull << 32);
    };
    auto run = [&](int c) {
        if (!fits(c)) c = big;
        for (uint64_t b0 = 0; b0 < P.nbatch; b0 += YMAX) {
            g.batch0 = (uint32_t)b0;
            g.tri = syrk ? 1 : 0;
            const uint32_t nb = (uint32_t)std::min<uint64_t>(YMAX, P.nbatch - b0);
            auto go = [&](auto cf) {
                tile_gemm_launch<T, decltype(cf), true, false>(ctx, g, nb, 1, ak, bk, run_if);
            };
            if (!v16 && c == small) tile_gemm_launch<T, TileLow, false, false>(ctx, g, nb, 1, ak, bk, run_if);
            else if (!v16) tile_gemm_launch<T, TileMid<T>, false, false>(ctx, g, nb, 1, ak, bk, run_if);
            else if (c == 0) go(typename S::S0{});
            else if (c == 1) go(typename S::S1{});
            else if (c == 2) go(typename S::S2{});
            else go(typename S::S3{});
        }
    };
    // untuned: the largest tile that still gives every CU a block
    const int64_t cu = std::max(ctx->num_cu, 1);
    auto tiles = [&](int64_t s) { return ((P.M + s - 1) / s) * ((P.N + s - 1) / s) * (int64_t)P.nbatch; };
    const int heur = tiles(128) >= cu ? big : (tiles(64) >= cu / 2 ? mid : small);
    auto bkt = [](int64_t x) {
        int b = 0;
        while ((1ll << b) < x) ++b;
        return b;
    };
    char key[160];
    std::snprintf(key, sizeof(key), "gemm:%s:m%d:n%d:k%d:b%d:f%d", tag, bkt(P.M), bkt(P.N), bkt(P.K), bkt((int64_t)P.nbatch),
                  (ak ? 1 : 0) | (bk ? 2 : 0) | (v16 ? 4 : 0) | (syrk ? 8 : 0));
    tune_select(ctx, key, S::COUNT, heur, beta_zero && run_if == nullptr && v16, std::function<void(int)>(run));
}

template <class T, class CF>
static void tile_grouped_launch(rstsr_hip_ctx* ctx, const std::vector<GemmProblem>& probs, T alpha, T beta,
                                bool beta_zero, const int* run_if) {
    // one launch per form present (row-major operands are all of form 1): bit 0 A's image is KC,
    // bit 1 B's; form 4: some operand has no 16-byte loads. Within a launch the longest K (the time of
    // one tile) goes first, so that short tiles fill the end of the launch instead of a few long ones
    // trailing it. Each problem writes only its own C, so the order changes no result.
    std::vector<uint32_t> form(probs.size()), order(probs.size());
    for (size_t i = 0; i < probs.size(); ++i) {
        const GemmProblem& P = probs[i];
        const bool ak = std::llabs(P.csa) <= std::llabs(P.rsa), bk = std::llabs(P.rsb) <= std::llabs(P.csb);
        const bool v16 = tile_chunks<T>(ak, P.csa, P.rsa) && tile_chunks<T>(bk, P.rsb, P.csb);
        form[i] = v16 ? (ak ? 1u : 0u) | (bk ? 2u : 0u) : 4u;
        order[i] = (uint32_t)i;
    }
    std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) {
        return form[x] != form[y] ? form[x] < form[y] : probs[x].K > probs[y].K;
    });
    // table: the problems in launch order, then for each of them its first tile within its launch
    const size_t n = probs.size(), poff = (n * sizeof(TileProblem<T>) + 255) & ~(size_t)255;
    const size_t bytes = poff + n * sizeof(uint32_t);
    char* meta = (char*)aux_buffer(ctx, bytes + 256);
    char* host = (char*)meta_stage(ctx, bytes, "grouped GEMM");
    TileProblem<T>* gp = (TileProblem<T>*)host;
    uint32_t* prefix = (uint32_t*)(host + poff);
    uint64_t total[5] = {};
    size_t first[6] = {};
    for (size_t i = 0; i < n; ++i) {
        const GemmProblem& P = probs[order[i]];
        const uint32_t f = form[order[i]], tm = ceil_div_u32(P.M, CF::BM), tn = ceil_div_u32(P.N, CF::BN);
        gp[i] = TileProblem<T>{P.M, P.N, P.K, (const T*)P.a, P.rsa, P.csa, (const T*)P.b, P.rsb, P.csb, (T*)P.c,
                               P.rsc, P.csc, tn};
        prefix[i] = (uint32_t)total[f];
        total[f] += (uint64_t)tm * tn;
        if (total[f] >= (1ull << 31)) RSTSR_RAISE(UnImplemented, "grouped GEMM has too many tiles");
        for (uint32_t g = f + 1; g < 6; ++g) first[g] = i + 1;
    }
    meta_upload(ctx, meta, bytes);
    auto launch = [&](uint32_t f, auto ak, auto bk, auto v16) {
        if (total[f] == 0) return;
        hipLaunchKernelGGL((k_gemm_tile_grouped<T, CF, decltype(ak)::value, decltype(bk)::value, decltype(v16)::value>),
                           dim3((uint32_t)total[f]), dim3(CF::NT), 0, ctx->stream,
                           (const TileProblem<T>*)meta + first[f], (int)(first[f + 1] - first[f]),
                           (const uint32_t*)(meta + poff) + first[f], alpha, beta, beta_zero ? 1 : 0, run_if);
        check_launch("grouped gemm");
    };
    using Y = std::true_type;
    using F = std::false_type;
    launch(0, F{}, F{}, Y{});
    launch(1, Y{}, F{}, Y{});
    launch(2, F{}, Y{}, Y{});
    launch(3, Y{}, Y{}, Y{});
    launch(4, Y{}, Y{}, F{});
}

// C_g = alpha A_g B_g + beta C_g of every problem (K > 0). With run_if (as for plain_dgemm) a fixed
// tile shape, since the tuner cannot time a launch that may not run.
template <class T>
static void tile_grouped_run(rstsr_hip_ctx* ctx, const char* tag, const std::vector<GemmProblem>& probs, T alpha, T beta,
                             bool beta_zero, const int* run_if) {
    if (probs.empty()) return;
    using S = TileGroupedShapes<T>;
    auto run = [&](int c) {
        auto go = [&](auto cf) { tile_grouped_launch<T, decltype(cf)>(ctx, probs, alpha, beta, beta_zero, run_if); };
        if (c == 0) go(typename S::S0{});
        else if (c == 1) go(typename S::S1{});
        else if (c == 2) go(typename S::S2{});
        else go(typename S::S3{});
    };
    if (run_if) {
        run(S::MID);
        return;
    }
    double mean = 0;
    int64_t work = 0, tiles = 0, area128 = 0, area64 = 0;  // areas: tiled outputs times K
    for (auto& p : probs) {
        mean += (double)std::min(p.M, p.N);
        work += p.M * p.N * p.K;
        const int64_t t = ((p.M + 127) / 128) * ((p.N + 127) / 128);
        tiles += t;
        area128 += 4 * t * p.K;
        area64 += ((p.M + 63) / 64) * ((p.N + 63) / 64) * p.K;
    }
    // Enough 128 x 128 tiles to keep every CU busy for many rounds, and at most a fifth more work in them
    // than in 64 x 64 ones (512 problems of 32 to 1024: a ninth): always the largest tile, which the
    // tuner's two timed runs at a changing clock miss by a few per cent (ms, 128 x 128 against 64 x 64:
    // 10700 tiles 2.72 and 2.88, 5000 tiles 1.98 and 2.11; 830 tiles 0.188 and 0.156; with more padding
    // 4500 problems of 140 1.37 and 0.79, 2500 of 192 1.01 and 0.64, 1200 of 260 1.24 and 1.07, 4500 of 48
    // 0.122 and 0.084).
    if (std::is_same<T, double>::value && tiles >= 16 * (int64_t)std::max(ctx->num_cu, 1) &&
        5 * area128 <= 6 * area64) {
        run(0);
        return;
    }
    mean /= (double)probs.size();
    auto bkt = [](int64_t x) {
        int b = 0;
        while ((1ll << b) < x) ++b;
        return b;
    };
    char key[160];
    std::snprintf(key, sizeof(key), "grouped:%s:n%d:mean%d:work%d", tag, bkt((int64_t)probs.size()), bkt((int64_t)mean),
                  bkt(work));
    tune_select(ctx, key, S::COUNT, S::MID, beta_zero, std::function<void(int)>(run));
}

}  // namespace hip
}  // namespace rstsr
