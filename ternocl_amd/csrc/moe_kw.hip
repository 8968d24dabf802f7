// moe_kw.hip -- the MoE prefill's grouped GEMMs for experts of few rows on gfx950
// (int2_moe/int2_moe_prefill.cl:72-141 and the layer sequence of
// int2_moe/prefill.cpp:268-279): the K walk over waves of int2_gemm_kw.hip
// (gemm_kw.hpp) on each expert's rows.
//
// With a few rows an expert (T = 16, 128 experts, top-8: one or two) the 128-row
// tiles stage and multiply mostly nothing and walk K stage by stage behind a
// barrier: ~32 us a GEMM whatever T is.  Here a workgroup of four waves takes 32 of
// an expert's rows and a strip of its columns, each wave a quarter of K.
// It finds its expert from the route's row offsets (a count and a scan over the
// experts, 64 a step), so the route and its tile list stay as they are.
#include "gemm_kw.hpp"

#include <algorithm>
#include <cmath>

namespace tcl {
int moe_bn(int N, int widest);  // int2_gemm_mfma.hip
namespace {

// The expert and the first row (within it) of row tile `tile`, tiles of bm rows
// numbered expert by expert; false past the last.
__device__ __forceinline__ bool moe_kw_tile(const int *meta, int E, int bm, int tile, int &e, int &first) {
    const int lane = threadIdx.x & 63;
    int before = 0;  // tiles of the experts already passed
    for (int b = 0; b < E; b += 64) {
        const int i = b + lane;
        const int rows = i < E ? max(meta[i + 1] - meta[i], 0) : 0, t = (rows + bm - 1) / bm;
        int s = t;  // inclusive scan
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int x = __shfl_up(s, o);
            if (lane >= o) s += x;
        }
        // the experts of this step whose tiles all come before
        const unsigned long long past = __ballot(before + s <= tile);
        const int n = __builtin_popcountll(past);
        if (n < 64) {
            e = __builtin_amdgcn_readfirstlane(b + n);
            if (e >= E) return false;
            first = __builtin_amdgcn_readfirstlane((tile - before - (n ? __shfl(s, n - 1) : 0)) * bm);
            return true;
        }
        before += __shfl(s, 63);
    }
    return false;
}

// C rows (expert-sorted) of one tile: A rows perm[p] / topk of A_all with perm,
// else its sorted rows; expert e's weights B_all + e (K / 16) N.  DUAL: B2 / S2 the
// gate, B / S the up projection, C = DT(silu(gate) * DT(up)).
template <class Cfg, bool BF16, bool DUAL>
__global__ void __launch_bounds__(Cfg::THREADS)
k_moe_gemm_kw(const int *__restrict__ meta, const uint16_t *__restrict__ A_all, const int *__restrict__ perm, int topk,
              const uint32_t *__restrict__ B_all, const uint16_t *__restrict__ S_all, const uint32_t *__restrict__ B2_all,
              const uint16_t *__restrict__ S2_all, void *__restrict__ C_all, const uint16_t *__restrict__ Other_all, int E,
              int G, int arows, int N, int K, int postop, int out_f32, int ntn) {
    constexpr int MB = Cfg::MB, CB = Cfg::CB, CS = DUAL ? CB / 2 : CB;
    static_assert(Cfg::WM == 1, "one wave row");
    extern __shared__ __attribute__((aligned(16))) uint8_t kw_lds[];
    const int tile = blockIdx.x / ntn, tn = blockIdx.x - tile * ntn;
    int e, first;
    if (!moe_kw_tile(meta, E, Cfg::BM, tile, e, first)) return;  // whole workgroup: past the last tile
    const int row0 = __builtin_amdgcn_readfirstlane(meta[e]) + first;
    if ((unsigned)row0 >= (unsigned)G) return;
    // (rows and gathered rows stay below G and arows whatever meta and perm hold)
    const int mrows = min(min(Cfg::BM, __builtin_amdgcn_readfirstlane(meta[e + 1]) - row0), G - row0);
    if (mrows < 1) return;
    const int n0 = tn * 32 * CS;
    const int lane = threadIdx.x & 63, kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 31, q = lane >> 5;
    const int units = K / 64, u0 = units * kw / Cfg::WK, u1 = units * (kw + 1) / Cfg::WK;
    uint32_t va[4 * MB];
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i) {
        const int r = row0 + min((lane >> 3) + 8 * i, mrows - 1);
        const uint32_t src = (uint32_t)(perm ? perm[r] / topk : r);
        va[i] = min(src, (uint32_t)arows - 1u) * (uint32_t)K + 8u * (lane & 7);
    }
    const uint32_t col = (uint32_t)min(n0 + CS * c, N - CS);
    const size_t bo = (size_t)e * (K / 16) * N, so = (size_t)e * (K / kGS) * N;
    f32x16_t acc[MB][CB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[mb][cb] = f32x16_t{};
    if constexpr (DUAL) {
        KwDual<CB, Cfg::PF> bs{{B_all + bo, S_all + so, N, units, col, q}, {B2_all + bo, S2_all + so, N, units, col, q}};
        kw_walk<Cfg, BF16>(kw_lds + kw * (MB * 8192), A_all, va, u0, u1, units, bs, acc);
    } else {
        KwInt2<CB, Cfg::PF> bs(B_all + bo, S_all + so, N, units, col, q);
        kw_walk<Cfg, BF16>(kw_lds + kw * (MB * 8192), A_all, va, u0, u1, units, bs, acc);
    }
    kw_finish<Cfg, BF16, DUAL>(acc, kw_lds, C_all, Other_all, nullptr, 0, N, row0, mrows, n0, postop, out_f32, 1, 0, nullptr,
                               nullptr);
}

template <class Cfg, bool BF16, bool DUAL>
void moe_kw_launch(const int *meta, const void *A, const int *perm, int topk, const uint32_t *B, const void *S,
                   const uint32_t *B2, const void *S2, void *C, const void *Other, int E, int G, int N, int K, int postop,
                   int out_f32, hipStream_t st) {
    const int bn = 32 * (DUAL ? Cfg::CB / 2 : Cfg::CB), ntn = (N + bn - 1) / bn;
    // each expert's last rows add at most one tile to the full ones
    const int tiles = std::min(G, G / Cfg::BM + std::min(E, G));
    hipLaunchKernelGGL((k_moe_gemm_kw<Cfg, BF16, DUAL>), dim3((unsigned)tiles * ntn), dim3(Cfg::THREADS), Cfg::LDS_BYTES, st,
                       meta, (const uint16_t *)A, perm, topk, B, (const uint16_t *)S, B2, (const uint16_t *)S2, C,
                       (const uint16_t *)Other, E, G, perm ? std::max(1, G / topk) : G, N, K, postop, out_f32, ntn);
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

// ---- host side: where this engine runs -------------------------------------------

// The times (us) of a whole layer with H x I experts (up and gate in one launch,
// K = H; down, K = I) on these tiles and on the 128-row ones, fitted to
// graph-timed layers of 20912 random sizes (both types; E = 8..256, H = 512..4096, I =
// 256..3072, up to 64 rows an expert, even to skewed routings): 5..95% of them
// within 0.84..1.16 and 0.80..1.15 of the fit.  rows per expert are taken as
// Poisson: E (1 - e^-l) experts with rows, l = G / E.
//   * here: a launch cannot be shorter than its waves' walk (by K), and a workgroup
//     costs its part of the decode (by K) and a fixed start and end; 64 columns x 32
//     rows a workgroup, past ~20 rows an expert some experts take a second tile;
//   * the 128-row tiles: K stages of constant length, dearer once the tiles (two
//     experts' rows share one, up to 64 each) pass one a CU.
struct MoeUs {
    double kw, tile;
};
MoeUs moe_layer_us(int G, int E, int H, int I) {
    const double l = (double)G / E, with = E * (1.0 - std::exp(-l)), h = H / 1024.0, i = I / 1024.0;
    const double t = l > 20.0 ? std::max(with, E * (l / 32.0 + 0.45)) : with, p = std::max(with / 2.0, 1.0);
    auto up_to = [](int n, int b) { return (double)((n + b - 1) / b); };
    const double wu = t * up_to(I, 64) / 256.0, wd = t * up_to(H, 64) / 256.0;
    const int bu = moe_bn(I, 256), bd = moe_bn(H, 512);
    const double ru = p * up_to(I, bu) / 256.0, rd = p * up_to(H, bd) / 256.0;
    MoeUs us;
    us.kw = 18.5 + std::hypot(2.5 * h, (3.25 * h + 2.35) * wu) + std::hypot(1.2 * i, (0.65 * i + 1.2) * wd);
    us.tile = 20.7 + (bu == 256 ? 17.8 : 9.9) * h * (1.0 + std::min(ru, 1.0) + 2.5 * std::max(ru - 1.0, 0.0)) +
              (bd == 512 ? 18.6 : bd == 256 ? 10.0 : 6.4) * i * (1.0 - 0.15 * std::min(rd, 1.0) + 1.6 * std::max(rd - 1.0, 0.0));
    return us;
}

}  // namespace

// Whether G rows over E experts of K x N weights run here.  A layer's products (K x
// N and N x K) and the single grouped GEMM ask alike, so their bits agree: a
// product does not know which of the two sizes is the layer's H: the layer with the
// larger one as H, the usual one, counts twice, the other once.  Ahead by more than
// the fits' spread: of the 20912 layers 78% run here and 13 lose more than 3%, two
// of them more than 10% (a bound on the weights decoded, with a row tile an expert,
// lost more than 3% in 1558, up to 2.5x).  Measured layers (bf16,
// top-8 unless said, us; 128-row tiles / here): E = 128 H = 2048 I = 768, T = 1 77 /
// 30, T = 8 78 / 50, T = 16 80 / 67, not taken T = 32 83 / 85, T = 64 85 / 92; E = 64
// I = 1408, T = 16 92 / 71, T = 64 93 / 81, T = 128 97 / 84, not taken T = 256 115 /
// 111, T = 512 171 / 171; E = 16 top-4, H = 1024 I = 512, T = 40 50 / 24, H = 3072 I =
// 1536, T = 128 122 / 61.  64-row tiles were faster than these 32-row ones by more
// than 3% in 9 of the layers taken (E = 64 I = 1408, T = 128 139; E = 16 H = 3072, T
// = 128 69).
static bool moe_kw_takes(int G, int E, int N, int K) {
    if ((long)G > 64L * E) return false;
    const int large = std::max(N, K), small = std::min(N, K);
    const MoeUs a = moe_layer_us(G, E, large, small), b = moe_layer_us(G, E, small, large);
    return 2.0 * a.kw + b.kw < 0.89 * (2.0 * a.tile + b.tile);
}

// (for ternocl_kw_tile_of: the tile of one of the layer's products)
bool moe_kw_tile_of(int G, int E, int N, int K, ternocl_kw_tile &t) {
    if (!moe_kw_takes(G, E, N, K)) return false;
    t = {32, 64, 4, 1, 0};
    return true;
}

// The grouped GEMM (B2 non-null: up and gate in one launch) where the rule above
// takes it and the operands are 16-byte aligned; returns whether it ran.
bool moe_gemm_kw_run(int dtype, const int *meta, const void *A, const int *perm, int topk, const uint32_t *B, const void *S,
                     const uint32_t *B2, const void *S2, void *C, const void *Other, int E, int G, int N, int K, int postop,
                     int out_f32, hipStream_t st, ternocl_status &s) {
    if (!moe_kw_takes(G, E, N, K) || !aligned16(A) || !aligned16(B) || !aligned16(S) || !aligned16(B2) || !aligned16(S2) ||
        !aligned16(C) || !aligned16(Other))
        return false;
    auto go = [&](auto bf, auto dual) {
        constexpr bool BF = decltype(bf)::value, D = decltype(dual)::value;
        moe_kw_launch<KwCfg<1, D ? 4 : 2, 1, 4, 2>, BF, D>(meta, A, perm, topk, B, S, B2, S2, C, Other, E, G, N, K, postop,
                                                           out_f32, st);
    };
    if (dtype == TERNOCL_BF16) B2 ? go(std::true_type{}, std::true_type{}) : go(std::true_type{}, std::false_type{});
    else B2 ? go(std::false_type{}, std::true_type{}) : go(std::false_type{}, std::false_type{});
    s = check_launch();
    return true;
}

}  // namespace tcl
