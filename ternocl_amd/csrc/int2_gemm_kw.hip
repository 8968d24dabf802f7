// int2_gemm_kw.hip -- GEMM of tens to hundreds of rows (batched decode, short
// prompts) on packed 2-bit ternary weights for gfx950: the C of
// int2_fp16_upcvt_gemm / int2_fp16_upcvt_gemm_mt (int2_fp16_upcvt/int2_fp16_upcvt.cl:
// 196-198, :341-343) with K split over the waves of a workgroup.
//
// Why: at these M a 128-row tile engine has few tiles (N = 4096: 32 at any
// M <= 128), and each walks all of K in 64-row stages behind one barrier and
// one stage of prefetch, ~0.6 us a stage: 40 us at K = 4096 whatever M is.  A
// workgroup here owns a narrow strip (32 WM MB rows x 32 CB columns) and its
// WK waves each take a contiguous part of K in 64-row units, on their own: a wave
// loads a unit's activation rows and packed words, multiplies, and meets no barrier
// until all of K is done; the waves' fp32 sums then meet in LDS and are added in
// wave order (the same bits on every run).  Each weight word is decoded once
// per row tile.
//   * Activations go global -> registers -> a wave-private LDS buffer (coalesced
//     16-byte loads; the LDS turns rows into MFMA fragments), two buffers in
//     turn: unit u + 1 is stored in the middle of unit u, so no MFMA waits for a
//     store of its own unit.  16-byte chunk j of row r lies at position j ^ (r %
//     8): stores and fragment reads of 8 lanes each cover the banks once.
//   * B fragments hold adjacent rows (2d, 2d + 1) of a word in dword d, so an A
//     fragment is 8 consecutive activations as they lie in memory (no
//     interleaving): the word and the word >> 2 spread one byte into (b, b, b',
//     b'), then a mask-and-set and a v_perm through the byte tables {0, s, 0,
//     -s} (both DT types: exact +-s, three operations per pair).  Code 2 reads
//     as 0.  CB adjacent columns per lane: one 4 CB-byte load per word row.
//   * What bounds it: a wave's own instructions in a row, with one wave a SIMD (the
//     64- and 128-column tiles) to cover them.  Counters: at M = 24, K = 4096, N =
//     24576 (32 x 128) a wave issues VALU 51% of its time (the decode), waits 25%, the
//     MFMAs are busy 24% and the LDS of a CU 15%; at M = 128, K = 4096, N = 14336 (64 x
//     128) 41, 24, 34 and 21%; at M = 24, K = N = 4096 (32 x 32, two waves a SIMD) it
//     waits 55%, for the first loads and the sums.  Not the weight stream: two or
//     four units of weights ahead measure the same.  The activations' way through L1
//     and LDS adds to all of it: a copy without their loads and stores takes half
//     the time at M = 64, K = 5120, N = 34816 (50 -> 22-33 us over the tiles).
//     Storing unit u itself at its start, on the critical path: 24 -> 21.7 us
//     with the two buffers (M = 128, K = 4096, N = 14336).
// Measured against the engines these calls took before (graph-timed, bf16,
// rotated weights, us; M = 9..16 the MFMA GEMV, above the 128-row tiles):
//   M = 16, K = 4096 N = 4096 16.6 -> 8.2, N = 14336 21.0 -> 10.6, K = 14336 N =
//   4096 54.0 -> 18.2; M = 32 39.8 -> 8.5, 40.5 -> 10.9, 130.6 -> 13.3; M = 128
//   40.2 -> 11.8, 40.6 -> 21.7, 130.9 -> 25.6; M = 256 K = 4096 N = 4096 40.5 ->
//   15.8; M = 512 43.5 -> 24.5.
#include "gemm_kw.hpp"

#include <algorithm>

namespace tcl {
// (int2_gemm_mfma.hip)
bool gemm_half_tile(int M, int N);
bool gemm_tile_is_square(int M, int N);
int gemm_splits(int M, int N, int K);
namespace {

// ksn > 1: workgroup (tile, slice sl) runs the units of its K slice (kw_finish).
template <class Cfg, bool BF16>
__global__ void __launch_bounds__(Cfg::THREADS)
k_int2_gemm_kw(const uint16_t *__restrict__ A, const uint32_t *__restrict__ B, const uint16_t *__restrict__ S,
               void *__restrict__ C, const uint16_t *__restrict__ Other, const void *__restrict__ Bias, int M, int N,
               int K, int postop, int out_f32, int ksn, float *part, uint64_t *cnt) {
    constexpr int MB = Cfg::MB, CB = Cfg::CB, WK = Cfg::WK;
    extern __shared__ __attribute__((aligned(16))) uint8_t kw_lds[];
    const int mt = (M + Cfg::BM - 1) / Cfg::BM, nt = (N + Cfg::BN - 1) / Cfg::BN;
    int tms, tn;
    if (!xcd_tile_ashare(blockIdx.x, mt * ksn, nt, tms, tn)) return;  // whole workgroup: padding
    const int tm = __builtin_amdgcn_readfirstlane(tms / ksn), sl = __builtin_amdgcn_readfirstlane(tms - tm * ksn);
    const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / Cfg::WM, wm = wave % Cfg::WM;
    const int c = lane & 31, q = lane >> 5;
    const int units = K / 64;
    // this wave's units: a contiguous part of the slice's
    const int s0 = (int)((long)units * sl / ksn), s1 = (int)((long)units * (sl + 1) / ksn);
    const int u0 = s0 + (s1 - s0) * kw / WK, u1 = s0 + (s1 - s0) * (kw + 1) / WK;
    const int mrows = min(Cfg::BM, M - m0);

    // A: chunk lane + 64 i of the unit -> row i * 8 + lane / 8, 16-byte chunk lane % 8
    // (rows past the tile's re-read its last row: their outputs are not stored)
    uint32_t va[4 * MB];
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i)
        va[i] = (uint32_t)min(32 * MB * wm + (lane >> 3) + 8 * i, mrows - 1) * (uint32_t)K + 8u * (lane & 7);
    KwInt2<CB, Cfg::PF> bs(B, S, N, units, (uint32_t)min(n0 + CB * c, N - CB), q);
    f32x16_t acc[MB][CB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[mb][cb] = f32x16_t{};
    kw_walk<Cfg, BF16>(kw_lds + wave * (MB * 8192), A + (size_t)m0 * K, va, u0, u1, units, bs, acc);
    kw_finish<Cfg, BF16>(acc, kw_lds, C, Other, Bias, M, N, m0, mrows, n0, postop, out_f32, ksn, sl, part,
                         ksn > 1 ? cnt + 2 * ((size_t)tm * nt + tn) : nullptr);
}

template <class Cfg, bool BF16>
hipError_t kw_launch(const void *A, const uint32_t *B, const void *S, void *C, const void *Other, const void *Bias, int M,
                     int N, int K, int postop, int out_f32, int ksn, float *part, uint64_t *cnt, hipStream_t st) {
    const int mt = (M + Cfg::BM - 1) / Cfg::BM, nt = (N + Cfg::BN - 1) / Cfg::BN;
    hipLaunchKernelGGL((k_int2_gemm_kw<Cfg, BF16>), dim3(xcd_ashare_grid(mt * ksn, nt)), dim3(Cfg::THREADS),
                       Cfg::LDS_BYTES, st, (const uint16_t *)A, B, (const uint16_t *)S, C, (const uint16_t *)Other, Bias,
                       M, N, K, postop, out_f32, ksn, part, cnt);
    return hipGetLastError();
}

// ---- host side: tile choice ----------------------------------------------------

// The compiled tiles, with what a launch of one round (<= 256 workgroups) of
// each costs: us = base + slope * (rows of K per workgroup) / 1024, fitted to
// graph-timed runs (bf16, rotated weights) over M = 16..2048, N = 1024..34816,
// K = 1024..14336.  A wider tile loads the activations and decodes the words
// fewer times; a narrower one fills the chip at small M N.
struct KwTile {
    int bm, bn;
    double base, slope;
};
constexpr KwTile kKwTiles[] = {{32, 32, 4.0, 1.3}, {32, 64, 5.2, 1.75}, {32, 128, 5.2, 2.5},
                               {64, 64, 4.3, 2.8}, {64, 128, 7.2, 4.4}, {128, 128, 8.8, 8.1}};
constexpr int kKwTileCount = sizeof(kKwTiles) / sizeof(kKwTiles[0]);

struct KwPlan {
    int tile, ks;  // ks: K slices (> 1 needs the workspace)
    double us;
};

// The cheapest tile and slice count by that model.  Further rounds cost their
// K walk and half a base each (M = 300, K = 4096, N = 14336 on 64 x 64 tiles, 5
// rounds: 64.9 modelled, 61.3 measured); a K split costs 1.2 us and its slice
// sums' round trip at 4 TB/s (M = 32, K = 14336, N = 4096 on 32 x 64 tiles, 4
// slices: 13.6 modelled, 13.3 measured against 23.6 unsplit).
KwPlan kw_plan(int M, int N, int K, bool split) {
    KwPlan best = {-1, 1, 1e30};
    for (int i = 0; i < kKwTileCount; ++i) {
        const KwTile &t = kKwTiles[i];
        if (t.bm > 32 && t.bm >= 2 * M) continue;  // half the tile's rows idle: a lower one does it
        const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
        for (int ks = 1; ks <= 8; ++ks) {
            if (ks > 1 && (!split || K / ks < 512 || tiles * ks > 1024 || tiles * 16 > (long)kWsHeader)) break;
            const double rounds = (double)((tiles * ks + 255) / 256);
            double us = t.base * (0.5 + 0.5 * rounds) + t.slope * rounds * K / (1024.0 * ks);
            if (ks > 1) us += 1.2 + 8e-6 * ks * M * N / 4.0;
            if (us < best.us - 1e-9) best = {i, ks, us};
        }
    }
    return best;
}

// The 128-row tile engine's time (int2_gemm_mfma.hip) by the same kind of fit, over its
// plan: 128 x 128 tiles (M = 32 / 512 / 1024, K = N = 4096: 39.8 / 43.5 / 48.9
// us), 128 x 256 tiles (M = 1236, K = 4096, N = 6320: 68.2; M = 164, K = 2816, N = 32528:
// 48.9), 128 x 512 tiles (N = 14336: 103; fewer than 192 of them, M = 1491, K = 9984, N =
// 5456: 220) and their K split (M = 212, K = 9728, N = 13760: 81.7; M = 774, K = 10752, N =
// 3600: 84.0).  Both fits are good to some 5%, so this engine is taken where it is
// ahead by more (kKwMargin): of 7780 random calls with 5e9 multiply-adds or more (M to
// 2048, K to 14336, N to 34816, both types, with and without the workspace, engines
// timed in random order) 2 lose more than 3%, 45 with 24.5 k / ks + 2e-6 ks M N for the
// split and 128 x 256 tiles dearer in bf16, which they are not: M = 164 took 53.2 us
// here, M = 212 87.7, M = 774 91.2.
constexpr double kKwMargin = 0.95;
double kw_other_us(int M, int N, int K, bool split) {
    auto tiles = [&](int BM, int BN) { return (double)((long)((M + BM - 1) / BM) * ((N + BN - 1) / BN)); };
    const double k = K / 1024.0, wide = tiles(128, 512), half = tiles(128, 256), square = tiles(128, 128);
    if (wide >= 192) return 5.0 + 24.5 * k * (wide <= 256 ? 1.0 : wide / 256.0);
    const bool h = gemm_half_tile(M, N);
    const int ks = split && !(h && half >= 192) ? gemm_splits(M, N, K) : 1;
    if (ks > 1) return 8.0 + 22.0 * k / ks * (wide * ks > 256 ? 2.0 : 1.0) + 1.4e-6 * ks * M * N;
    if (h) return 7.1 + (9.9 + 5.6 * half / 256.0) * k;
    if (square <= 512) return 3.2 + (9.3 + 1.8 * std::min(square, 256.0) / 256.0) * k * (square > 256 ? 1.5 : 1.0);
    return 5.0 + 22.0 * k;
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// The times the two models give a call without a K split (the M-tiled BITCOS
// GEMM's choice, bitcos_kw.hip); wk: the waves over K of this engine's tile; square:
// whether the other runs 128 x 128 tiles.
void int2_gemm_kw_model(int M, int N, int K, double &kw_us, double &other_us, int &wk, bool &square) {
    const KwPlan p = kw_plan(M, N, K, false);
    kw_us = p.us;
    other_us = kw_other_us(M, N, K, false);
    wk = p.tile <= 1 ? 8 : 4;
    square = gemm_tile_is_square(M, N);
}

// Whether plan p is the automatic engine of a call of M > 8 rows: always up to 16
// rows (the MFMA GEMV is 2-3x its time there from K = 4096 on; with K <= 512 it is 2-20%
// ahead, 0.2-0.9 us, but its sums are less exact), above where its model is ahead of
// the 128-row tile engine's.  split: whether K slices may use a workspace.
static bool kw_wins(const KwPlan &p, int M, int N, int K, bool split) {
    return M <= 16 || (M <= 2048 && p.us < kKwMargin * kw_other_us(M, N, K, split));
}

// Workspace of the automatic plan's K split (0: none; none up to 16 rows).
size_t int2_gemm_kw_ws_need(int M, int N, int K) {
    if (M <= 16 || M > 2048) return 0;
    const KwPlan p = kw_plan(M, N, K, true);
    if (p.ks == 1 || !kw_wins(p, M, N, K, true)) return 0;
    return kWsHeader + (size_t)p.ks * M * N * 4;
}

// The tile and K slices of an automatic call on aligned operands with ws_bytes of
// workspace (0: none), false where another engine runs it: the choice of
// int2_gemm_kw_run, for ternocl_kw_tile_of.
static bool kw_choose(int M, int N, int K, size_t ws_bytes, bool force, KwPlan &p) {
    bool split = ws_bytes > kWsHeader && M > 16;
    p = kw_plan(M, N, K, split);
    if (p.ks > 1 && ws_bytes < kWsHeader + (size_t)p.ks * M * N * 4) {
        p = kw_plan(M, N, K, false);
        split = false;
    }
    return force || kw_wins(p, M, N, K, split);
}

bool int2_gemm_kw_tile(int M, int N, int K, size_t ws_bytes, bool force, ternocl_kw_tile &t) {
    KwPlan p;
    if (M <= 8 || M > 2048 || !kw_choose(M, N, K, ws_bytes, force, p)) return false;
    t = {kKwTiles[p.tile].bm, kKwTiles[p.tile].bn, p.tile <= 1 ? 8 : 4, p.ks, 0};
    return true;
}

// Runs the call here if this is its automatic engine (force: whichever the
// models prefer) and returns whether it did; the status in s.  A K split needs
// its slice sums in ws; with less the unsplit plan is weighed.  The vector
// loads and stores need 16-byte aligned operands.
bool int2_gemm_kw_run(int dtype, const void *A, const uint32_t *B, const void *S, void *C, const void *Other,
                      const void *Bias, int M, int N, int K, int postop, int out_f32, hipStream_t st, void *ws,
                      size_t ws_bytes, bool force, ternocl_status &s) {
    const bool bf = dtype == TERNOCL_BF16;
    if (M <= 8 || M > 2048 || !aligned16(A) || !aligned16(B) || !aligned16(S) || !aligned16(C) || !aligned16(Other) ||
        !aligned16(Bias))
        return false;
    KwPlan p;
    if (!kw_choose(M, N, K, ws && aligned16(ws) ? ws_bytes : 0, force, p)) return false;
    uint64_t *cnt = p.ks > 1 ? (uint64_t *)ws : nullptr;
    float *part = p.ks > 1 ? (float *)((uint8_t *)ws + kWsHeader) : nullptr;
    auto go = [&](auto cfg) {
        typedef decltype(cfg) Cfg;
        return bf ? kw_launch<Cfg, true>(A, B, S, C, Other, Bias, M, N, K, postop, out_f32, p.ks, part, cnt, st)
                  : kw_launch<Cfg, false>(A, B, S, C, Other, Bias, M, N, K, postop, out_f32, p.ks, part, cnt, st);
    };
    hipError_t e;
    switch (p.tile) {
    case 0: e = go(KwCfg<1, 1, 1, 8, 4>{}); break;
    case 1: e = go(KwCfg<1, 2, 1, 8, 2>{}); break;
    case 2: e = go(KwCfg<1, 4, 1, 4, 2>{}); break;
    case 3: e = go(KwCfg<2, 2, 1, 4, 4>{}); break;
    case 4: e = go(KwCfg<2, 4, 1, 4, 2>{}); break;
    default: e = go(KwCfg<2, 4, 2, 4, 2>{}); break;
    }
    s = launch_status(e);
    return true;
}

}  // namespace tcl
