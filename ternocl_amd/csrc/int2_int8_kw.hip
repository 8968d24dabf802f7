// int2_int8_kw.hip -- the s8 x s2 GEMM of a few to hundreds of rows on gfx950:
// the C of int2_int8_gemv / int2_int8_gemm_mt (int2_via_int2_x_int8_dpas/
// int2_int8_dpas.cl:213-215, :316-318) in both quantization modes, with K split
// over the waves of a workgroup as in int2_gemm_kw.hip (gemm_kw.hpp).
//
// A unit of a wave's K walk is one 128-row scale group: 32 MB rows of int8
// (128 bytes each, the DT walk's chunk layout), 8 packed words and one scale a
// column, and SA of the wave's rows.  The group's int32 dots (four chained
// v_mfma_i32_32x32x32_i8) are exact; acc += float(dot) * (SB * (1 / SA)) as the
// tile engines fold them (int2_int8.hip), with the groups of a column added in
// another order: a wave's groups, then the waves.  QA (the reference's QMODE 1):
// DT rows quantized while they are stored into LDS, the same int8 values and so
// the same bits as the upfront mode.
//
// The tile engines take ~35 us at K = 4096 and ~115 us at K = 14336 for any M in
// 5..256 where their tiles are few (each walks all of K group by group behind a
// barrier); the times here are at kI8Tiles.  What bounds it is the VALU work of a
// group, 3 instructions an output for the fold and the decode, beside the LDS
// and L1 traffic of the rows (int2_gemm_kw.hip).
#include "gemm_kw.hpp"
#include "int8_frag.hpp"

#include <algorithm>
#include <cmath>

namespace tcl {
// (int2_gemm_mfma.hip)
bool gemm_half_tile(int M, int N);
int gemm_splits(int M, int N, int K);
namespace {

typedef int i32x16_t __attribute__((ext_vector_type(16)));

template <class Cfg, bool BF16, bool QA>
__global__ void __launch_bounds__(Cfg::THREADS)
k_int2_int8_kw(const void *__restrict__ Asrc, const uint16_t *__restrict__ SA, const uint32_t *__restrict__ B,
               const uint16_t *__restrict__ SB, void *__restrict__ C, const uint16_t *__restrict__ Other,
               const void *__restrict__ Bias, int M, int N, int K, int postop, int out_f32, int ksn, float *part,
               uint64_t *cnt) {
    constexpr int MB = Cfg::MB, CB = Cfg::CB, WK = Cfg::WK, PF = Cfg::PF;
    static_assert(MB <= 2, "a lane per row for 1 / SA");
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
    const int groups = K / kGS, lda = ldsa_of(M);
    // this wave's groups: a contiguous part of the slice's
    const int s0 = (int)((long)groups * sl / ksn), s1 = (int)((long)groups * (sl + 1) / ksn);
    const int g0 = s0 + (s1 - s0) * kw / WK, g1 = s0 + (s1 - s0) * (kw + 1) / WK;
    const int mrows = min(Cfg::BM, M - m0);

    // A: chunk lane + 64 i of the group -> row i * 8 + lane / 8, 16 k rows lane % 8
    // (rows past the tile's re-read its last row: their outputs are not stored)
    constexpr int ES = QA ? 2 : 1;  // bytes per element in memory
    uint32_t row[4 * MB];
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i) row[i] = (uint32_t)min(32 * MB * wm + (lane >> 3) + 8 * i, mrows - 1);
    const uint8_t *Ab = (const uint8_t *)Asrc + (size_t)m0 * K * ES;
    const uint16_t *SAb = SA + m0;
    const uint32_t srow = (uint32_t)min(32 * MB * wm + (lane & (32 * MB - 1)), mrows - 1);
    u32x4_t av[4 * MB][ES];
    uint32_t sq[QA ? 4 * MB : 1], sa_raw = 0;
    auto a_load = [&](int g) __attribute__((always_inline)) {  // (past the last: re-read, never used)
        const int gc = min(g, groups - 1);
        const uint8_t *p = Ab + (size_t)gc * kGS * ES;
        const uint16_t *sp = SAb + (size_t)gc * lda;
#pragma unroll
        for (int i = 0; i < 4 * MB; ++i) {
#pragma unroll
            for (int e = 0; e < ES; ++e)
                av[i][e] = *(const u32x4_t *)(p + (row[i] * (uint32_t)K + 16u * (lane & 7)) * ES + 16 * e);
            if constexpr (QA) sq[i] = sp[row[i]];
        }
        sa_raw = sp[srow];
    };
    uint8_t *abuf = kw_lds + wave * (MB * 8192);
    float *inv = (float *)(kw_lds + Cfg::A_BYTES) + wave * (64 * MB);  // two groups' 1 / SA of the wave's rows
    uint8_t *aw = abuf + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    auto a_store = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4 * MB; ++i) {
            uint32_t o[4];
            if constexpr (QA) {
                const float sa = dt2f<BF16>(sq[i]);
                uint32_t h[8], qb[16];
                __builtin_memcpy(h, &av[i][0], 32);
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    qb[2 * j] = q8_bits<BF16>(h[j] & 0xffffu, sa);
                    qb[2 * j + 1] = q8_bits<BF16>(h[j] >> 16, sa);
                }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    o[j] = __builtin_amdgcn_perm(qb[4 + j], qb[j], 0x0c0c0400u) |
                           __builtin_amdgcn_perm(qb[12 + j], qb[8 + j], 0x04000c0cu);
            } else {
                uint32_t d[4];
                __builtin_memcpy(d, &av[i][0], 16);
                transpose4x4(d, o);
            }
            *(u32x4_t *)(aw + p * (MB * 4096) + 1024 * i) = u32x4_t{o[0], o[1], o[2], o[3]};
        }
        const float sa = dt2f<BF16>(sa_raw);
        inv[32 * MB * p + (lane & (32 * MB - 1))] = sa != 0.0f ? 1.0f / sa : 0.0f;
    };
    uint32_t ar[4];  // k-chunk kc of lane (c, q): row c's chunk 2 kc + q
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) ar[kc] = (uint32_t)(c * 128 + (((2 * kc + q) ^ (c & 7)) << 4));
    i32x4_t af[4];
    auto a_frags = [&](int p, int mb) __attribute__((always_inline)) {
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) af[kc] = *(const i32x4_t *)(abuf + p * (MB * 4096) + ar[kc] + 4096 * mb);
    };

    // B: lane (c, q) holds words 8 g + 2 kc + q of its CB columns (past N: the last ones)
    typedef typename KwVec<CB>::W W;
    typedef typename KwVec<CB>::S SV;
    const uint32_t col = (uint32_t)min(n0 + CB * c, N - CB);
    W bw[PF][4];
    SV sr[PF];
    auto b_load = [&](int g, int s) __attribute__((always_inline)) {
        const int gc = min(g, groups - 1);
        const uint32_t *p = B + (size_t)(8 * gc) * N;
#pragma unroll
        for (int kc = 0; kc < 4; ++kc)
            bw[s][kc] = __builtin_nontemporal_load((const W *)(p + (2 * kc + q) * (uint32_t)N + col));
        sr[s] = *(const SV *)(SB + (size_t)gc * N + col);
    };

    f32x16_t acc[MB][CB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[mb][cb] = f32x16_t{};

    // Group g from slot s and LDS buffer p = s % 2: the next group's rows are
    // stored in the middle, its first fragments read at the end.
    auto unit = [&](int g, int s, bool more) __attribute__((always_inline)) {
        const int p = s & 1;
        i32x4_t bf[CB][4];
        float sb[CB];
        uint32_t sw[(CB + 1) / 2] = {};
        __builtin_memcpy(sw, &sr[s], sizeof(SV));
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) {
            uint32_t t[CB];
            __builtin_memcpy(t, &bw[s][kc], sizeof(W));
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) bf[cb][kc] = decode_s2(t[cb]);
        }
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) sb[cb] = dt2f<BF16>((sw[cb >> 1] >> (16 * (cb & 1))) & 0xffffu);
        if (more) b_load(g + PF, s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            f32x4_t iv[4];  // 1 / SA of rows 32 mb + 8 j + 4 q + (0..3)
#pragma unroll
            for (int j = 0; j < 4; ++j) iv[j] = *(const f32x4_t *)(inv + 32 * MB * p + 32 * mb + 8 * j + 4 * q);
            i32x16_t dot[CB];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                dot[cb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[0], bf[cb][0], i32x16_t{}, 0, 0, 0);
#pragma unroll
                for (int kc = 1; kc < 4; ++kc)
                    dot[cb] = __builtin_amdgcn_mfma_i32_32x32x32_i8(af[kc], bf[cb][kc], dot[cb], 0, 0, 0);
            }
            if (mb == 0) {
                __builtin_amdgcn_sched_barrier(0);
                a_store(p ^ 1);
                a_load(g + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
            if (mb + 1 < MB) a_frags(p, mb + 1);
            else a_frags(p ^ 1, 0);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[mb][cb][v] += (float)dot[cb][v] * (sb[cb] * iv[v >> 2][v & 3]);
        }
    };
    if (g0 < g1) {
        a_load(g0);
#pragma unroll
        for (int s = 0; s < PF; ++s) b_load(g0 + s, s);
        __builtin_amdgcn_sched_barrier(0);
        a_store(0);
        a_load(g0 + 1);
        __builtin_amdgcn_sched_barrier(0);
        a_frags(0, 0);
        int g = g0;
        for (; g + PF - 1 < g1; g += PF)
#pragma unroll
            for (int s = 0; s < PF; ++s) unit(g + s, s, true);
#pragma unroll
        for (int s = 0; s < PF - 1; ++s) {
            if (g + s >= g1) break;
            unit(g + s, s, false);
        }
    }
    kw_finish<Cfg, BF16>(acc, kw_lds, C, Other, Bias, M, N, m0, mrows, n0, postop, out_f32, ksn, sl, part,
                         ksn > 1 ? cnt + 2 * ((size_t)tm * nt + tn) : nullptr);
}

template <class Cfg> constexpr int i8kw_lds() {
    const int walk = Cfg::A_BYTES + Cfg::WM * Cfg::WK * 256 * Cfg::MB;
    return walk > Cfg::LDS_BYTES ? walk : Cfg::LDS_BYTES;
}

template <class Cfg, bool BF16, bool QA>
hipError_t i8kw_launch(const void *A, const void *SA, const uint32_t *B, const void *SB, void *C, const void *Other,
                       const void *Bias, int M, int N, int K, int postop, int out_f32, int ksn, float *part, uint64_t *cnt,
                       hipStream_t st) {
    const int mt = (M + Cfg::BM - 1) / Cfg::BM, nt = (N + Cfg::BN - 1) / Cfg::BN;
    hipLaunchKernelGGL((k_int2_int8_kw<Cfg, BF16, QA>), dim3(xcd_ashare_grid(mt * ksn, nt)), dim3(Cfg::THREADS),
                       i8kw_lds<Cfg>(), st, A, (const uint16_t *)SA, B, (const uint16_t *)SB, C, (const uint16_t *)Other,
                       Bias, M, N, K, postop, out_f32, ksn, part, cnt);
    return hipGetLastError();
}

// ---- host side: tile choice ----------------------------------------------------

// The compiled tiles and what their launches cost (us, K in 1024 rows per
// workgroup), fitted to graph-timed runs (bf16, upfront mode) over M = 4..1024,
// N = 1024..34816, K = 1024..14336: 0: 32 x 32, eight waves over K; 1: 32 x 64,
// eight waves; 2: 32 x 64, four waves, two workgroups a CU; 3: 64 x 64, two
// times four waves.  Measured, the tile engines' times first (without quant_a):
// K = N = 4096, M = 8 / 32 / 128 / 256 34.9 / 35.4 / 36.2 / 36.7 -> 7.3 / 7.5 /
// 11.4 / 15.5; K = 4096 N = 14336, M = 8 / 32 / 64 36.5 / 36.9 / 37.5 -> 9.9 /
// 10.4 / 14.5; K = 14336 N = 4096, M = 8 / 48 / 256 114 / 115 / 116 -> 11.4 /
// 15.4 / 39.5; K = 5120 N = 34816, M = 32 60.9 -> 27.3.
struct I8Tile {
    int bm, bn;
};
constexpr I8Tile kI8Tiles[] = {{32, 32}, {32, 64}, {32, 64}, {64, 64}};

double i8kw_us(int tile, double wgs, double k) {
    const double rounds = std::ceil(wgs / 256.0);
    switch (tile) {
    case 0: return 4.0 * (0.5 + 0.5 * rounds) + 1.0 * rounds * k;
    case 1: return 4.8 * (0.5 + 0.5 * rounds) + 1.55 * rounds * k;
    case 2: return wgs <= 256 ? 5.2 + 1.55 * k : wgs <= 512 ? 6.2 + 2.6 * k : 8.0 + 3.05 * k * wgs / 512.0;
    default: return 5.5 * (0.5 + 0.5 * rounds) + 2.45 * rounds * k;
    }
}

struct I8Plan {
    int tile, ks;  // ks: K slices (> 1 needs the workspace)
    double us;
};

// The cheapest tile and slice count by that model (a K split: 1.2 us and its
// slice sums' round trip at 4 TB/s; M = 48, K = 14336, N = 4096 on 32 x 64 tiles:
// 21.0 unsplit, 15.4 on 2 slices).
I8Plan i8kw_plan(int M, int N, int K, bool split) {
    I8Plan best = {-1, 1, 1e30};
    for (int i = 0; i < 4; ++i) {
        const I8Tile &t = kI8Tiles[i];
        if (t.bm > 32 && t.bm >= 2 * M) continue;  // half the tile's rows idle
        const long tiles = (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
        for (int ks = 1; ks <= 8; ++ks) {
            if (ks > 1 && (!split || K / ks < 512 || tiles * ks > 1024 || tiles * 16 > (long)kWsHeader)) break;
            double us = i8kw_us(i, (double)tiles * ks, K / (1024.0 * ks));
            if (ks > 1) us += 1.2 + 8e-6 * ks * M * N / 4.0;
            if (us < best.us - 1e-9) best = {i, ks, us};
        }
    }
    return best;
}

// The tile engines' time (int2_int8.hip, upfront mode) by the same kind of fit: 128
// x 512 tiles (M = 1024, K = 4096, N = 14336: 85 us), 128 x 256 (M = 512: 60; M = 128,
// K = 5120, N = 34816: 62), the K split, and 128 x 128 (K = 4096: 35-43).
double i8_other_us(int M, int N, int K, bool split) {
    auto tiles = [&](int BM, int BN) { return (double)((long)((M + BM - 1) / BM) * ((N + BN - 1) / BN)); };
    const double k = K / 1024.0, wide = tiles(128, 512), half = tiles(128, 256), square = tiles(128, 128);
    if (wide >= 192) return 4.0 + 20.0 * k * (wide <= 256 ? 1.0 : wide / 256.0);
    if (gemm_half_tile(M, N)) return 4.0 + (8.5 + 6.0 * half / 256.0) * k;
    const int ks = split ? gemm_splits(M, N, K) : 1;
    if (ks > 1) return 4.0 + 20.0 * k / ks + 7e-6 * ks * M * N / 4.0;
    return 3.2 + (7.85 + 2.2 * std::min(square, 256.0) / 256.0) * k * std::max(1.0, square / 256.0);
}

// Both fits are good to some 5%: this engine where it is ahead by more.
constexpr double kI8Margin = 0.95;

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

static bool i8kw_wins(const I8Plan &p, int M, int N, int K, bool split) {
    return p.us < kI8Margin * i8_other_us(M, N, K, split);
}

// Workspace of the automatic plan's K split (0: none).
size_t int2_int8_kw_ws_need(int M, int N, int K) {
    if (M <= 4 || M > 2048) return 0;
    const I8Plan p = i8kw_plan(M, N, K, true);
    return p.ks > 1 && i8kw_wins(p, M, N, K, true) ? kWsHeader + (size_t)p.ks * M * N * 4 : 0;
}

// The tile and K slices of a call on aligned operands with ws_bytes of workspace
// (0: none), false where the tile engines run it: the choice of int2_int8_kw_run,
// for ternocl_kw_tile_of.
static bool i8kw_choose(int M, int N, int K, size_t ws_bytes, I8Plan &p) {
    bool split = ws_bytes > kWsHeader;
    p = i8kw_plan(M, N, K, split);
    if (p.ks > 1 && ws_bytes < kWsHeader + (size_t)p.ks * M * N * 4) {
        p = i8kw_plan(M, N, K, false);
        split = false;
    }
    return i8kw_wins(p, M, N, K, split);
}

bool int2_int8_kw_tile(int M, int N, int K, size_t ws_bytes, ternocl_kw_tile &t) {
    I8Plan p;
    if (M <= 4 || M > 2048 || !i8kw_choose(M, N, K, ws_bytes, p)) return false;
    t = {kI8Tiles[p.tile].bm, kI8Tiles[p.tile].bn, p.tile <= 1 ? 8 : 4, p.ks, 0};
    return true;
}

// Runs the call here if the models prefer this engine and returns whether it
// did; the error in e.  Aq non-null: upfront mode, else A's DT rows; the choice
// is the same in both, whose bits agree.  A K split needs its slice sums in ws;
// with less the unsplit plan is weighed.  The vector loads and stores need
// 16-byte aligned operands.
bool int2_int8_kw_run(int dtype, const void *A, const int8_t *Aq, const void *SA, const uint32_t *B, const void *SB,
                      void *C, const void *Other, const void *Bias, int M, int N, int K, int postop, int out_f32,
                      hipStream_t st, void *ws, size_t ws_bytes, hipError_t &e) {
    if (M > 2048 || !aligned16(Aq ? (const void *)Aq : A) || !aligned16(B) || !aligned16(SB) || !aligned16(C) ||
        !aligned16(Other) || !aligned16(Bias))
        return false;
    I8Plan p;
    if (!i8kw_choose(M, N, K, ws && aligned16(ws) ? ws_bytes : 0, p)) return false;
    uint64_t *cnt = p.ks > 1 ? (uint64_t *)ws : nullptr;
    float *part = p.ks > 1 ? (float *)((uint8_t *)ws + kWsHeader) : nullptr;
    auto go = [&](auto cfg) {
        typedef decltype(cfg) Cfg;
        auto one = [&](auto bf, auto qa) {
            constexpr bool BF = decltype(bf)::value, QA = decltype(qa)::value;
            return i8kw_launch<Cfg, BF, QA>(QA ? A : (const void *)Aq, SA, B, SB, C, Other, Bias, M, N, K, postop, out_f32,
                                            p.ks, part, cnt, st);
        };
        if (dtype == TERNOCL_BF16) return Aq ? one(std::true_type{}, std::false_type{}) : one(std::true_type{}, std::true_type{});
        return Aq ? one(std::false_type{}, std::false_type{}) : one(std::false_type{}, std::true_type{});
    };
    switch (p.tile) {
    case 0: e = go(KwCfg<1, 1, 1, 8>{}); break;
    case 1: e = go(KwCfg<1, 2, 1, 8>{}); break;
    case 2: e = go(KwCfg<1, 2, 1, 4>{}); break;
    default: e = go(KwCfg<1, 2, 2, 4>{}); break;
    }
    return true;
}

}  // namespace tcl
