// bitcos_kw.hip -- the M-tiled BITCOS GEMM of tens to hundreds of rows on gfx950
// (bitcos_fp16_upcvt_gemm_mt, bitcos_fp16_upcvt/bitcos_fp16_upcvt.cl:303-305): the
// K walk over waves of int2_gemm_kw.hip (gemm_kw.hpp), decoding the BITCOS
// weights on the way.
//
// The re-pack followed by the int2 engine streams the weights twice through a
// pass that is latency-bound at these sizes (10.5 us at K = N = 4096, 17.4 at K =
// 5376 N = 21504), and the 128-row tiles that decode in place take 70-92 us for
// any M.  Here a workgroup's waves each count their part's bitmap (a popcount a
// word, the ranks meet in LDS), then walk it: a word costs ~30 instructions more
// than the packed format's, once per row tile.  Measured (fp16, z = .5,
// graph-timed, us; with the re-pack workspace / without -> this): K = N = 4096, M =
// 16 52.9 / 71.9 -> 13.2, M = 128 52.3 / 72.2 -> 17.7, M = 256 53.6 / 71.9 -> 24.2; K = N =
// 5120, M = 128 62.8 / 89.9 -> 26.9; K = 5376 N = 21504, M = 32 74.2 / 95.5 -> 33.2, M =
// 64 74.3 / 95.5 -> 46.5.  What bounds it is the decode: ~24 instructions and four table reads per 16 rows.
#include "gemm_kw.hpp"

#include <algorithm>

namespace tcl {
int bitcos_pick_ls(int N, int K);  // bitcos.hip
// (int2_gemm_kw.hip)
void int2_gemm_kw_model(int M, int N, int K, double &kw_us, double &other_us, int &wk, bool &square);
namespace {

// BITCOS weights as the walk's B source (gemm_kw.hpp): per unit of 64 rows the
// lane's CB columns have two bitmap words each and, from the running rank on, up
// to 64 sign bits in three words of the column's stream.  Lane (c, q) decodes
// rows 32 t + 16 q .. + 15 (t = 0, 1) into the int2 word the packed format has
// there: each presence nibble and the next four sign bits index a 256-byte table
// of four codes.  Bitmap words are loaded PF units ahead, sign words two (their
// address needs the rank, which follows from the bitmaps).
template <int CB, int PF> struct KwBitcos {
    static_assert(PF >= 4, "sign words two units ahead of their unit, bitmaps two ahead of those");
    typedef typename KwVec<CB>::W W;
    typedef typename KwVec<CB>::S SV;
    const uint32_t *B;     // bitmap [K / 32][N] | offsets [N] | streams | pad
    const uint32_t *sg[CB];  // the columns' sign streams
    const uint16_t *S;
    const uint8_t *lut;
    int N, units, q;
    uint32_t col;
    W bm[PF][2];
    uint32_t sw[PF][CB][3], r0[PF][CB], rn[CB];
    SV sr[PF];
    __device__ __forceinline__ void load(int u, int s) {
        const int uc = min(u, units - 1);
        const uint32_t *p = B + (size_t)(2 * uc) * N + col;
        bm[s][0] = *(const W *)p;
        bm[s][1] = *(const W *)(p + N);
        sr[s] = *(const SV *)(S + (size_t)(uc >> 1) * N + col);
    }
    // unit u's sign words (past the end: the last unit's end, inside the pad), then
    // the rank after it
    __device__ __forceinline__ void signs(int u, int s) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const uint32_t *p = sg[cb] + (rn[cb] >> 5);
            r0[s][cb] = rn[cb];
#pragma unroll
            for (int i = 0; i < 3; ++i) sw[s][cb][i] = p[i];
        }
        if (u < units) {
            uint32_t a[CB], b[CB];
            __builtin_memcpy(a, &bm[s][0], sizeof(W));
            __builtin_memcpy(b, &bm[s][1], sizeof(W));
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) rn[cb] += __builtin_popcount(a[cb]) + __builtin_popcount(b[cb]);
        }
    }
    __device__ __forceinline__ void start(int u0) {
#pragma unroll
        for (int s = 0; s < PF; ++s) load(u0 + s, s);
        signs(u0, 0);
        signs(u0 + 1, 1);
    }
    __device__ __forceinline__ void next(int u, int s, bool more) {
        if (more) load(u + PF, s);
        signs(u + 2, (s + 2) % PF);
    }
    __device__ __forceinline__ void get(int s, uint32_t w[CB][2], uint32_t lo[CB], uint32_t hi[CB]) {
        uint32_t sc[(CB + 1) / 2] = {}, b[2][CB];
        __builtin_memcpy(sc, &sr[s], sizeof(SV));
        __builtin_memcpy(b[0], &bm[s][0], sizeof(W));
        __builtin_memcpy(b[1], &bm[s][1], sizeof(W));
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            kw_tables(sc[cb >> 1], cb & 1, lo[cb], hi[cb]);
            const uint32_t base = r0[s][cb] >> 5;
            uint32_t rt = r0[s][cb];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t x = b[t][cb], half = q ? x >> 16 : x & 0xffffu;
                const uint32_t r = rt + (q ? __builtin_popcount(x & 0xffffu) : 0u);
                if (t == 0) rt += __builtin_popcount(x);
                const uint32_t k = (r >> 5) - base;  // 0, 1 or 2 (2: its 16 bits end in that word)
                const uint32_t w0 = k == 0 ? sw[s][cb][0] : k == 1 ? sw[s][cb][1] : sw[s][cb][2];
                const uint32_t w1 = k == 0 ? sw[s][cb][1] : sw[s][cb][2];
                const uint32_t sign = __builtin_amdgcn_alignbit(w1, w0, r & 31u);
                uint32_t o = 0, p = 0;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t m4 = (half >> (4 * i)) & 15u;
                    const uint32_t s4 = (sign >> p) & 15u;
                    p += __builtin_popcount(m4);
                    o |= (uint32_t)lut[(m4 << 4) | s4] << (8 * i);
                }
                w[cb][t] = o;
            }
        }
    }
};

// (after the walk's LDS: the code table, then the waves' non-zero counts)
template <class Cfg> constexpr int bckw_lds() { return Cfg::LDS_BYTES + 256 + Cfg::WK * 32 * Cfg::CB * 4; }

template <class Cfg, bool BF16>
__global__ void __launch_bounds__(Cfg::THREADS)
k_bitcos_gemm_kw(const uint16_t *__restrict__ A, const uint32_t *__restrict__ Bc, const uint16_t *__restrict__ S,
                 void *__restrict__ C, const uint16_t *__restrict__ Other, const void *__restrict__ Bias, int M, int N,
                 int K, int postop, int out_f32) {
    constexpr int MB = Cfg::MB, CB = Cfg::CB, WK = Cfg::WK;
    extern __shared__ __attribute__((aligned(16))) uint8_t kw_lds[];
    const int mt = (M + Cfg::BM - 1) / Cfg::BM, nt = (N + Cfg::BN - 1) / Cfg::BN;
    int tm, tn;
    if (!xcd_tile_ashare(blockIdx.x, mt, nt, tm, tn)) return;  // whole workgroup: padding
    const int m0 = tm * Cfg::BM, n0 = tn * Cfg::BN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kw = wave / Cfg::WM, wm = wave % Cfg::WM;
    const int c = lane & 31, q = lane >> 5;
    const int units = K / 64, u0 = units * kw / WK, u1 = units * (kw + 1) / WK;
    const int mrows = min(Cfg::BM, M - m0);
    uint8_t *lut = kw_lds + Cfg::LDS_BYTES;
    uint32_t *cnt = (uint32_t *)(lut + 256);  // [WK][32 CB]: non-zeros of each wave's part per column
    for (int i = tid; i < 256; i += Cfg::THREADS) {
        // (presence nibble m, next four sign bits): row j present takes the next sign
        const uint32_t m = (uint32_t)i >> 4, sgn = (uint32_t)i & 15u;
        uint32_t taken = 0, out = 0;
        for (int j = 0; j < 4; ++j)
            if ((m >> j) & 1u) {
                out |= (((sgn >> taken) & 1u) ? 3u : 1u) << (2 * j);
                ++taken;
            }
        lut[i] = (uint8_t)out;
    }
    const uint32_t col = (uint32_t)min(n0 + CB * c, N - CB);
    KwBitcos<CB, Cfg::PF> bs;
    typedef typename KwVec<CB>::W W;
    bs.B = Bc;
    bs.S = S;
    bs.lut = lut;
    bs.N = N;
    bs.units = units;
    bs.q = q;
    bs.col = col;
    // The wave's first rank: every wave counts its own part's bitmap (lane q: word 2 u +
    // q), the sums meet in LDS.
    uint32_t n[CB] = {};
    for (int u = u0; u < u1; u += 8) {
        W x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) x[i] = *(const W *)(Bc + (size_t)(2 * min(u + i, u1 - 1) + q) * N + col);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            uint32_t y[CB];
            __builtin_memcpy(y, &x[i], sizeof(W));
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) n[cb] += u + i < u1 ? __builtin_popcount(y[cb]) : 0;
        }
    }
    const uint32_t *off = Bc + (size_t)(K >> 5) * N;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        n[cb] += __shfl_xor(n[cb], 32);
        bs.sg[cb] = off + N + off[col + cb];
        if (wm == 0) cnt[kw * 32 * CB + CB * c + cb] = n[cb];  // (both lanes q: the same value)
    }
    __syncthreads();
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        uint32_t r = 0;
        for (int k = 0; k < kw; ++k) r += cnt[k * 32 * CB + CB * c + cb];
        bs.rn[cb] = r;
    }
    uint32_t va[4 * MB];
#pragma unroll
    for (int i = 0; i < 4 * MB; ++i)
        va[i] = (uint32_t)min(32 * MB * wm + (lane >> 3) + 8 * i, mrows - 1) * (uint32_t)K + 8u * (lane & 7);
    f32x16_t acc[MB][CB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[mb][cb] = f32x16_t{};
    kw_walk<Cfg, BF16>(kw_lds + wave * (MB * 8192), A + (size_t)m0 * K, va, u0, u1, units, bs, acc);
    kw_finish<Cfg, BF16>(acc, kw_lds, C, Other, Bias, M, N, m0, mrows, n0, postop, out_f32, 1, 0, nullptr, nullptr);
}

template <class Cfg, bool BF16>
hipError_t bckw_launch(const void *A, const uint32_t *Bc, const void *S, void *C, const void *Other, const void *Bias, int M,
                       int N, int K, int postop, int out_f32, hipStream_t st) {
    const int mt = (M + Cfg::BM - 1) / Cfg::BM, nt = (N + Cfg::BN - 1) / Cfg::BN;
    hipLaunchKernelGGL((k_bitcos_gemm_kw<Cfg, BF16>), dim3(xcd_ashare_grid(mt, nt)), dim3(Cfg::THREADS), bckw_lds<Cfg>(),
                       st, (const uint16_t *)A, Bc, (const uint16_t *)S, C, (const uint16_t *)Other, Bias, M, N, K, postop,
                       out_f32);
    return hipGetLastError();
}

// ---- host side: tile choice ----------------------------------------------------

// The compiled tiles (rows, columns, waves over K) and their launches' times: once +
// round R + (once_k + round_k R) k us for R rounds of 256 workgroups (a last one of
// few costs a whole one; the 64 x 64 tile of four waves and the 32 x 32 one, two a
// CU, less), k in 1024 rows.  Fitted to 15754 graph-timed sizes (both types, z = .3,
// .5, .7, M = 9..1024, K = 128..14336, N = 16..34816), within 6% for 5..95% of each
// round's.  A fit linear in the workgroups took a tile at 1.2 rounds for 1.2 times
// one round's time: M = 459 K = 768 N = 2400 19.6 us against the re-pack and the
// 128-row tiles' 17.6, M = 54 K = 896 N = 33376 29.2 against 21.9 for those decoding
// in place.
struct BcTile {
    int bm, bn, wk;
    double once, round, once_k, round_k;
};
constexpr BcTile kBcTiles[] = {{32, 32, 8, 4.5, 1.6, 0.6, 1.28}, {64, 32, 8, 3.3, 3.95, 0.2, 2.2},
                               {64, 64, 8, 3.4, 5.4, 0.3, 3.45}, {64, 64, 4, 5.3, 2.2, 1.5, 3.05}};

double bckw_us(const BcTile &t, long wgs, double k) {
    const double r = (double)((wgs + 255) / 256);
    return t.once + t.round * r + (t.once_k + t.round_k * r) * k;
}

// The cheapest tile with wk waves over K (0: any).
int bckw_tile(int M, int N, int K, int wk, double &us) {
    int best = -1;
    us = 1e30;
    for (int i = 0; i < 4; ++i) {
        const BcTile &t = kBcTiles[i];
        if ((wk && t.wk != wk) || (wk == 0 && t.bm > 32 && t.bm >= 2 * M)) continue;
        const double u = bckw_us(t, (long)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn), K / 1024.0);
        if (u < us) {
            us = u;
            best = i;
        }
    }
    return best;
}

// The route of a call by (M, N, K) alone, the same with and without the
// re-pack workspace: a sum's bits depend on the waves over K only, so the two
// calls agree bit for bit -- through these tiles, or the re-packed words on the
// int2 engine's with as many waves over K, or (false) the 128-row tiles.  tile: of
// kBcTiles; repacked: with a workspace the re-pack is ahead.
bool bckw_route(int M, int N, int K, int &tile, bool &repacked) {
    if (M <= 8 || M > 1024) return false;
    double direct, kw, other, chosen;
    int kwk, wk;
    bool square;
    const int t = bckw_tile(M, N, K, 0, direct);
    int2_gemm_kw_model(M, N, K, kw, other, kwk, square);
    // k_bitcos_to_int2: a wave a slice walks its rows.  The slices are the caller's and bits
    // must not depend on them: the library's own choice counts.  (5..95% of the sizes
    // above within 0.88..1.09; without the slices 10 - 16 us were counted for 27 - 60 at K
    // above ~5000 with few slices: M = 71 K = 10624 N = 4560 73.5 us against 40.4 direct.)
    const double k = K / 1024.0, repack = 4.3 + 6.35 * k / bitcos_pick_ls(N, K) + 0.67 * k + 7.4e-8 * K * N;
    repacked = repack + kw < direct;
    wk = repacked ? kwk : kBcTiles[t].wk;
    tile = bckw_tile(M, N, K, wk, chosen);
    // ahead (by more than the fits' spread) of the re-pack and the 128-row tiles, and
    // without the workspace of the tiles that decode in place: 1.7 - 1.9x the int2 ones
    // on 128 x 128, 1.15 - 1.3x on the wider
    return std::min(direct, repack + kw) < 0.95 * (repack + other) && chosen < 0.95 * (square ? 1.5 : 1.2) * other;
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// (for ternocl_kw_tile_of: the tile of an M-tiled call on aligned operands; repacked:
// the workspace form runs int2_gemm_kw_run on the re-packed words)
bool bitcos_kw_tile(int M, int N, int K, ternocl_kw_tile &t) {
    int tile;
    bool repacked;
    if (!bckw_route(M, N, K, tile, repacked)) return false;
    const BcTile &b = kBcTiles[tile];
    t = {b.bm, b.bn, b.wk, 1, repacked};
    return true;
}

// How a call of the M-tiled entry runs here: 0 not, 1 bitcos_kw_run on `tile`, 2
// (repack: the caller re-packs the weights) int2_gemm_kw_run on the re-packed words.
int bitcos_kw_auto(int M, int N, int K, bool repack, const void *A, const void *Bc, const void *S, const void *C,
                   const void *Other, const void *Bias, int &tile) {
    bool repacked;
    if (!aligned16(A) || !aligned16(Bc) || !aligned16(S) || !aligned16(C) || !aligned16(Other) || !aligned16(Bias) ||
        !bckw_route(M, N, K, tile, repacked))
        return 0;
    return repack && repacked ? 2 : 1;
}

ternocl_status bitcos_kw_run(int dtype, const void *A, const uint32_t *Bc, const void *S, void *C, const void *Other,
                             const void *Bias, int M, int N, int K, int postop, int out_f32, int tile, hipStream_t st) {
    const bool bf = dtype == TERNOCL_BF16;
    auto go = [&](auto cfg) {
        typedef decltype(cfg) Cfg;
        return bf ? bckw_launch<Cfg, true>(A, Bc, S, C, Other, Bias, M, N, K, postop, out_f32, st)
                  : bckw_launch<Cfg, false>(A, Bc, S, C, Other, Bias, M, N, K, postop, out_f32, st);
    };
    hipError_t e;
    switch (tile) {
    case 0: e = go(KwCfg<1, 1, 1, 8, 4>{}); break;
    case 1: e = go(KwCfg<2, 1, 1, 8, 4>{}); break;
    case 2: e = go(KwCfg<2, 2, 1, 8, 4>{}); break;
    default: e = go(KwCfg<2, 2, 1, 4, 4>{}); break;
    }
    return launch_status(e);
}

}  // namespace tcl
