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
//   * What bounds it: the traffic of the activations through L1 and LDS (each
//     wave stores and reads every chunk of its rows once per 32 CB columns), not
//     the weight stream: prefetching weights two or four units ahead measures
//     the same, and a copy without the activation loads and stores takes half
//     the time (M = 64, K = 5120, N = 34816: 50 -> 22-33 us over the tiles).
//     Storing unit u itself at its start, on the critical path: 24 -> 21.7 us
//     with the two buffers (M = 128, K = 4096, N = 14336).
// Measured against the engines these calls took before (graph-timed, bf16,
// rotated weights, us; M = 9..16 the MFMA GEMV, above the 128-row tiles):
//   M = 16, K = 4096 N = 4096 16.6 -> 8.2, N = 14336 21.0 -> 10.6, K = 14336 N =
//   4096 54.0 -> 18.2; M = 32 39.8 -> 8.5, 40.5 -> 10.9, 130.6 -> 13.3; M = 128
//   40.2 -> 11.8, 40.6 -> 21.7, 130.9 -> 25.6; M = 256 K = 4096 N = 4096 40.5 ->
//   15.8; M = 512 43.5 -> 24.5.
#include "common.hpp"

#include <algorithm>

namespace tcl {
// (int2_gemm_mfma.hip)
bool gemm_half_tile(int M, int N);
int gemm_splits(int M, int N, int K);
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf168_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

template <bool BF16>
__device__ __forceinline__ f32x16_t kw_mfma(const u32x4_t &a, const uint32_t b[4], f32x16_t c) {
    if constexpr (BF16) {
        bf168_t x, y;
        __builtin_memcpy(&x, &a, 16);
        __builtin_memcpy(&y, b, 16);
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    } else {
        half8_t x, y;
        __builtin_memcpy(&x, &a, 16);
        __builtin_memcpy(&y, b, 16);
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(x, y, c, 0, 0, 0);
    }
}

// A tile of WM x WK waves: wave (wm, kw) computes rows 32 MB wm .. + 32 MB of the
// tile's 32 CB columns over the kw-th part of the K units.  PF: units of weights
// in flight per wave.
template <int MB_, int CB_, int WM_, int WK_, int PF_ = 2> struct KwCfg {
    static constexpr int MB = MB_, CB = CB_, WM = WM_, WK = WK_;
    static constexpr int PF = PF_;
    static_assert(PF % 2 == 0, "two LDS buffers in turn");
    static constexpr int THREADS = 64 * WM * WK;
    static constexpr int BM = 32 * MB * WM, BN = 32 * CB;
    static constexpr int NRB = WM * MB;                  // 32-row blocks of the tile
    static constexpr int A_BYTES = WM * WK * MB * 8192;        // two 64-k units of each wave's rows
    static constexpr int RB_BYTES = CB * WK * 4096;      // the wave partials of one row block
    static constexpr int RPR = NRB * RB_BYTES <= 131072 ? NRB : 131072 / RB_BYTES;  // row blocks per round
    static constexpr int LDS_BYTES = A_BYTES > RPR * RB_BYTES ? A_BYTES : RPR * RB_BYTES;
    static constexpr int ITEMS = (RPR * 256 + THREADS - 1) / THREADS;
    static_assert(NRB % RPR == 0, "whole rounds");
};

// CB consecutive words / scales of one row
template <int CB> struct KwVec;
template <> struct KwVec<1> { typedef uint32_t W; typedef uint16_t S; };
template <> struct KwVec<2> { typedef u32x2_t W; typedef uint32_t S; };
template <> struct KwVec<4> { typedef u32x4_t W; typedef u32x2_t S; };

// Epilogue and store of CB adjacent outputs (m, n .. n + CB - 1), n a multiple of CB.
template <int CB, bool BF16, int P, bool F32>
__device__ __forceinline__ void kw_store(void *C, const uint16_t *Other, const void *Bias, int N, int m, int n,
                                         const float v[CB]) {
    if constexpr (CB == 4) {
        epi_store4_c<BF16, P, F32>(C, Other, Bias, N, m, n, v);
    } else if constexpr (CB == 1) {
        epi_store1_c<BF16, P, F32>(C, Other, Bias, N, m, n, v[0]);
    } else {
        const size_t i = (size_t)m * N + n;
        float o[2] = {0.f, 0.f}, b[2] = {0.f, 0.f};
        if constexpr (postop_needs_other(P)) {
            const uint32_t t = *(const uint32_t *)(Other + i);
            o[0] = dt2f<BF16>(t & 0xffffu);
            o[1] = dt2f<BF16>(t >> 16);
        }
        if constexpr (postop_needs_bias(P)) {
            if constexpr (F32) {
                const float2 t = *(const float2 *)((const float *)Bias + n);
                b[0] = t.x;
                b[1] = t.y;
            } else {
                const uint32_t t = *(const uint32_t *)((const uint16_t *)Bias + n);
                b[0] = dt2f<BF16>(t & 0xffffu);
                b[1] = dt2f<BF16>(t >> 16);
            }
        }
        const float r0 = epi_apply_c<P>(v[0], o[0], b[0]), r1 = epi_apply_c<P>(v[1], o[1], b[1]);
        if constexpr (F32) *(float2 *)((float *)C + i) = make_float2(r0, r1);
        else *(uint32_t *)((uint16_t *)C + i) = f2dt<BF16>(r0) | (f2dt<BF16>(r1) << 16);
    }
}

// ksn > 1: workgroup (tile, slice sl) runs the units of its K slice and stores
// its sums in part [ksn][M][N] (agent-scope stores); the last of a tile's ksn
// workgroups (its counter, split_arrive) adds the slices in order and applies
// the epilogue -- the handoff of the decode GEMV's K split (int2_gemv_f4.hip).
template <class Cfg, bool BF16>
__global__ void __launch_bounds__(Cfg::THREADS)
k_int2_gemm_kw(const uint16_t *__restrict__ A, const uint32_t *__restrict__ B, const uint16_t *__restrict__ S,
               void *__restrict__ C, const uint16_t *__restrict__ Other, const void *__restrict__ Bias, int M, int N,
               int K, int postop, int out_f32, int ksn, float *part, uint32_t *cnt) {
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
    const uint16_t *Ab = A + (size_t)m0 * K;
    // B: lane (c, q) holds word 4 u + 2 t + q (t = 0, 1) of columns n0 + CB c .. + CB - 1
    // (columns past N re-read the last ones); MFMA k-step 2 t + h multiplies rows
    // 8 h .. 8 h + 7 of words 2 t, 2 t + 1
    const uint32_t col = (uint32_t)min(n0 + CB * c, N - CB);
    const uint32_t vb0 = q * (uint32_t)N + col, vb1 = vb0 + 2u * (uint32_t)N;
    u32x4_t av[4 * MB];
    typedef typename KwVec<CB>::W W;
    typedef typename KwVec<CB>::S SV;
    constexpr int PF = Cfg::PF;
    W bw[PF][2];
    SV sr[PF];
    // (units past the end re-read the last one: loaded, never multiplied)
    auto a_load = [&](int u) __attribute__((always_inline)) {
        const uint16_t *p = Ab + 64 * (size_t)min(u, units - 1);
#pragma unroll
        for (int i = 0; i < 4 * MB; ++i) av[i] = *(const u32x4_t *)(p + va[i]);
    };
    auto b_load = [&](int u, int s) __attribute__((always_inline)) {
        const int uc = min(u, units - 1);
        const uint32_t *p = B + (size_t)(4 * uc) * N;
        bw[s][0] = __builtin_nontemporal_load((const W *)(p + vb0));
        bw[s][1] = __builtin_nontemporal_load((const W *)(p + vb1));
        sr[s] = *(const SV *)(S + (size_t)(uc >> 1) * N + col);
    };
    uint8_t *abuf = kw_lds + wave * (MB * 8192);
    uint8_t *aw = abuf + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    uint32_t ar[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ar[i] = (uint32_t)(c * 128 + (((4 * (i >> 1) + 2 * q + (i & 1)) ^ (c & 7)) << 4));

    f32x16_t acc[MB][CB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[mb][cb] = f32x16_t{};
    uint32_t km = 0x03030303u, ko = 0x04000400u;
    asm("" : "+v"(km));
    asm("" : "+s"(ko));

    auto a_store = [&](int p) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4 * MB; ++i) *(u32x4_t *)(aw + p * (MB * 4096) + 1024 * i) = av[i];
    };
    u32x4_t af[2][MB];
    auto a_frag = [&](int p, int i, u32x4_t f[MB]) __attribute__((always_inline)) {
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) f[mb] = *(const u32x4_t *)(abuf + p * (MB * 4096) + ar[i] + 4096 * mb);
    };
    auto unit = [&](int u, int s, bool more) __attribute__((always_inline)) {
        const int p = s & 1;
        uint32_t w[CB][2], lo[CB], hi[CB];
        uint32_t sw[(CB + 1) / 2];
        __builtin_memcpy(sw, &sr[s], sizeof(SV));
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            uint32_t t0[CB], t1[CB];
            __builtin_memcpy(t0, &bw[s][0], sizeof(W));
            __builtin_memcpy(t1, &bw[s][1], sizeof(W));
            w[cb][0] = t0[cb];
            w[cb][1] = t1[cb];
            const uint32_t x = sw[cb >> 1];
            lo[cb] = __builtin_amdgcn_perm(x, x, (cb & 1) ? 0x020c020cu : 0x000c000cu);
            hi[cb] = __builtin_amdgcn_perm(x, x, (cb & 1) ? 0x030c030cu : 0x010c010cu) ^ 0x80000000u;
        }
        if (more) b_load(u + PF, s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // MFMA k-steps: word t = i / 2, half h = i % 2
            if (i == 2) {
                __builtin_amdgcn_sched_barrier(0);
                a_store(p ^ 1);
                a_load(u + 2);
                __builtin_amdgcn_sched_barrier(0);
            }
            a_frag(i < 3 ? p : p ^ 1, (i + 1) & 3, af[(i + 1) & 1]);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                const uint32_t x = w[cb][i >> 1], x2 = x >> 2;
                uint32_t b[4];
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const uint32_t y = 2 * (i & 1) + d;  // byte of the word
                    const uint32_t t = __builtin_amdgcn_perm(x2, x, ((4 + y) << 24) | ((4 + y) << 16) | (y << 8) | y);
                    b[2 * d] = __builtin_amdgcn_perm(hi[cb], lo[cb], (t & km) | ko);
                    b[2 * d + 1] = __builtin_amdgcn_perm(hi[cb], lo[cb], ((t >> 4) & km) | ko);
                }
#pragma unroll
                for (int mb = 0; mb < MB; ++mb) acc[mb][cb] = kw_mfma<BF16>(af[i & 1][mb], b, acc[mb][cb]);
            }
        }
    };
    if (u0 < u1) {
        a_load(u0);
#pragma unroll
        for (int s = 0; s < PF; ++s) b_load(u0 + s, s);
        __builtin_amdgcn_sched_barrier(0);
        a_store(0);
        a_load(u0 + 1);
        __builtin_amdgcn_sched_barrier(0);
        a_frag(0, 0, af[0]);
        int u = u0;
        for (; u + PF - 1 < u1; u += PF)
#pragma unroll
            for (int s = 0; s < PF; ++s) unit(u + s, s, true);
#pragma unroll
        for (int s = 0; s < PF - 1; ++s) {
            if (u + s >= u1) break;
            unit(u + s, s, false);
        }
    }

    // sums of the waves' K parts in wave order, a round of row blocks at a time
    auto rows_of = [&](int it, int &r, int &n) __attribute__((always_inline)) {
        // item `it` of a round: row block it / 256, register quad (it / 64) % 4, this lane
        r = 32 * (it >> 8) + 8 * ((it >> 6) & 3) + 4 * q;
        n = n0 + CB * c;
    };
    auto finish = [&](int r, int n, const float (*v)[4]) __attribute__((always_inline)) {
        epi_dispatch(postop, out_f32, [&](auto P_, auto F_) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (r + i < mrows && n < N) {
                    float x[CB];
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb) x[cb] = v[cb][i];
                    kw_store<CB, BF16, decltype(P_)::value, decltype(F_)::value>(C, Other, Bias, N, m0 + r + i, n, x);
                }
        });
    };
    float *red = (float *)kw_lds;
#pragma unroll
    for (int rd = 0; rd < Cfg::NRB / Cfg::RPR; ++rd) {
        __syncthreads();  // the A buffers, or the last round's partials, are free
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int rb = wm * MB + mb;
            if (rb / Cfg::RPR == rd)  // (uniform)
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        *(f32x4_t *)(red + (size_t)((((rb % Cfg::RPR) * CB + cb) * WK + kw) * 256 + j * 64 + lane) * 4) =
                            f32x4_t{acc[mb][cb][4 * j], acc[mb][cb][4 * j + 1], acc[mb][cb][4 * j + 2], acc[mb][cb][4 * j + 3]};
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < Cfg::ITEMS; ++t) {
            const int it = tid + Cfg::THREADS * t;
            if (it >= Cfg::RPR * 256) break;  // (whole waves)
            float v[CB][4];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                f32x4_t s = f32x4_t{};
#pragma unroll
                for (int k = 0; k < WK; ++k) {
                    const f32x4_t x = *(const f32x4_t *)(red + (size_t)((((it >> 8) * CB + cb) * WK + k) * 256 + (it & 255)) * 4);
                    if (k == 0) s = x;
                    else
#pragma unroll
                        for (int i = 0; i < 4; ++i) s[i] += x[i];
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) v[cb][i] = s[i];
            }
            int r, n;
            rows_of(it, r, n);
            r += 32 * Cfg::RPR * rd;
            if (ksn == 1) {
                finish(r, n, v);
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (r + i < mrows && n < N) {
                        float *p = part + ((size_t)sl * M + m0 + r + i) * N + n;
                        if constexpr (CB == 1) {
                            __hip_atomic_store(p, v[0][i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        } else {
#pragma unroll
                            for (int cb = 0; cb < CB; cb += 2) {
                                const uint64_t x = (uint64_t)__float_as_uint(v[cb][i]) | ((uint64_t)__float_as_uint(v[cb + 1][i]) << 32);
                                __hip_atomic_store((uint64_t *)(p + cb), x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            }
                        }
                    }
            }
        }
    }
    if (ksn == 1) return;
    // the last of the tile's ksn workgroups adds the slices in order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();  // every wave's sums are stored
    uint32_t *flag = (uint32_t *)kw_lds;
    if (wave == 0) {
        const uint32_t prev = split_arrive(cnt + (size_t)tm * nt + tn, ksn, lane);
        if (lane == 0) *flag = prev;
    }
    __syncthreads();
    if (*flag != (uint32_t)(ksn - 1)) return;  // (uniform)
    for (int it = tid; it < Cfg::NRB * 256; it += Cfg::THREADS) {
        int r, n;
        rows_of(it, r, n);
        if (n >= N) continue;
        float v[CB][4];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int i = 0; i < 4; ++i) v[cb][i] = 0.0f;
        for (int s0 = 0; s0 < ksn; s0 += 2) {  // two slices' loads in flight
            float x[2][CB][4];
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float *p = part + ((size_t)min(s0 + e, ksn - 1) * M + m0 + min(r + i, mrows - 1)) * N + n;
                    if constexpr (CB == 1) {
                        x[e][0][i] = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    } else {
#pragma unroll
                        for (int cb = 0; cb < CB; cb += 2) {
                            const uint64_t y = __hip_atomic_load((const uint64_t *)(p + cb), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            x[e][cb][i] = __uint_as_float((uint32_t)y);
                            x[e][cb + 1][i] = __uint_as_float((uint32_t)(y >> 32));
                        }
                    }
                }
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                if (s0 + e >= ksn) break;
#pragma unroll
                for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                    for (int i = 0; i < 4; ++i) v[cb][i] = s0 + e == 0 ? x[e][cb][i] : v[cb][i] + x[e][cb][i];
            }
        }
        finish(r, n, v);
    }
}

template <class Cfg, bool BF16>
hipError_t kw_launch(const void *A, const uint32_t *B, const void *S, void *C, const void *Other, const void *Bias, int M,
                     int N, int K, int postop, int out_f32, int ksn, float *part, uint32_t *cnt, hipStream_t st) {
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
            if (ks > 1 && (!split || K / ks < 512 || tiles * 4 > (long)kWsHeader)) break;
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
// us), 128 x 256 tiles (M = 1024, K = 4096, N = 6144: 66.7; M = 194, K = 13184, N =
// 23936: 183), 128 x 512 tiles (N = 14336: 103) and their K split.  Both fits are
// good to some 5%, so this engine is taken where it is ahead by more (kKwMargin).
constexpr double kKwMargin = 0.95;
double kw_other_us(int M, int N, int K, bool split) {
    auto tiles = [&](int BM, int BN) { return (double)((long)((M + BM - 1) / BM) * ((N + BN - 1) / BN)); };
    const double k = K / 1024.0, wide = tiles(128, 512), half = tiles(128, 256), square = tiles(128, 128);
    if (wide >= 192) return 5.0 + 24.5 * k * (wide <= 256 ? 1.0 : wide / 256.0);
    const bool h = gemm_half_tile(M, N);
    const int ks = split && !(h && half >= 192) ? gemm_splits(M, N, K) : 1;
    if (ks > 1) return 8.0 + 24.5 * k / ks + 8e-6 * ks * M * N / 4.0;
    if (h) return 8.0 + 13.8 * k;
    if (square <= 512) return 3.2 + (9.3 + 1.8 * std::min(square, 256.0) / 256.0) * k * (square > 256 ? 1.5 : 1.0);
    return 5.0 + 24.5 * k * (wide <= 256 ? 1.0 : wide / 256.0);
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }

}  // namespace

// Whether the automatic engine of a call of M > 8 rows is this one: always up
// to 16 rows (the MFMA GEMV is 2-3x its time there), above where its model is
// ahead of the 128-row tile engine's.  split: whether K slices may use a
// workspace.  The vector loads and stores need 16-byte aligned operands.
bool int2_gemm_kw_auto(int M, int N, int K, bool split, const void *A, const void *B, const void *S, const void *C,
                       const void *Other, const void *Bias) {
    if (M <= 8 || !aligned16(A) || !aligned16(B) || !aligned16(S) || !aligned16(C) || !aligned16(Other) || !aligned16(Bias))
        return false;
    if (M <= 16) return true;
    return M <= 2048 && kw_plan(M, N, K, split).us < kKwMargin * kw_other_us(M, N, K, split);
}

// Workspace of the automatic plan's K split (0: none; none up to 16 rows).
size_t int2_gemm_kw_ws_need(int M, int N, int K) {
    if (M <= 16 || M > 2048) return 0;
    const KwPlan p = kw_plan(M, N, K, true);
    return p.ks > 1 && p.us < kKwMargin * kw_other_us(M, N, K, true) ? kWsHeader + (size_t)p.ks * M * N * 4 : 0;
}

// split: K slices may use ws (int2_gemm_kw_ws_need bytes, 16-byte aligned).
ternocl_status int2_gemm_kw_run(int dtype, const void *A, const uint32_t *B, const void *S, void *C, const void *Other,
                                const void *Bias, int M, int N, int K, int postop, int out_f32, hipStream_t st,
                                bool split, void *ws) {
    const KwPlan p = kw_plan(M, N, K, split && M > 16);
    uint32_t *cnt = p.ks > 1 ? (uint32_t *)ws : nullptr;
    float *part = p.ks > 1 ? (float *)((uint8_t *)ws + kWsHeader) : nullptr;
    const bool bf = dtype == TERNOCL_BF16;
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
    return launch_status(e);
}

}  // namespace tcl
