// gemm_kw.hpp -- the GEMMs that split K over the waves of a workgroup
// (int2_gemm_kw.hip): tile shapes, the K walk on DT activations, and the wave
// and slice sums with the epilogue.
#pragma once

#include "common.hpp"

namespace tcl {
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

// Byte tables of one column's scale (half `odd` of the pair x): lo = {0, s.lo, 0,
// s.lo}, hi = {0, s.hi, 0, s.hi ^ 0x80}
__device__ __forceinline__ void kw_tables(uint32_t x, int odd, uint32_t &lo, uint32_t &hi) {
    lo = __builtin_amdgcn_perm(x, x, odd ? 0x020c020cu : 0x000c000cu);
    hi = __builtin_amdgcn_perm(x, x, odd ? 0x030c030cu : 0x010c010cu) ^ 0x80000000u;
}

// Packed int2 weights as the walk's B source: lane (c, q) holds words 4 u + q and
// 4 u + 2 + q of unit u for its CB adjacent columns, and their scales.  B and S
// start at the matrix; col is the lane's first column, below N.
template <int CB, int PF> struct KwInt2 {
    typedef typename KwVec<CB>::W W;
    typedef typename KwVec<CB>::S SV;
    const uint32_t *B;
    const uint16_t *S;
    int N, units;
    uint32_t vb0, vb1, col;
    W bw[PF][2];
    SV sr[PF];
    __device__ __forceinline__ KwInt2(const uint32_t *B_, const uint16_t *S_, int N_, int units_, uint32_t col_, int q)
        : B(B_), S(S_), N(N_), units(units_), vb0(q * (uint32_t)N_ + col_), vb1((q + 2) * (uint32_t)N_ + col_), col(col_) {}
    // (units past the end re-read the last one: loaded, never multiplied)
    __device__ __forceinline__ void load(int u, int s) {
        const int uc = min(u, units - 1);
        const uint32_t *p = B + (size_t)(4 * uc) * N;
        bw[s][0] = __builtin_nontemporal_load((const W *)(p + vb0));
        bw[s][1] = __builtin_nontemporal_load((const W *)(p + vb1));
        sr[s] = *(const SV *)(S + (size_t)(uc >> 1) * N + col);
    }
    __device__ __forceinline__ void start(int u0) {
#pragma unroll
        for (int s = 0; s < PF; ++s) load(u0 + s, s);
    }
    // unit u's words are taken from slot s: refill it (more: a unit u + PF may follow)
    __device__ __forceinline__ void next(int u, int s, bool more) {
        if (more) load(u + PF, s);
    }
    // slot s's words and each column's scale byte tables {0, s, 0, -s}
    __device__ __forceinline__ void get(int s, uint32_t w[CB][2], uint32_t lo[CB], uint32_t hi[CB]) {
        uint32_t sw[(CB + 1) / 2] = {}, t0[CB], t1[CB];
        __builtin_memcpy(sw, &sr[s], sizeof(SV));
        __builtin_memcpy(t0, &bw[s][0], sizeof(W));
        __builtin_memcpy(t1, &bw[s][1], sizeof(W));
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            w[cb][0] = t0[cb];
            w[cb][1] = t1[cb];
            kw_tables(sw[cb >> 1], cb & 1, lo[cb], hi[cb]);
        }
    }
};

// Two matrices of the same shape side by side (the MoE layer's up and gate): the
// lane's first CB / 2 column blocks are a's columns, the others b's same columns.
template <int CB, int PF> struct KwDual {
    KwInt2<CB / 2, PF> a, b;
    __device__ __forceinline__ void start(int u0) {
        a.start(u0);
        b.start(u0);
    }
    __device__ __forceinline__ void next(int u, int s, bool more) {
        a.next(u, s, more);
        b.next(u, s, more);
    }
    __device__ __forceinline__ void get(int s, uint32_t w[CB][2], uint32_t lo[CB], uint32_t hi[CB]) {
        a.get(s, w, lo, hi);
        b.get(s, w + CB / 2, lo + CB / 2, hi + CB / 2);
    }
};

// The K walk of one wave: units [u0, u1) (64 rows of K each) of its 32 MB rows
// into acc.  abuf: the wave's LDS (two units); A + va[i] (elements) + 64 u: the
// 16-byte chunk lane % 8 of its row i * 8 + lane / 8.
template <class Cfg, bool BF16, class BS>
__device__ __forceinline__ void kw_walk(uint8_t *abuf, const uint16_t *A, const uint32_t va[4 * Cfg::MB], int u0, int u1,
                                        int units, BS &bs, f32x16_t acc[Cfg::MB][Cfg::CB]) {
    constexpr int MB = Cfg::MB, CB = Cfg::CB, PF = Cfg::PF;
    const int lane = threadIdx.x & 63, c = lane & 31, q = lane >> 5;
    u32x4_t av[4 * MB];
    auto a_load = [&](int u) __attribute__((always_inline)) {
        const uint16_t *p = A + 64 * (size_t)min(u, units - 1);
#pragma unroll
        for (int i = 0; i < 4 * MB; ++i) av[i] = *(const u32x4_t *)(p + va[i]);
    };
    // chunk j of row r at position j ^ (r % 8) of its 128 bytes; MFMA k-step 2 t + h
    // of lane (c, q) reads row c's chunk 4 t + 2 q + h: rows 8 h .. 8 h + 7 of word 2 t + q
    uint8_t *aw = abuf + (lane >> 3) * 128 + (((lane & 7) ^ (lane >> 3)) << 4);
    uint32_t ar[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) ar[i] = (uint32_t)(c * 128 + (((4 * (i >> 1) + 2 * q + (i & 1)) ^ (c & 7)) << 4));
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
        bs.get(s, w, lo, hi);
        bs.next(u, s, more);
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
        bs.start(u0);
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
}

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

// A slice's arrival at its tile's counter (lane 0's atomics, broadcast): whether it
// is the last of ksn.  Two 64-bit words, 0 between calls; the first counts in steps
// of kKwStep.  A value that no count gives is left from another use of the
// workspace's memory (these calls' earlier engines took a workspace that nothing
// had zeroed): every slice of the tile then sees one, and they count again in the
// second word, by exchanges that take any value but a count of theirs for none.
// The last arrival zeroes the words.  One atomic addition on a zeroed workspace:
// counting by exchanges alone, retried whenever another slice arrives, took 4 us
// more at 7 and 8 slices (M = 43 K = 7040 N = 512 9.0 -> 13.2).
constexpr uint64_t kKwStep = 0x9E6D3A5171C3B20Full;
__device__ __forceinline__ bool kw_arrive(uint64_t *c, int ksn, int lane) {
    bool last = false;
    if (lane == 0) {
        const uint64_t seen = __hip_atomic_fetch_add(c, kKwStep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        last = seen == (uint64_t)(ksn - 1) * kKwStep;
        bool count = last;
        for (int n = 0; n < ksn - 1 && !count; ++n) count = seen == (uint64_t)n * kKwStep;
        if (!count) {
            uint64_t e = 0;
            uint32_t n;
            do {  // (again only where another of the ksn slices arrived, or after the first guess)
                n = 0;
                for (int i = 1; i < ksn; ++i)
                    if (e == kKwStep + (uint64_t)i) n = (uint32_t)i;
                last = n == (uint32_t)(ksn - 1);
            } while (!last && !__hip_atomic_compare_exchange_strong(c + 1, &e, kKwStep + n + 1, __ATOMIC_RELAXED,
                                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
            if (last) __hip_atomic_store(c + 1, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (last) __hip_atomic_store(c, (uint64_t)0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return __builtin_amdgcn_readfirstlane((uint32_t)last) != 0;
}

// The sums of the waves' K parts in wave order (through LDS, a round of row
// blocks at a time), then the epilogue of the tile's rows [0, mrows) (C rows from
// m0) and columns [n0, n0 + 32 CB) (below N).  ksn > 1: slice sl's sums go to part
// [ksn][M][N] (agent-scope stores), and the last of the tile's ksn workgroups
// (its counter cnt, kw_arrive) adds the slices in order -- the handoff of the
// decode GEMV's K split (int2_gemv_f4.hip).  DUAL (KwDual's sums, ksn == 1): C =
// DT(silu(gate) * DT(up)) on CB / 2 columns a lane, the bits of the up product
// stored in DT and read by the gate product's epilogue.
template <class Cfg, bool BF16, bool DUAL = false>
__device__ __forceinline__ void kw_finish(f32x16_t acc[Cfg::MB][Cfg::CB], uint8_t *lds, void *C, const uint16_t *Other,
                                          const void *Bias, int M, int N, int m0, int mrows, int n0, int postop, int out_f32,
                                          int ksn, int sl, float *part, uint64_t *cnt) {
    constexpr int MB = Cfg::MB, CB = Cfg::CB, WK = Cfg::WK, CS = DUAL ? CB / 2 : CB;
    const int tid = threadIdx.x, lane = tid & 63, c = lane & 31, q = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kw = wave / Cfg::WM, wm = wave % Cfg::WM;
    auto rows_of = [&](int it, int &r, int &n) __attribute__((always_inline)) {
        // item `it` of a round: row block it / 256, register quad (it / 64) % 4, this lane
        r = 32 * (it >> 8) + 8 * ((it >> 6) & 3) + 4 * q;
        n = n0 + CS * c;
    };
    auto finish = [&](int r, int n, const float (*v)[4]) __attribute__((always_inline)) {
        if constexpr (DUAL) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (r + i < mrows && n < N) {
                    float x[CS];
#pragma unroll
                    for (int cb = 0; cb < CS; ++cb)
                        x[cb] = epi_apply_c<1>(v[CS + cb][i], dt2f<BF16>(f2dt<BF16>(v[cb][i])), 0.0f);
                    kw_store<CS, BF16, 0, false>(C, nullptr, nullptr, N, m0 + r + i, n, x);
                }
            return;
        }
        epi_dispatch(postop, out_f32, [&](auto P_, auto F_) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (r + i < mrows && n < N) {
                    float x[CS];
#pragma unroll
                    for (int cb = 0; cb < CS; ++cb) x[cb] = v[cb][i];
                    kw_store<CS, BF16, decltype(P_)::value, decltype(F_)::value>(C, Other, Bias, N, m0 + r + i, n, x);
                }
        });
    };
    float *red = (float *)lds;
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
    uint32_t *flag = (uint32_t *)lds;
    if (wave == 0) {
        const bool last = kw_arrive(cnt, ksn, lane);
        if (lane == 0) *flag = last;
    }
    __syncthreads();
    if (!*flag) return;  // (uniform)
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

}  // namespace
}  // namespace tcl
