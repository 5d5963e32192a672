// orkh_grouped.hip -- the tiled MFMA kernel of grouped-scale runs (many rows; int8 and uniform int4 weights).
//
// C[m][n] = sum over K-groups g ascending of ((float)P_g * aS[m][g]) * bS[g][n], P_g the group's exact int32 partial, each
// product and sum rounded (no fused multiply-add): the float sequence of the reference's grouped accumulate
// (src/npu/core/buf.c:501-520), bit for bit.
//
// k_tiled2g: one 8-wave workgroup per BM x BN tile; both operands HBM/L2 -> LDS with direct-to-LDS loads into a ring of
// stages of SU x 128 k (whole 128-byte lines of A, a stage's panel blocks of B), one barrier a stage, the next step's
// operands read into registers before the current step's MFMAs. Bound by the closing of groups on the VALU for small G
// (four float operations per output and group: at G=32 they are 16 per 16 x 16 x 32 MFMA, which takes 16 cycles against
// their 64), else by operand delivery: one CU's loads and LDS reads (M=64 and M=256 take the same time on 64 x 64, 64 and
// 256 of 256 CUs). Against the former kernel (16 waves, a masked MFMA per group and 128-k block, the tile's scales whole
// in LDS), us at K=N=4096: W4A4 M=256 G=32 57.2 -> 27.3, G=64 36.1 -> 16.3, G=128 15.4 -> 12.8, G=512 11.1 -> 10.5; int8
// M=256 G=32 46.0 -> 24.9, G=64 21.9 -> 16.3, G=128 18.3 -> 13.6, G=512 14.8 -> 12.4; M=2048 G=128 W4A4 95.0 -> 56.5
// (1.21 PFLOP/s), int8 85.1 -> 53.5. What the layout is for:
//  - MFMA steps hold SK consecutive k, SK dividing every group: 64 (v_mfma_i32_16x16x64_i8) where G % 64 == 0, else 32
//    (v_mfma_i32_16x16x32_i8). The steps' operands are picked from the stage's LDS image in k order (a lane's 16 or 8 k
//    of A are a chunk or half of one; of B, half or all of a lane's chunk of the panel block, or a dword of nibbles), so a
//    step never mixes groups and nothing is masked: one kernel for every group size;
//  - the scales of the groups that end in a stage ride in its ring slot (4-byte direct-to-LDS loads: rows of aS, columns of
//    bS), so their LDS use does not grow with K / G and no wait drains the ring;
//  - MFMA operands swapped (D = B^T A^T): a lane holds four columns of one row, so a group's close needs one aS value per
//    row block and one 16-byte read of bS per column block, and C goes out 16 bytes a store;
//  - where a group is a compile-time number of steps or whole stages (GS), its end is known without a test, and its first
//    step starts the accumulators from zero (W4A4 M=256 G=512, 64 x 64: 15.0 us with a test a step, 10.5 without). Where
//    the steps of a group do not divide a stage's the stage is compiled once for each place a group can stand in it (PH):
//    us, a run-time count of steps or stages, then this: W4A4 64 x 64 K=6144 N=2048 M=256 G=192 20.5 -> 15.5, G=384 18.5
//    -> 14.0, G=768 17.3 -> 13.2, K=N=3072 G=512 9.1 -> 8.7; int8 64 x 192 K=N=3072 M=768 G=192 22.0 -> 19.0, G=256 19.8
//    -> 18.6, K=2048 N=6144 M=384 G=512 13.5 -> 13.0. Groups of whole 128-k spans of any other count are tested once a
//    span (int8 64 x 64 K=6144 N=2048 M=256 G=384 19.6, tested each step, 17.4);
//  - a stage's loads go out between the MFMAs of the steps before it, not all after the barrier, where they stall the waves
//    while no MFMA runs (W4A4 M=256 G=128, 64 x 64: 14.3 -> 12.9); each load's kind is a compile-time one (15.7 to 15.1
//    at two-line stages);
//  - stage depth: a barrier and its refill cost about 0.2 us a stage on 64 x 64, so nibbles take four lines a stage where
//    the group's closes leave the registers (SK 64: 13.0 us at M=256 G=128 against 15.3 with two); int8 takes two (with
//    four the ring holds two stages only: 15.4 against 14.4).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>
#include <utility>

#include "orkh_dev.h"

namespace {

struct TG {
    int G;
    const float *aS, *bS; // [M][K/G], [K/G][N]
};

// GS: steps per group at compile time, where they divide a stage's or the ends recur after a few stages (launch_g), -1: whole
// stages per group, -2: whole 128-k spans per group, 0: any other count
constexpr int lcm_of(int a, int b) {
    int x = a;
    while (x % b) x += a;
    return x;
}
constexpr int ends_in(int gs, int t, int ph, int to) { // groups of gs steps that end in the first `to` of a stage's t steps, phase ph
    int n = 0;
    for (int i = 0; i < to; i++) n += (ph * t + i + 1) % gs == 0;
    return n;
}
constexpr int most_ends(int gs, int t) {
    int m = 0;
    for (int ph = 0; ph < lcm_of(gs, t) / t; ph++) m = ends_in(gs, t, ph, t) > m ? ends_in(gs, t, ph, t) : m;
    return m;
}
template <int KIND, int SK, int GS, int BM, int BN, int SU> struct TGP {
    static constexpr bool NIB = KIND == ORKH_I4U;
    static constexpr int NW = 8, WM = 2, WN = 4;
    static constexpr int MTW = BM / 16 / WM, NTW = BN / 16 / WN;
    static constexpr int T = SU * 128 / SK;                                        // MFMA steps per stage
    static constexpr bool RT = GS == 0 || GS == -2;                                // a run-time count of steps or spans
    static constexpr int PH = GS > 0 ? lcm_of(GS > 0 ? GS : 1, T) / T : 1;         // stages after which the ends recur
    static constexpr int NG = GS == -1 ? 1 : RT ? (SK == 32 ? 2 : 1) * SU : most_ends(GS > 0 ? GS : 1, T); // groups that can end in a stage
    static constexpr int BPS = (NIB ? 1 : 2) * SU;                                 // panel blocks per panel and stage
    // Direct-to-LDS loads per stage: 1 KiB of A (a line of 8 rows) or B (a panel block), 256 bytes of aS or bS; QA, QB, QS
    // per wave (so that a load's kind is known at compile time), those without work landing in a junk block
    static constexpr int NA = BM / 8 * SU, NB = BN / 16 * BPS, NSA = NG * BM / 64, NSB = NG * BN / 64;
    static constexpr int QA = NA / NW, QB = (NB + NW - 1) / NW, QS = (NSA + NSB + NW - 1) / NW, LPW = QA + QB + QS;
    static constexpr int SCA = (NA + NB) * 1024, SCB = SCA + NSA * 256; // byte offsets of the scales in a slot
    static constexpr int SLOT = SCB + NSB * 256, RMAX = (163840 - 1024) / SLOT, R = RMAX < 4 ? RMAX : 4;
    static constexpr int JUNK = R * SLOT, LDS = JUNK + 1024;
    static_assert(R >= 2 && MTW * WM * 16 == BM && NTW * WN * 16 == BN && T % 2 == 0 && QA * NW == NA && (R - 1) * LPW < 64 &&
                      (GS != -2 || SK == 64),
                  "tile");
};

template <int... T, class F> __device__ __forceinline__ void each(std::integer_sequence<int, T...>, F &&f) {
    (f(std::integral_constant<int, T>{}), ...);
}

template <int SK> struct Op { // an MFMA operand of SK k: 16 or 8 bytes a lane
    typedef typename std::conditional<SK == 64, v4i, long>::type t;
};
__device__ __forceinline__ v4i gmma(v4i a, v4i b, v4i c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ v4i gmma(long a, long b, v4i c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0); }

template <int KIND, int SK, int GS, int BM, int BN, int SU>
__global__ __launch_bounds__(512, 1) void k_tiled2g(orkh_mm p, TG gp, int mtiles, int ntiles) {
#pragma clang fp contract(off)
    using P = TGP<KIND, SK, GS, BM, BN, SU>;
    typedef typename Op<SK>::t op_t;
    typedef float v4f_t __attribute__((ext_vector_type(4)));
    typedef int v2i __attribute__((ext_vector_type(2)));
    constexpr int R = P::R, LPW = P::LPW, NW = P::NW;
    extern __shared__ char smb[];
    asm volatile("" ::"s"(p.M), "s"(p.K), "s"(p.N), "s"(p.KB), "s"(p.lda), "s"(p.A), "s"(p.B), "s"(p.C), "s"(p.ldc),
                 "s"(p.c_wt), "s"(mtiles), "s"(ntiles), "s"(gp.G), "s"(gp.aS), "s"(gp.bS));
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wv % P::WM, wn = wv / P::WM;
    // XCD-aware order, as k_big: each XCD's run of tiles covers up to 1024 rows, M fastest
    constexpr int GM = 1024 / BM;
    const int nT = mtiles * ntiles, per = nT / 8, rem = nT % 8, x = (int)blockIdx.x % 8, j = (int)blockIdx.x / 8;
    const int tl = x < rem ? x * (per + 1) + j : rem * (per + 1) + (x - rem) * per + j;
    int gt, in, tn, tm, gq, gr, Sk, krem;
    udivmod(tl, GM * ntiles, gt, in);
    const int gm = min(mtiles - gt * GM, GM);
    udivmod(in, gm, tn, tm);
    const int m0 = (gt * GM + tm) * BM, nb0 = tn * (BN / 16), NBt = p.N / 16;
    udivmod(SU * 128, gp.G, gq, gr); // groups per stage
    udivmod(p.K, gp.G, Sk, krem);
    const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A, (uint32_t)p.M * (uint32_t)p.lda);
    const __amdgpu_buffer_rsrc_t Br = make_rsrc(p.B, (uint32_t)NBt * p.KB * 1024u);
    const __amdgpu_buffer_rsrc_t Sa = make_rsrc(gp.aS, (uint32_t)p.M * Sk * 4u);
    const __amdgpu_buffer_rsrc_t Sb = make_rsrc(gp.bS, (uint32_t)Sk * p.N * 4u);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)smb;

    // this wave's loads: i = wv + q * NW of each kind
    uint32_t va[P::QA], vb[P::QB], vs[P::QS];
    const uint32_t ch = (uint32_t)(((lane & 7) ^ (lane >> 3) ^ (wv & 1)) * 16); // k_big's swizzle
#pragma unroll
    for (int q = 0; q < P::QA; q++) { // line i / (BM / 8) of rows 8 g8 .. 8 g8 + 7
        const int i = wv + q * NW, row = m0 + i % (BM / 8) * 8 + (lane >> 3);
        va[q] = row < p.M ? (uint32_t)row * (uint32_t)p.lda + (uint32_t)(i / (BM / 8)) * 128u + ch : OOB;
    }
#pragma unroll
    for (int q = 0; q < P::QB; q++) {
        const int i = wv + q * NW, nb = nb0 + i / P::BPS;
        vb[q] = i < P::NB && nb < NBt ? ((uint32_t)nb * p.KB + i % P::BPS) * 1024u + lane * 16u : OOB;
    }
#pragma unroll
    for (int q = 0; q < P::QS; q++) { // aS: 64 rows of a group; bS: 64 columns of a group
        const int i = wv + q * NW, is = i - P::NSA;
        const int row = m0 + i % (BM / 64) * 64 + lane, n = nb0 * 16 + is % (BN / 64) * 64 + lane;
        vs[q] = i < P::NSA ? (row < p.M ? (uint32_t)row * Sk * 4u : OOB) : is < P::NSB && n < p.N ? (uint32_t)n * 4u : OOB;
    }
    const int nst = (p.KB + P::BPS - 1) / P::BPS;
    int ist = 0, islot = 0, ig = 0, ir = 0; // the next stage to issue, its slot, the first group that ends in it, its start there
    // loads [q0, q1) of stage ist; past K and the last group, everything reads zeros
    auto issue = [&](auto q0, auto q1) {
        if (ist >= nst) return;
        const uint32_t slot = lds0 + (uint32_t)islot * P::SLOT, k0 = (uint32_t)ist * (SU * 128);
#pragma unroll
        for (int z = decltype(q0)::value; z < decltype(q1)::value; z++) {
            if (z < P::QA) {
                const int q = z, i = wv + q * NW;
                lds_dma16s(Ar, k0 + (uint32_t)(i / (BM / 8)) * 128u + ch < (uint32_t)p.K ? va[q] : OOB, k0, slot + i * 1024);
            } else if (z < P::QA + P::QB) {
                const int q = z - P::QA, i = wv + q * NW;
                lds_dma16s(Br, ist * P::BPS + i % P::BPS < p.KB ? vb[q] : OOB, (uint32_t)ist * (P::BPS * 1024),
                      i < P::NB ? slot + (P::NA + i) * 1024 : lds0 + P::JUNK);
            } else {
                const int q = z - P::QA - P::QB, i = wv + q * NW, is = i - P::NSA;
                const bool isa = i < P::NSA;
                const int g = ig + (isa ? i / (BM / 64) : is / (BN / 64));
                const bool ok = g < Sk;
                lds_dma4s(isa ? Sa : Sb, ok ? vs[q] : OOB, ok ? (uint32_t)g * (isa ? 4u : (uint32_t)p.N * 4u) : 0u,
                     i < P::NSA + P::NSB ? slot + P::SCA + i * 256 : lds0 + P::JUNK);
            }
        }
    };
    auto next = [&] { // stage ist is issued: on to the next one
        ist++;
        islot = islot + 1 == R ? 0 : islot + 1;
        ig += gq;
        ir += gr;
        if (ir >= gp.G) {
            ir -= gp.G;
            ig++;
        }
    };

    v4i acc[P::MTW][P::NTW];
    v4f_t c[P::MTW][P::NTW];
#pragma unroll
    for (int a = 0; a < P::MTW; a++)
#pragma unroll
        for (int b = 0; b < P::NTW; b++) {
            acc[a][b] = v4i{0, 0, 0, 0};
            c[a][b] = v4f_t{0.f, 0.f, 0.f, 0.f};
        }
    op_t a[2][P::MTW];
    typename std::conditional<P::NIB, typename std::conditional<SK == 64, v2i, int>::type, op_t>::type b[2][P::NTW];
    const int h = (lane >> 3) & 1, r7 = lane & 7, gl = lane >> 4, col = lane & 15;
    // operands of step t of the stage in a slot: lane group gl holds k [t SK + gl SK / 4, + SK / 4)
    auto rd = [&](int slot, int t, int d) {
        const char *sl = smb + slot * P::SLOT;
        const int k16 = SK == 64 ? t * 4 + gl : t * 2 + (gl >> 1), li = k16 >> 3; // 16-k chunk, line
        const int off = (li * (BM / 8) + h) * 1024 + r7 * 128 + (((k16 & 7) ^ r7 ^ h) * 16) + (SK == 64 ? 0 : (gl & 1) * 8);
#pragma unroll
        for (int i = 0; i < P::MTW; i++) a[d][i] = *(const op_t *)(sl + off + (wm * P::MTW + i) * 2048);
        const char *bl = sl + P::NA * 1024;
#pragma unroll
        for (int i = 0; i < P::NTW; i++) {
            const int panel = (wn * P::NTW + i) * P::BPS;
            if constexpr (!P::NIB) { // block t SK / 64, chunk of the lane's 16-k group
                if constexpr (SK == 64) b[d][i] = *(const op_t *)(bl + (panel + t) * 1024 + lane * 16);
                else b[d][i] = *(const op_t *)(bl + (panel + t / 2) * 1024 + (((t & 1) * 2 + (gl >> 1)) * 16 + col) * 16 + (gl & 1) * 8);
            } else { // nibbles: 8 bytes (16 k) or 4 (8 k) of the chunk of 32-k group
                const char *bb = bl + (panel + t * SK / 128) * 1024;
                if constexpr (SK == 64)
                    b[d][i] = *(const v2i *)(bb + (((t & 1) * 2 + (gl >> 1)) * 16 + col) * 16 + (gl & 1) * 8);
                else b[d][i] = *(const int *)(bb + ((t & 3) * 16 + col) * 16 + gl * 4);
            }
        }
    };
    auto opB = [&](auto raw) -> op_t {
        if constexpr (!P::NIB) return raw;
        else if constexpr (SK == 64) {
            const uint32_t u = raw.x, v = raw.y;
            return v4i{(int)((u << 4) & 0xf0f0f0f0u), (int)(u & 0xf0f0f0f0u), (int)((v << 4) & 0xf0f0f0f0u), (int)(v & 0xf0f0f0f0u)};
        } else {
            const uint32_t u = (uint32_t)raw;
            return (long)((uint64_t)((u << 4) & 0xf0f0f0f0u) | ((uint64_t)(u & 0xf0f0f0f0u) << 32));
        }
    };
    auto mm = [&](int d, auto fresh) { // fresh: the group's first step, from zero
        op_t bo[P::NTW];
#pragma unroll
        for (int jn = 0; jn < P::NTW; jn++) bo[jn] = opB(b[d][jn]);
#pragma unroll
        for (int i = 0; i < P::MTW; i++)
#pragma unroll
            for (int jn = 0; jn < P::NTW; jn++)
                acc[i][jn] = gmma(bo[jn], a[d][i], decltype(fresh)::value ? v4i{0, 0, 0, 0} : acc[i][jn]);
    };
    float sa[P::MTW];
    v4f_t sb[P::NTW];
    auto rdS = [&](int slot, int e) { // scales of the e-th group ending in the slot's stage
        const char *sl = smb + slot * P::SLOT;
#pragma unroll
        for (int i = 0; i < P::MTW; i++) sa[i] = *(const float *)(sl + P::SCA + (e * BM + (wm * P::MTW + i) * 16 + col) * 4);
#pragma unroll
        for (int jn = 0; jn < P::NTW; jn++)
            sb[jn] = *(const v4f_t *)(sl + P::SCB + (e * BN + (wn * P::NTW + jn) * 16 + gl * 4) * 4);
    };
    auto close = [&] {
#pragma unroll
        for (int i = 0; i < P::MTW; i++)
#pragma unroll
            for (int jn = 0; jn < P::NTW; jn++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float t = ((float)finish<KIND>(acc[i][jn][r]) * sa[i]) * sb[jn][r];
                    c[i][jn][r] = c[i][jn][r] + t;
                    if (GS <= 0) acc[i][jn][r] = 0;
                }
    };
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };

#pragma unroll 1
    for (int st = 0; st + 1 < R; st++) {
        issue(std::integral_constant<int, 0>{}, std::integral_constant<int, LPW>{});
        next();
    }
    if (nst >= R - 1) wait_vmcnt<(R - 2) * LPW>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    constexpr int GQ = GS == -1 ? SU * 128 : GS == -2 ? 128 : SK; // k of what cnt counts
    const int gsteps = gp.G / GQ;
    int cnt = 0; // of the running group done: steps (GS -1: stages, -2: spans)
    // Stage s + 1 has landed (this wave's share; the barrier covers the others'), and every wave's reads of stage s are done,
    // so its slot takes stage s + R
    auto turn = [&](int s) {
        if (s + R <= nst) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((R - 2) * LPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    rd(0, 0, 0);
    int rs = 0; // slot of stage s
    auto stage = [&](int s, auto phc) {
        constexpr int ph = decltype(phc)::value, GC = GS > 0 ? GS : 1;
        const int rn = rs + 1 == R ? 0 : rs + 1;
        int e = 0; // groups ended in this stage (run-time counts)
        auto at = [&](auto tc) {
            constexpr int t = decltype(tc)::value, TI = P::T - 1; // the next stage to issue goes out over the first TI steps
            constexpr bool place = (t + 1) * SK % GQ == 0;         // a group can end here
            const bool ends = GS > 0 ? (ph * P::T + t + 1) % GC == 0 : place && cnt + 1 == gsteps;
            // (a run-time count: within a stage the close reads them itself: a branch a place, not two)
            if (ends && (!P::RT || t == TI)) rdS(rs, GS > 0 ? ends_in(GC, P::T, ph, t) : GS == -1 ? 0 : e);
            if constexpr (t < TI) {
                rd(rs, t + 1, (t + 1) & 1);
            } else {
                turn(s);
                if (s + 1 < nst) rd(rn, 0, 0);
            }
            fence();
            if constexpr (GS > 0 && (ph * P::T + t) % GC == 0) mm(t & 1, std::true_type{});
            else mm(t & 1, std::false_type{});
            if constexpr (t < TI) issue(std::integral_constant<int, LPW * t / TI>{}, std::integral_constant<int, LPW *(t + 1) / TI>{});
            if constexpr (t == TI - 1) next();
            fence();
            if (ends) {
                if (P::RT && t < TI) rdS(rs, e);
                close();
                e++;
                cnt = 0;
            } else if (GS <= 0 && place) {
                cnt++;
            }
        };
        each(std::make_integer_sequence<int, P::T>{}, at);
        rs = rn;
    };
    for (int s = 0; s < nst; s += P::PH)
        each(std::make_integer_sequence<int, P::PH>{}, [&](auto phc) {
            if (decltype(phc)::value == 0 || s + decltype(phc)::value < nst) stage(s + decltype(phc)::value, phc);
        });

    const int n0 = (nb0 + wn * P::NTW) * 16 + gl * 4;
    const bool vec = p.ldc % 4 == 0 && ((uintptr_t)p.C & 15) == 0;
#pragma unroll
    for (int i = 0; i < P::MTW; i++) {
        const int m = m0 + (wm * P::MTW + i) * 16 + col;
        if (m >= p.M) continue;
        float *Cr = (float *)p.C + (size_t)m * p.ldc + n0;
#pragma unroll
        for (int jn = 0; jn < P::NTW; jn++) {
            if (nb0 + wn * P::NTW + jn >= NBt) continue;
            float *dst = Cr + jn * 16;
            if (vec) {
                if (p.c_wt) store_wt4(dst, __builtin_bit_cast(v4i, c[i][jn]));
                else *(v4f_t *)dst = c[i][jn];
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (p.c_wt) store_wt(&dst[r], c[i][jn][r]);
                    else dst[r] = c[i][jn][r];
                }
            }
        }
    }
}

template <int KIND, int SK, int GS, int BM, int BN, int SU>
int launch_t(const orkh_mm *p, const TG &gp, hipStream_t s) {
    using P = TGP<KIND, SK, GS, BM, BN, SU>;
    static lds_flags attr;
    auto kern = k_tiled2g<KIND, SK, GS, BM, BN, SU>;
    if (lds_limit((const void *)kern, P::LDS, attr)) return -1;
    const int mtiles = (p->M + BM - 1) / BM, ntiles = (p->N + BN - 1) / BN;
    if ((long)mtiles * ntiles >= (1L << 24) || p->K >= (1 << 24)) { // the kernel's divisions are exact below 2^24
        snprintf(g_lerr, sizeof g_lerr, "grouped tiled: %ld workgroups, K=%d", (long)mtiles * ntiles, p->K);
        return -2;
    }
    hipLaunchKernelGGL(kern, dim3(mtiles * ntiles), dim3(P::NW * 64), P::LDS, s, *p, gp, mtiles, ntiles);
    return 0;
}

// The form of the groups' ends
template <int KIND, int SK, int BM, int BN, int SU> int launch_g(const orkh_mm *p, const TG &gp, hipStream_t s) {
    if (gp.G == SK) return launch_t<KIND, SK, 1, BM, BN, SU>(p, gp, s);
    if constexpr (SK == 64) {
        if (gp.G == 128) return launch_t<KIND, SK, 2, BM, BN, SU>(p, gp, s);
        if constexpr (SU == 4 || (KIND == ORKH_I8 && BN == 192)) { // (the tiles that ran slower with run-time counts)
            if (gp.G == 192) return launch_t<KIND, SK, 3, BM, BN, SU>(p, gp, s);
            if (gp.G == 256) return launch_t<KIND, SK, 4, BM, BN, SU>(p, gp, s);
            if (gp.G == 384) return launch_t<KIND, SK, 6, BM, BN, SU>(p, gp, s);
            if (gp.G == 512) return launch_t<KIND, SK, 8, BM, BN, SU>(p, gp, s);
            if (gp.G == 768) return launch_t<KIND, SK, 12, BM, BN, SU>(p, gp, s);
        }
        if (gp.G % (SU * 128) == 0) return launch_t<KIND, SK, -1, BM, BN, SU>(p, gp, s);
        if constexpr (SU > 1)
            if (gp.G % 128 == 0) return launch_t<KIND, SK, -2, BM, BN, SU>(p, gp, s);
    }
    return launch_t<KIND, SK, 0, BM, BN, SU>(p, gp, s);
}

template <int KIND, int SK> int launch_k(const orkh_mm *p, const orkh_plan *q, const TG &gp, hipStream_t s) {
    constexpr bool L = SK == 64 && KIND == ORKH_I4U;
    if (q->bm == 64 && q->bn == 64) return launch_g<KIND, SK, 64, 64, L ? 4 : 2>(p, gp, s);
    if (q->bm == 64 && q->bn == 128) return launch_g<KIND, SK, 64, 128, 2>(p, gp, s);
    if (q->bm == 64 && q->bn == 192) return launch_g<KIND, SK, 64, 192, L ? 2 : 1>(p, gp, s);
    if (q->bm == 128 && q->bn == 128) return launch_g<KIND, SK, 128, 128, L ? 2 : 1>(p, gp, s);
    if constexpr (SK == 64) // (32-k steps: the closes of a stage spill, and the VALU bounds them on 128 x 128 too)
        if (q->bm == 128 && q->bn == 256) return launch_g<KIND, SK, 128, 256, 1>(p, gp, s);
    snprintf(g_lerr, sizeof g_lerr, "grouped tiled plan: %dx%d at G=%d unsupported", q->bm, q->bn, gp.G);
    return -2;
}

} // namespace

// The ORKH_ALGO_TILED2 launch of a grouped run (int8 and uniform int4; arguments checked by orkh_mm_launch_grouped)
extern "C" int orkh_tiled2g_launch(const orkh_mm *p, const orkh_plan *q, int G, const float *aS, const float *bS, void *stream) {
    const TG gp = {G, aS, bS};
    hipStream_t st = (hipStream_t)stream;
    if (G % 64 == 0) return p->kind == ORKH_I8 ? launch_k<ORKH_I8, 64>(p, q, gp, st) : launch_k<ORKH_I4U, 64>(p, q, gp, st);
    return p->kind == ORKH_I8 ? launch_k<ORKH_I8, 32>(p, q, gp, st) : launch_k<ORKH_I4U, 32>(p, q, gp, st);
}
