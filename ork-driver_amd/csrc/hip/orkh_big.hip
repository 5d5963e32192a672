// orkh_big.hip -- the tiled MFMA kernel for many rows (long prompts, batched prefill): 128- and 256-row tiles, every
// weight kind.
//
// k_big: one workgroup per BM x BN output tile. Like k_tiled2 (orkh_kernels.hip) it brings both operands HBM/L2 -> LDS
// with direct-to-LDS loads into a ring of stages and reads MFMA operands from there; what differs is what a large grid
// needs. Bound by operand delivery to the CUs (an L1's outstanding requests to L2 pass ~22-25 bytes per clock and CU),
// then by MFMA:
//  - tiles of up to 256 x 256, so that a byte delivered to a CU feeds up to 256 multiply-accumulates, in four shapes so
//    that a grid fills its last round of the CUs (256 x 192 takes K=2048 N=6144 M=4096 in two full rounds where
//    256 x 256 takes one and a half);
//  - stages of 128 activation bytes a row (whole cache lines, a_lds's swizzle) and one barrier per stage, with the
//    next phase's LDS operands read into registers before the current phase's MFMAs;
//  - load addresses as one per-lane offset plus a scalar stage offset, and each load's kind known at compile time, so a
//    load costs one instruction (us at M=K=N=4096 with a test of the kind per load: uniform int4 54.8, then 53.4, NF4 73.7,
//    then 70.4, fp16 117.5, then 116.4; fp16 K=N=4096 M=500 on 128 x 192 48.3, then 44.5);
//  - an XCD's run of tiles covers GM rows of tiles x several columns instead of one column of all rows, so its L2 takes
//    about a third less from the next level;
//  - the MFMA operands swapped (D = B^T A^T), so that a lane holds four consecutive columns of one row and C goes out
//    16 bytes a store;
//  - int4 blocks decoded in registers by 8 waves of 128 x 64 (two decodes per block), int8 and fp16 on 16 waves.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <type_traits>

#include "orkh_dev.h"

namespace {

template <int KIND, int BM, int BN> struct BG {
    using T = KT<KIND>;
    static constexpr bool NIB = KIND == ORKH_I4U || KIND == ORKH_NF4;
    static constexpr int NW = NIB ? 8 : 16, WM = NIB ? 2 : 4, WN = 4;
    static constexpr int MTW = BM / 16 / WM, NTW = BN / 16 / WN; // 16 x 16 blocks per wave
    static constexpr int MHN = MTW >= 4 ? 2 : 1, MH = MTW / MHN; // a phase: one K step x MH row blocks
    static constexpr int BPP = NIB ? 1 : 2;                      // panel blocks per panel and stage
    // fp32 sums per output: two on fp16's 128-row tiles, over the even and the odd 32-k blocks, as the smaller tiles they
    // replace have (relative error against fp64, one sum, two: K=2048 N=6144 M=1000 2.87e-7, 2.06e-7; K=8192 N=2048 M=2500
    // 5.74e-7, 4.07e-7; time +0.5%). The 256-row tiles have no registers for a second one (MTW * NTW * 8 of 128 a lane)
    static constexpr int CH = KIND == ORKH_F16 && BM == 128 ? 2 : 1;
    // 1 KiB loads per stage: 8 rows of A, or one block of B. QA and QB per wave (so that a load's kind is known at compile
    // time); a B load without work (QB * NW > NBL) lands in a junk block
    static constexpr int NA = BM / 8, NBL = BN / 16 * BPP;
    static constexpr int QA = NA / NW, QB = (NBL + NW - 1) / NW, LPW = QA + QB;
    static constexpr int SLOT = (NA + NBL + (QB * NW > NBL)) * 64; // 16-byte units
    static constexpr int RMAX = 163840 / (SLOT * 16), R = RMAX < 4 ? RMAX : 4;
    static constexpr int LDS = R * SLOT * 16;
    // Where the loads of a stage go out (us at K=N=4096, all at the barrier, then spread): between the MFMA phases of the stage
    // that runs R - 1 before it, where they do not hold the waves back while no MFMA runs: uniform int4 M=4096 256 x 256
    // 53.4 -> 52.3, M=1000 128 x 192 26.4 -> 24.2; NF4 M=4096 256 x 256 70.8 -> 67.3; int8 M=1000 128 x 256 29.3 -> 27.6; fp16
    // M=1000 128 x 256 51.6 -> 48.8. All at once after the barrier, R stages ahead, on two-slot rings (spread, a stage
    // would have less than a stage's time to arrive) and NF4's 128-row tiles (its decode fills the phases: 40.3 -> 41.0).
    static constexpr bool SPREAD = R >= 3 && !(KIND == ORKH_NF4 && BM == 128);
    static constexpr int RA = SPREAD ? R - 1 : R; // stages issued ahead
    static constexpr int GM = 1024 / BM; // tile rows of an XCD's run: 1024 rows
    static_assert(R >= 2 && MTW * WM * 16 == BM && NTW * WN * 16 == BN && MH * MHN == MTW && QA * NW == NA && NW % BPP == 0,
                  "tile");
};

// MFMA operand of K step kk from a lane's panel chunk (nibble kinds: half the chunk per step, as decode())
template <int KIND> __device__ __forceinline__ v4i step_op(v4i raw, int kk, const Lut &L) {
    const uint32_t x = kk ? raw.z : raw.x, y = kk ? raw.w : raw.y;
    if constexpr (KIND == ORKH_I4U) {
        return v4i{(int)((x << 4) & 0xf0f0f0f0u), (int)(x & 0xf0f0f0f0u), (int)((y << 4) & 0xf0f0f0f0u), (int)(y & 0xf0f0f0f0u)};
    } else {
        uint32_t a, b, c, d;
        nf4_map8(x, L, a, b);
        nf4_map8(y, L, c, d);
        return v4i{(int)a, (int)b, (int)c, (int)d};
    }
}

template <int KIND, int BM, int BN>
__device__ __forceinline__ void big_body(const orkh_mm &p, int mtiles, int ntiles, int bid) {
    using T = KT<KIND>;
    using P = BG<KIND, BM, BN>;
    typedef typename T::acc_t acc_t;
    typedef typename T::c_t c_t;
    constexpr int R = P::R, LPW = P::LPW, NW = P::NW, NA = P::NA;
    extern __shared__ v4i sm[];
    // every kernel argument in one batch of scalar loads behind one wait (as tiled2_body)
    asm volatile("" ::"s"(p.M), "s"(p.K), "s"(p.N), "s"(p.KB), "s"(p.lda), "s"(p.A), "s"(p.B), "s"(p.C), "s"(p.ldc),
                 "s"(p.c_wt), "s"(mtiles), "s"(ntiles));
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wv % P::WM, wn = wv / P::WM;
    // XCD-aware order: workgroup b runs on XCD b % 8, each XCD a contiguous run of tiles; runs go down GM tile rows at a
    // time, M fastest, so that a run is about as many rows of A as columns of B
    const int nT = mtiles * ntiles, per = nT / 8, rem = nT % 8, x = bid % 8, j = bid / 8;
    const int tl = x < rem ? x * (per + 1) + j : rem * (per + 1) + (x - rem) * per + j;
    int g, in, tn, tm;
    udivmod(tl, P::GM * ntiles, g, in);
    const int gm = min(mtiles - g * P::GM, P::GM);
    udivmod(in, gm, tn, tm);
    const int m0 = (g * P::GM + tm) * BM, nb0 = tn * (BN / 16), NBt = p.N / 16;
    const uint32_t lda_b = (uint32_t)p.lda * T::ESZ, kbytes = (uint32_t)p.K * T::ESZ;
    const __amdgpu_buffer_rsrc_t Ar = make_rsrc(p.A, (uint32_t)p.M * lda_b);
    const __amdgpu_buffer_rsrc_t Br = make_rsrc(p.B, (uint32_t)NBt * p.KB * 1024u);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)sm;
    const Lut L = {p.lut[0], p.lut[1], p.lut[2], p.lut[3]};

    // this wave's loads: A rows 8 i .. 8 i + 7, i = wv + q * NW (lane l: row l / 8, slot l % 8 holds chunk
    // slot ^ (l / 8) ^ (i & 1)), and panel blocks i = wv + q * NW
    uint32_t va[P::QA], vb[P::QB];
    const uint32_t ch = (uint32_t)(((lane & 7) ^ (lane >> 3) ^ (wv & 1)) * 16); // the chunk's byte in the stage row (NW is even)
#pragma unroll
    for (int q = 0; q < P::QA; q++) {
        const int row = m0 + (wv + q * NW) * 8 + (lane >> 3);
        va[q] = row < p.M ? (uint32_t)row * lda_b + ch : OOB;
    }
#pragma unroll
    for (int q = 0; q < P::QB; q++) {
        const int i = wv + q * NW, nb = nb0 + i / P::BPP;
        vb[q] = i < P::NBL && nb < NBt ? ((uint32_t)nb * p.KB + i % P::BPP) * 1024u + lane * 16u : OOB;
    }
    const int nst = (p.KB + P::BPP - 1) / P::BPP;
    int ist = 0, islot = 0; // the next stage to issue and its slot
    // part j of n of stage ist's loads, the last part going on to the next stage; straight-line: past K, A chunks and panel
    // blocks read zeros
    auto issue = [&](auto j, auto n) {
        constexpr int q0 = LPW * decltype(j)::value / decltype(n)::value, q1 = LPW * (decltype(j)::value + 1) / decltype(n)::value;
        if (ist >= nst) return;
        const uint32_t slot = lds0 + (uint32_t)islot * (P::SLOT * 16), sa = (uint32_t)ist * 128;
        const bool oka = sa + ch < kbytes, okb = ist * P::BPP + wv % P::BPP < p.KB;
#pragma unroll
        for (int z = q0; z < q1; z++) {
            const int q = z < P::QA ? z : z - P::QA;
            if (z < P::QA) lds_dma16s(Ar, oka ? va[q] : OOB, sa, slot + (wv + q * NW) * 1024);
            else lds_dma16s(Br, okb ? vb[q] : OOB, (uint32_t)ist * (P::BPP * 1024), slot + (NA + min(wv + q * NW, P::NBL)) * 1024);
        }
        if (q1 == LPW) {
            ist++;
            islot = islot + 1 == R ? 0 : islot + 1;
        }
    };
    auto part = [&](auto j) { // after the stage's j-th phase but the last
        if constexpr (P::SPREAD) issue(j, std::integral_constant<int, 2 * P::MHN - 1>{});
    };
    using J0 = std::integral_constant<int, 0>;
    using J1 = std::integral_constant<int, 1>;
    using J2 = std::integral_constant<int, 2>;

    acc_t acc[P::CH][P::MTW][P::NTW];
#pragma unroll
    for (int c = 0; c < P::CH; c++)
#pragma unroll
        for (int a = 0; a < P::MTW; a++)
#pragma unroll
            for (int b = 0; b < P::NTW; b++) acc[c][a][b] = acc_t{0, 0, 0, 0};
    // A operand of (row block mb, step kk): chunk c of row lane % 16, at (mb * 2 + h) * 64 + r7 * 8 + (c ^ r7 ^ h)
    const int h = (lane >> 3) & 1, r7 = lane & 7;
    const int c0 = P::NIB ? (lane >> 4) * 2 : lane >> 4, c1 = P::NIB ? c0 + 1 : c0 + 4;
    const int ao0 = h * 64 + r7 * 8 + (c0 ^ r7 ^ h), ao1 = h * 64 + r7 * 8 + (c1 ^ r7 ^ h);
    v4i a[2][P::MH], b[2][P::NTW], raw[P::NIB ? P::NTW : 1];
    auto rdA = [&](int slot, int kk, int hh, v4i (&d)[P::MH]) {
        const v4i *As = sm + slot * P::SLOT + (wm * P::MTW + hh * P::MH) * 128 + (kk ? ao1 : ao0);
#pragma unroll
        for (int i = 0; i < P::MH; i++) d[i] = As[i * 128];
    };
    auto rdB = [&](int slot, int kk) { // nibble kinds: the stage's chunks (kk = 0), decoded by opB
        const v4i *Bs = sm + slot * P::SLOT + NA * 64 + (wn * P::NTW * P::BPP + kk) * 64 + lane;
#pragma unroll
        for (int i = 0; i < P::NTW; i++) {
            if constexpr (P::NIB) raw[i] = Bs[i * 64];
            else b[kk][i] = Bs[i * 128];
        }
    };
    auto opB = [&](int kk) {
        if constexpr (P::NIB) {
#pragma unroll
            for (int i = 0; i < P::NTW; i++) b[kk][i] = step_op<KIND>(raw[i], kk, L);
        }
    };
    auto mm = [&](int kk, int hh) { // K step kk (its operands are in a[] and b[]) of row blocks hh * MH ..
        const int c = kk % P::CH;
#pragma unroll
        for (int i = 0; i < P::MH; i++)
#pragma unroll
            for (int jn = 0; jn < P::NTW; jn++)
                acc[c][hh * P::MH + i][jn] = mma(b[kk][jn], a[P::MHN == 2 ? hh : kk][i], acc[c][hh * P::MH + i][jn]);
    };
    // keeps each phase's LDS reads in front of its MFMAs
    auto fence = [] { __builtin_amdgcn_sched_barrier(0); };

#pragma unroll 1
    for (int st = 0; st < P::RA; st++) issue(J0{}, J1{});
    if (nst >= P::RA) wait_vmcnt<(P::RA - 1) * LPW>();
    else wait_vmcnt<0>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    rdB(0, 0);
    rdA(0, 0, 0, a[0]);
    opB(0);
    int rs = 0; // slot of stage s
    for (int s = 0; s < nst; s++) {
        const int rn = rs + 1 == R ? 0 : rs + 1;
        if constexpr (P::MHN == 2) {
            rdA(rs, 0, 1, a[1]);
            fence();
            mm(0, 0);
            part(J0{});
            fence();
            if constexpr (!P::NIB) rdB(rs, 1);
            rdA(rs, 1, 0, a[0]);
            opB(1);
            fence();
            mm(0, 1);
            part(J1{});
            fence();
            rdA(rs, 1, 1, a[1]);
            fence();
            mm(1, 0);
            part(J2{});
            fence();
        } else {
            if constexpr (!P::NIB) rdB(rs, 1);
            rdA(rs, 1, 0, a[1]);
            opB(1);
            fence();
            mm(0, 0);
            part(J0{});
            fence();
        }
        // Stage s + 1 has landed (this wave's share of it; the barrier covers the others'), and every wave's reads of
        // stage s are done, so its slot takes stage s + R (spread: while stage s + 1 runs)
        if (s + R <= nst) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"i"((R - 2) * LPW) : "memory");
        else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (!P::SPREAD) issue(J0{}, J1{});
        if (s + 1 < nst) {
            rdB(rn, 0);
            rdA(rn, 0, 0, a[0]);
        }
        fence();
        mm(1, P::MHN - 1);
        fence();
        opB(0); // (after the last stage: of what it holds, unused)
        rs = rn;
    }

    // a lane holds row lane % 16, columns 4 (lane / 16) .. + 3 of each block
    const int n0 = (nb0 + wn * P::NTW) * 16 + (lane >> 4) * 4;
    const bool vec = p.ldc % 4 == 0 && ((uintptr_t)p.C & 15) == 0;
#pragma unroll
    for (int i = 0; i < P::MTW; i++) {
        const int m = m0 + (wm * P::MTW + i) * 16 + (lane & 15);
        if (m >= p.M) continue;
        c_t *Cr = (c_t *)p.C + (size_t)m * p.ldc + n0;
#pragma unroll
        for (int jn = 0; jn < P::NTW; jn++) {
            if (nb0 + wn * P::NTW + jn >= NBt) continue;
            acc_t o = acc[0][i][jn];
            if constexpr (P::CH == 2) o += acc[1][i][jn];
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = finish<KIND>(o[r]);
            c_t *dst = Cr + jn * 16;
            if (vec) {
                if (p.c_wt) store_wt4(dst, __builtin_bit_cast(v4i, o));
                else *(acc_t *)dst = o;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    if (p.c_wt) store_wt(&dst[r], o[r]);
                    else dst[r] = o[r];
                }
            }
        }
    }
}

template <int KIND, int BM, int BN>
__global__ __launch_bounds__((BG<KIND, BM, BN>::NW * 64), 1) void k_big(orkh_mm p, int mtiles, int ntiles) {
    big_body<KIND, BM, BN>(p, mtiles, ntiles, (int)blockIdx.x);
}

// k_bigm: up to ORKH_TGROUP_MAX matmuls of one kind, M and K in one launch (the multi-matmul submit), as k_tiled2m: task
// t's tiles are workgroups [wg0[t], wg0[t] + tiles), each start a multiple of 8; the padding workgroups exit at once.
struct BigMulti {
    int n, mtiles;
    int wg0[ORKH_TGROUP_MAX], ntiles[ORKH_TGROUP_MAX];
    orkh_mm p[ORKH_TGROUP_MAX];
};
template <int KIND, int BM, int BN>
__global__ __launch_bounds__((BG<KIND, BM, BN>::NW * 64), 1) void k_bigm(BigMulti g) {
    int t = 0;
    while (t + 1 < g.n && (int)blockIdx.x >= g.wg0[t + 1]) t++;
    const int local = (int)blockIdx.x - g.wg0[t];
    if (local >= g.mtiles * g.ntiles[t]) return;
    big_body<KIND, BM, BN>(g.p[t], g.mtiles, g.ntiles[t], local);
}

template <int KIND, int BM, int BN> int launch(const orkh_mm *p, int n, const orkh_plan *q, hipStream_t s) {
    using P = BG<KIND, BM, BN>;
    static lds_flags attr[2];
    const int mtiles = (p->M + BM - 1) / BM;
    if (n == 1) {
        const int ntiles = (p->N + BN - 1) / BN;
        if ((long)mtiles * ntiles >= (1L << 24)) { // the kernel's tile-index division is exact below 2^24
            snprintf(g_lerr, sizeof g_lerr, "big: %ld workgroups", (long)mtiles * ntiles);
            return -2;
        }
        auto kern = k_big<KIND, BM, BN>;
        if (lds_limit((const void *)kern, P::LDS, attr[0])) return -1;
        orkh_mm pc = *p;
        pc.c_wt = q->cwt;
        hipLaunchKernelGGL(kern, dim3(mtiles * ntiles), dim3(P::NW * 64), P::LDS, s, pc, mtiles, ntiles);
        return 0;
    }
    BigMulti g;
    memset(&g, 0, sizeof g);
    g.n = n;
    g.mtiles = mtiles;
    long wg = 0;
    for (int t = 0; t < n; t++) {
        g.p[t] = p[t];
        g.p[t].c_wt = q->cwt;
        g.ntiles[t] = (p[t].N + BN - 1) / BN;
        g.wg0[t] = (int)wg;
        wg += ((long)mtiles * g.ntiles[t] + 7) / 8 * 8;
    }
    if (wg >= (1L << 24)) {
        snprintf(g_lerr, sizeof g_lerr, "big group: %ld workgroups", wg);
        return -2;
    }
    auto kern = k_bigm<KIND, BM, BN>;
    if (lds_limit((const void *)kern, P::LDS, attr[1])) return -1;
    hipLaunchKernelGGL(kern, dim3((unsigned)wg), dim3(P::NW * 64), P::LDS, s, g);
    return 0;
}

template <int KIND> int launch_kind(const orkh_mm *p, int n, const orkh_plan *q, hipStream_t s) {
    if (q->bm == 256 && q->bn == 256) return launch<KIND, 256, 256>(p, n, q, s);
    if (q->bm == 256 && q->bn == 192) return launch<KIND, 256, 192>(p, n, q, s);
    if (q->bm == 128 && q->bn == 256) return launch<KIND, 128, 256>(p, n, q, s);
    if (q->bm == 128 && q->bn == 192) return launch<KIND, 128, 192>(p, n, q, s);
    snprintf(g_lerr, sizeof g_lerr, "big plan: %dx%d unsupported", q->bm, q->bn);
    return -2;
}

} // namespace

// n = 1, or 2..ORKH_TGROUP_MAX matmuls of one kind, M and K (checked by the caller)
extern "C" int orkh_big_launch(const orkh_mm *p, int n, const orkh_plan *q, void *stream) {
    hipStream_t s = (hipStream_t)stream;
    if (q->ksplit > 1) {
        snprintf(g_lerr, sizeof g_lerr, "big plan: ksplit %d", q->ksplit);
        return -2;
    }
    switch (p->kind) {
    case ORKH_I8: return launch_kind<ORKH_I8>(p, n, q, s);
    case ORKH_I4U: return launch_kind<ORKH_I4U>(p, n, q, s);
    case ORKH_NF4: return launch_kind<ORKH_NF4>(p, n, q, s);
    case ORKH_F16: return launch_kind<ORKH_F16>(p, n, q, s);
    default: snprintf(g_lerr, sizeof g_lerr, "big plan: kind %d", p->kind); return -2;
    }
}
