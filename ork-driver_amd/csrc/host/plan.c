/* plan.c -- the MI355X matmul planner: which kernel, what grid, how K is split.
 *
 * Replaces the reference's K-split / N-tile / M-tile / core-count policy (orki_int8_ks, orki_budget,
 * orki_run_loop_chunk, the mg_max*64 M-tile: src/npu.c:131-160, :1598-1610, :1693-1694;
 * orki_f16_ks, src/npu/f16/regcmd.c:120-125). The NPU needed K cut into 1024-wide slices, N into
 * 8192-wide outputs and M into CBUF-sized row groups, each a separate submit with a host int32
 * accumulate. On MI355X every shape is one launch (plus a reduce pass when K is split across
 * workgroups); the planner only decides how to fill 256 CUs:
 *   M = 1    GEMV: half a 16-column panel per workgroup (whole panels where those already spread evenly over
 *            the CUs), waves split K in runs of ~8 KiB; K is split across workgroups only for long-K,
 *            few-panel shapes that leave the machine underfilled.
 *   M <= 64  the streaming kernel (same grid, runs of 1-4 KiB) or the LDS-ring tiled kernel, whichever a
 *            delivery model of both prices lower, each with its best K split.
 *   M >  64  the LDS-ring tiled kernel: the tile and K split with the least modelled time.
 *            Above 64 rows, large grids of every kind take the many-row kernel k_big instead (orki_plan_mm).
 *   NF4      (M > 1) the streaming kernel, k_tiled and the LDS-ring kernel, every tile and split, each priced by
 *            its own fit (nf4_best).
 * Both time models charge a workgroup for a fixed set-up, the operand bytes that must reach its CU and
 * its multiply-accumulates; a K split adds its partials' round trip and the reduce launch.
 * ORK_PLAN=stream|tiled, ORK_TILE=BMxBN (with ORK_PLAN=tiled: a k_tiled tile) and ORK_KSPLIT=n force a kernel,
 * tile or split (tests, A/B); they and
 * the other overrides below are read only on a context made with ORK_PLAN_DEBUG set (knob()), so a stray
 * variable cannot change the kernels of a production context. */
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

#include "internal.h"

static int cdiv(int a, int b) { return (a + b - 1) / b; }

/* A planner test override: the environment variable on a context made with ORK_PLAN_DEBUG, else nothing. */
static const char *knob(const ork_npu *c, const char *name) { return (c && c->plan_knobs) ? getenv(name) : NULL; }

/* A bytes per activation row per 1 KiB weight block (K-block of the panel layout) */
static int a_bytes_per_kb(int rkind) { return rkind == ORKH_F16 ? 64 : (rkind == ORKH_I8 ? 64 : 128); }
static int kpb_of(int rkind) { return rkind == ORKH_I8 ? 64 : rkind == ORKH_F16 ? 32 : 128; }

/* Streaming-kernel geometry for a K split of ks (1 = unsplit). Run length per wave: 8 KiB in flight per
 * wave for the int8/fp16 GEMV (M = 1); more waves with shorter runs where each block costs more issue
 * (more rows, int4 decode). Measured on the K=2048, N=6144 panels; the run lengths on either side were
 * within 2-4%. */
/* Paired panels for the streaming kernel: with more panels than CUs (but fewer than two per CU), one round of
 * cu workgroups, the first NB - cu owning two adjacent panels, balances the bytes per CU, and each wave loads
 * an A chunk once for both panels. Measured (K=2048 N=6144, us, single -> paired): int8 M=16 4.81 -> 4.43,
 * M=32 7.39 -> 5.60; fp16 M=16 8.17 -> 6.71; W4A8 M=16 4.25 -> 3.96, M=32 6.65 -> 4.85; M <= 8 no gain (M=2
 * 4.25 -> 4.43). The kernel holds up to two row tiles per panel. ORK_STREAM_NP=1 / 2 turns it off / on
 * wherever it applies (tests). */
static int stream_paired(const ork_npu *c, int M, int mt, int NB, int cu, int ks) {
    if (ks != 1 || mt > 2 || NB <= cu || NB >= 2 * cu || M < 2) return 0;
    const char *e = knob(c, "ORK_STREAM_NP");
    if (e) return atoi(e) == 2;
    return M > 8;
}

static void stream_geom(const ork_npu *c, int rkind, int M, int KB, int NB, int cu, int ks, orkh_plan *q) {
    const int kbw_target = (rkind == ORKH_I4U || rkind == ORKH_NF4) ? 2 : (M > 1 ? 4 : 8);
    const int need = cdiv(KB, kbw_target); /* waves per panel at the target run length */
    int wpg = need <= 4 ? 4 : 8;
    /* an int8 GEMV with fewer panels than CUs runs 8 shorter waves per panel: 2.94 -> 2.84 us at K=N=2048,
     * 2.80 -> 2.67 us at N=1024; with more panels than CUs 4 stay ahead (3.94 vs 4.04 us at N=6144) */
    if (M == 1 && rkind == ORKH_I8 && NB < cu) wpg = 8;
    const char *fw = knob(c, "ORK_WPG"); /* testing / A-B: waves per panel of the GEMV (4 or 8) */
    if (M == 1 && fw && (atoi(fw) == 4 || atoi(fw) == 8)) wpg = atoi(fw);
    if (ks > KB) ks = KB;
    if (ks < 1) ks = 1;
    const int kbs = cdiv(KB, ks);
    q->mt = cdiv(M, 16);
    q->wpg = wpg;
    q->kbs = kbs;
    q->kbw = cdiv(kbs, wpg);
    q->ksplit = cdiv(KB, kbs);
    q->np = stream_paired(c, M, q->mt, NB, cu, q->ksplit) ? 2 : 1;
    q->npg = q->np == 2 ? cu : NB;
}

/* The GEMV's split rule: split only when the panels leave the machine underfilled (< 4 waves per CU) AND
 * each wave would otherwise stream more than two runs back to back; the split costs a second launch
 * (the fixed-order reduce), which a one-run wave never repays. */
static int stream_rule_ks(const ork_npu *c, int rkind, int M, int KB, int NB, int cu) {
    orkh_plan g;
    stream_geom(c, rkind, M, KB, NB, cu, 1, &g);
    const int kbw_target = (rkind == ORKH_I4U || rkind == ORKH_NF4) ? 2 : (M > 1 ? 4 : 8);
    const int runs = cdiv(cdiv(KB, g.wpg), kbw_target);
    int ks = 1;
    if ((long)NB * g.wpg < 4L * cu && runs > 2) {
        ks = cdiv(4 * cu, NB * g.wpg);
        if (ks > runs) ks = runs; /* every wave keeps a full run */
    }
    return ks;
}

/* The GEMV's half-panel geometry (k_gemv_half: 8 columns per workgroup, so the bytes spread evenly over the CUs
 * whatever N/16 is): waves whose runs are about four load instructions (eight K-blocks; two instructions for
 * NF4, whose codebook decode is heavier), 2, 4 or 8 waves. Measured against whole panels (graph-timed, us):
 *   int8  K=2048 N=6144 3.95 -> 3.82; K=N=2048 2.77 -> 2.50; K=6144 N=2048 4.33 -> 3.77; K=8192 N=512 4.30 -> 3.39;
 *         K=2048 N=151936 (an LM head) 45.9 -> 44.6
 *   fp16  K=N=2048 3.52 -> 3.17
 *   W4A8  uniform K=2048 N=6144 3.14 -> 3.10, K=6144 N=2048 3.94 -> 3.15; NF4 K=2048 N=6144 3.58 -> 3.28,
 *         K=6144 N=2048 4.44 -> 3.35; W4A4 K=N=4096 3.60 -> 3.33
 * Where whole panels already spread evenly (N/16 x the K split a multiple of the CU count) they stay: K=2048
 * N=4096 int8 3.19 whole, 3.22 halves. ORK_GEMV_HALF=0/1 forces either and ORK_WPG=2/4/8 the waves (tests, A/B). */
static void gemv_half_geom(const ork_npu *c, int rkind, int NB, int cu, orkh_plan *q) {
    const char *e = knob(c, "ORK_GEMV_HALF");
    if (e && atoi(e) == 0) return;
    const long wgs = (long)NB * q->ksplit;
    if (!e && wgs >= cu && cdiv((int)(2 * wgs), cu) >= 2 * cdiv((int)wgs, cu)) return;
    const int blocks_per_wave = rkind == ORKH_NF4 ? 4 : 8;
    const int need = cdiv(q->kbs, blocks_per_wave);
    q->half = 1;
    q->wpg = need <= 2 ? 2 : need <= 4 ? 4 : 8;
    const char *fw = knob(c, "ORK_WPG");
    if (fw && (atoi(fw) == 2 || atoi(fw) == 4 || atoi(fw) == 8)) q->wpg = atoi(fw);
    q->kbw = cdiv(q->kbs, q->wpg);
}

int orki_gemv_panel_wpg(const ork_npu *c, int rkind, int KB, int NB) {
    orkh_plan g;
    memset(&g, 0, sizeof g);
    stream_geom(c, rkind, 1, KB, NB, (c && c->cores > 0) ? c->cores : 256, 1, &g);
    return g.wpg;
}

/* Time models (us) of the two MFMA kernels, for int8, fp16 and uniform int4 weights. A workgroup's time is
 * the sum of
 *   a fixed launch / drain cost and a cost per workgroup placed on the busiest CU ("per"),
 *   the operand bytes that must reach its CU (A rows, B blocks, C tile), per KiB: the ~15 B/clk per CU
 *   that L2 delivers, and (LDS-ring kernel) a further share that grows with the number of CUs pulling
 *   at once, and
 *   its multiply-accumulates at the kind's rate (per million MACs: int8 ~0.1 us, fp16 ~0.19 us, int4
 *   with decode ~0.2 us in the LDS-ring kernel -- the MFMA peaks; ~10x that in the streaming kernel,
 *   whose few waves per panel keep dependent MFMA chains);
 * with nothing overlapped between the three. A K split adds the reduce launch and the int32/fp32
 * partials written and read back. Least-squares fits to 588 timed launches (int8, fp16, W4A8, W4A4;
 * M = 16..4096, K = 2048..6144, N = 2048..22016; every tile and split on offer): 4% rms error for the
 * streaming kernel, 7% for the tiled one, and the pick within 1% of the fastest timed candidate. */
static double mac_rate(int rkind, int tiled) {
    if (rkind == ORKH_I8) return tiled ? 0.100 : 0.94;
    if (rkind == ORKH_F16) return tiled ? 0.187 : 1.90;
    if (rkind == ORKH_NF4) return tiled ? 0.40 : 0.91; /* tiled: with the per-stage decode into LDS (12% rms) */
    return tiled ? 0.199 : 0.91;
}

/* Half panels on the streaming kernel (8 columns per workgroup, twice the workgroups): each workgroup loads half
 * of its panel's B but all of its rows of A. Offered for int8 and fp16, whose panel bytes are a large share of a
 * workgroup's; priced by the same model with the halved B and C bytes. Measured against whole panels (graph-timed,
 * best split of each, us): fp16 K=N=2048 M=16 4.98 -> 4.41, M=8 4.18 -> 3.94; K=2048 N=768 M=16 4.74 -> 4.17; int8
 * K=N=2048 M=32 4.54 -> 4.13, K=6144 N=2048 M=16 6.74 -> 5.87, K=8192 N=1024 M=8 5.88 -> 5.21; where the halves
 * need a second round of the CUs they lose (int8 K=N=4096 M=16 5.55 -> 6.79). The uniform-int4 and NF4 nibbles are
 * a small share of a workgroup's bytes next to its int8 rows of A: half panels lost 2-8% below 32 rows and gained
 * 2-5% above, so they keep whole panels. Over 72 int8 / fp16 shapes (K x N = 2048 x 2048, 2048 x 768, 4096 x 4096,
 * 6144 x 2048, 8192 x 1024, 2048 x 6144; M = 2..64) the model's picks come within 3% of the fastest streaming
 * candidate of each. */
static int stream_half_offered(int rkind) { return rkind == ORKH_I8 || rkind == ORKH_F16; }

static double stream_us(const ork_npu *c, int rkind, int M, int N, int KB, int cu, int ks, int half) {
    orkh_plan g;
    stream_geom(c, rkind, M, KB, N / 16, cu, ks, &g);
    if (half && g.np == 2) return -1; /* paired and half panels exclude each other */
    const int pp = g.np == 2 ? 2 : 1; /* panels of the busiest workgroup */
    const long wgs = g.np == 2 ? g.npg : (long)(N / 16) * g.ksplit * (half ? 2 : 1);
    const double per = (double)((wgs + cu - 1) / cu);
    const double kib = ((double)M * a_bytes_per_kb(rkind) * g.kbs +
                        pp * ((half ? 512.0 : 1024.0) * g.kbs + (half ? 32.0 : 64.0) * M)) / 1024;
    const double mmac = (double)pp * g.mt * 16 * 16 * g.kbs * kpb_of(rkind) / 1e6;
    double t = 1.74 + per * (0.103 + 0.017 * kib + mac_rate(rkind, 0) * mmac);
    if (g.ksplit > 1) t += 2.81 + 0.327 * g.ksplit * (double)M * N * 4 / 1e6;
    return t;
}

/* NF4 above one row. Its codebook decode shifts each kernel's balance of operand delivery and VALU work differently
 * per tile, so every candidate has its own least-squares fit (relative error, non-negative terms) to graph-timed
 * launches on MI355X: 45 shapes (K x N = 2048 x 6144, 6144 x 2048, 4096 x 4096, 2048 x 2048, 2048 x 12288;
 * M = 32..1024), 1007 kernel / tile / split candidates in all (tests/golden/nf4_plan_sweep.json),
 *   t = a + rounds * (b + c * KiB) + [ks > 1] (d + e * ks * M * N * 4 / 1e6)   us,
 * KiB being the A and B bytes one workgroup loads (the streaming kernel: the form of stream_us). The fits are
 * within 4-7% rms per candidate; over the 45 shapes the picks total within 0.6% of the fastest timed candidate of
 * each. Refitted after the LDS-ring kernel's stage loads moved behind the first K-block of stage work (128 x 128
 * and 64 x 64 ran 2-7% faster) and with its 128 x 96 tile offered: the earlier fits, without it, totalled 2.2%
 * above the fastest on the same launches (K=4096 N=4096 M=384 24.1 us against 22.8 on 128 x 96, K=2048 N=6144
 * M=128 10.0 on k_tiled against 9.5 on the LDS ring's 64 x 64). */
static const struct nf4_fit {
    int algo, bm, bn, ksmax;
    double a, b, c, d, e;
} nf4_fits[] = {
    {ORKH_ALGO_TILED2, 128, 128, 4, 4.1310, 0.6805, 0.0272, 1.7563, 0.4771},
    {ORKH_ALGO_TILED2, 128, 96, 4, 2.4251, 2.0721, 0.0268, 2.2542, 0.5308},
    {ORKH_ALGO_TILED2, 64, 64, 4, 3.9420, 0.0000, 0.0287, 2.0167, 0.5399},
    {ORKH_ALGO_TILED2, 32, 64, 4, 1.0803, 2.1819, 0.0297, 2.6830, 0.3840},
    {ORKH_ALGO_TILED, 128, 128, 8, 5.3951, 3.6657, 0.0342, 2.9489, 0.4949},
    {ORKH_ALGO_TILED, 128, 96, 8, 3.8782, 3.9816, 0.0295, 2.9108, 0.4612},
    {ORKH_ALGO_TILED, 64, 64, 8, 3.5590, 1.4223, 0.0257, 2.7922, 0.4108},
};

static void nf4_best(const ork_npu *c, int M, int N, int KB, int cu, orkh_plan *q) {
    const int NB = N / 16;
    const double part = (double)M * N * 4 / 1e6; /* MB of one K slice's partials */
    double best = -1;
    for (int ks = 1; ks <= 8; ks *= 2) {
        const int kbs = cdiv(KB, ks);
        if (cdiv(KB, kbs) != ks || (ks > 1 && kbs < 2)) continue;
        if (M <= 64 && ks <= 4) { /* the streaming kernel holds up to 64 rows */
            orkh_plan g;
            memset(&g, 0, sizeof g);
            stream_geom(c, ORKH_NF4, M, KB, NB, cu, ks, &g);
            const int pp = g.np == 2 ? 2 : 1;
            const long wgs = g.np == 2 ? g.npg : (long)NB * g.ksplit;
            const double per = (double)((wgs + cu - 1) / cu);
            const double kib = ((double)M * 128 * g.kbs + pp * (1024.0 * g.kbs + 64.0 * M)) / 1024;
            const double mmac = (double)pp * g.mt * 16 * 16 * g.kbs * 128 / 1e6;
            double t = 2.0835 + per * (0.0241 * kib + 0.2942 * mmac);
            if (ks > 1) t += 2.0516 + 0.6116 * ks * part;
            if (best < 0 || t < best - 1e-9) {
                best = t;
                *q = g;
                q->algo = ORKH_ALGO_STREAM;
            }
        }
        for (size_t i = 0; i < sizeof nf4_fits / sizeof nf4_fits[0]; i++) {
            const struct nf4_fit *f = &nf4_fits[i];
            if (ks > f->ksmax) continue;
            const long wgs = (long)cdiv(M, f->bm) * cdiv(NB, f->bn / 16) * ks;
            const double rounds = (double)((wgs + cu - 1) / cu);
            const double kib = ((double)f->bm * 128 + (double)f->bn * 64) * kbs / 1024;
            double t = f->a + rounds * (f->b + f->c * kib);
            if (ks > 1) t += f->d + f->e * ks * part;
            if (best < 0 || t < best - 1e-9) {
                best = t;
                memset(q, 0, sizeof *q);
                q->algo = f->algo;
                q->bm = f->bm;
                q->bn = f->bn;
                q->ksplit = ks;
                q->kbs = kbs;
            }
        }
    }
}

/* int8, fp16 and uniform int4 above 64 rows: like NF4, every LDS-ring tile has its own least-squares fit (relative
 * error, non-negative terms) to graph-timed launches on MI355X, in the form of nf4_fits, KiB being the A and B bytes
 * one workgroup loads (tests/golden/mma_plan_sweep.json: every tile and K split of 1, 2 and 4 on offer at
 * K x N = 2048 x 6144, 2048 x 2048, 4096 x 4096, 6144 x 2048, 2048 x 12288 and M = 96..2048; the 32- and 16-row
 * tiles for one round of the CUs only). A tile is priced only where its rows are at most twice M, as timed. */
static const struct mma_fit {
    int rkind, bm, bn, ksmax; /* ksmax: the largest K split timed (and offered) */
    double a, b, c, d, e;
} mma_fits[] = { /* kind, tile, ksmax, a..e; then the launches fitted and the fit's rms relative error */
    {ORKH_I8, 256, 256, 4, 5.8440, 0.0000, 0.0241, 0.0000, 0.3994}, /* 16, 3.1% */
    {ORKH_I8, 128, 128, 4, 2.1719, 1.6437, 0.0156, 2.4427, 0.4431}, /* 82, 7.2% */
    {ORKH_I8, 128, 96, 4, 2.9512, 2.1169, 0.0143, 2.2673, 0.4083}, /* 75, 5.9% */
    {ORKH_I8, 64, 192, 4, 3.4918, 0.7902, 0.0145, 2.0294, 0.4527}, /* 74, 7.5% */
    {ORKH_I8, 64, 64, 4, 2.4453, 0.5219, 0.0160, 2.5433, 0.4340}, /* 79, 4.6% */
    {ORKH_I8, 32, 64, 2, 2.7092, 0.0000, 0.0223, 2.3342, 0.4118}, /* 14, 0.6% */
    {ORKH_I8, 32, 32, 1, 0.0000, 2.2276, 0.0188, 0.0000, 0.0000}, /* 4, 0.2% */
    {ORKH_I8, 16, 64, 1, 0.0000, 2.6950, 0.0192, 0.0000, 0.0000}, /* 4, 0.1% */
    {ORKH_F16, 256, 256, 4, 0.0880, 6.1768, 0.0227, 0.0000, 0.3771}, /* 38, 4.7% */
    {ORKH_F16, 128, 128, 4, 4.0377, 0.2295, 0.0161, 1.6667, 0.4677}, /* 92, 6.6% */
    {ORKH_F16, 128, 96, 4, 5.2807, 0.7426, 0.0150, 0.9779, 0.4447}, /* 91, 6.2% */
    {ORKH_F16, 64, 192, 4, 5.9856, 0.0000, 0.0145, 0.6252, 0.4682}, /* 89, 7.1% */
    {ORKH_F16, 64, 64, 4, 2.8047, 0.0000, 0.0180, 2.8555, 0.4211}, /* 92, 6.4% */
    {ORKH_F16, 32, 64, 2, 2.6572, 0.0000, 0.0223, 2.4686, 0.3812}, /* 13, 1.6% */
    {ORKH_F16, 32, 32, 1, 0.0000, 2.7401, 0.0175, 0.0000, 0.0000}, /* 4, 0.2% */
    {ORKH_F16, 16, 64, 1, 0.0000, 3.4902, 0.0175, 0.0000, 0.0000}, /* 4, 0.3% */
    {ORKH_I4U, 128, 128, 4, 2.1327, 1.8768, 0.0211, 2.5510, 0.4127}, /* 57, 5.8% */
    {ORKH_I4U, 128, 96, 4, 0.7882, 4.7886, 0.0180, 2.3200, 0.4005}, /* 46, 4.9% */
    {ORKH_I4U, 64, 192, 4, 0.1933, 4.9232, 0.0174, 2.4635, 0.3617}, /* 57, 5.8% */
    {ORKH_I4U, 64, 64, 4, 0.3768, 3.0260, 0.0137, 2.3979, 0.4614}, /* 60, 3.8% */
    {ORKH_I4U, 32, 64, 2, 0.0000, 2.8698, 0.0196, 2.1311, 0.5144}, /* 14, 0.5% */
    {ORKH_I4U, 32, 32, 1, 0.0000, 2.7500, 0.0158, 0.0000, 0.0000}, /* 4, 0.1% */
    {ORKH_I4U, 16, 64, 1, 0.0000, 3.0075, 0.0175, 0.0000, 0.0000}, /* 4, 0.1% */
};

static double mma_fit_best(int rkind, int M, int N, int KB, int cu, int ks_force, orkh_plan *q) {
    const int NB = N / 16;
    const double part = (double)M * N * 4 / 1e6;
    double best = -1;
    for (size_t i = 0; i < sizeof mma_fits / sizeof mma_fits[0]; i++) {
        const struct mma_fit *f = &mma_fits[i];
        if (f->rkind != rkind || f->bm > 2 * M) continue;
        for (int ks = 1; ks <= f->ksmax; ks *= 2) {
            if (ks_force > 0 && ks != ks_force) continue;
            const int kbs = cdiv(KB, ks);
            if (cdiv(KB, kbs) != ks || (ks > 1 && kbs < 4)) continue;
            const long wgs = (long)cdiv(M, f->bm) * cdiv(NB, f->bn / 16) * ks;
            if (f->bm <= 32 && wgs > cu) continue;
            const double rounds = (double)((wgs + cu - 1) / cu);
            const double kib = ((double)f->bm * a_bytes_per_kb(rkind) + (double)f->bn * 64) * kbs / 1024;
            double t = f->a + rounds * (f->b + f->c * kib);
            if (ks > 1) t += f->d + f->e * ks * part;
            if (best < 0 || t < best - 1e-9) {
                best = t;
                memset(q, 0, sizeof *q);
                q->algo = ORKH_ALGO_TILED2;
                q->bm = f->bm;
                q->bn = f->bn;
                q->ksplit = ks;
                q->kbs = kbs;
            }
        }
    }
    return best;
}

/* The LDS-ring kernel (k_tiled2): every tile and split on offer priced by the model above; A counts the
 * whole tile height, since rows past M still issue (zero-filled) loads. Returns the modelled time of
 * the best and fills q with it. */
static double tiled2_best(int rkind, int M, int N, int KB, int cu, int ks_force, int cfg_from, orkh_plan *q) {
    /* 32-row tiles split each stage's K-blocks over groups of waves; the model prices them unchanged (measured:
     * fp16 M=128 K=N=2048 32x32 9.0 us vs 9.04 modelled, W4A8 M=64 K=2048 N=6144 32x64 7.27 vs 7.28) */
    static const int cfg2[][2] = {{256, 256}, {128, 128}, {64, 192}, {64, 64}, {32, 64}, {32, 32}, {16, 64}, {16, 32}};
    const int NB = N / 16;
    const int abpk = a_bytes_per_kb(rkind), kpb = kpb_of(rkind);
    double best = -1;
    for (int i = cfg_from; i < (int)(sizeof cfg2 / sizeof cfg2[0]); i++) {
        const int bm = cfg2[i][0], bn = cfg2[i][1];
        /* NF4's decoded (int8) B doubles the LDS reads of the 3-panel wave tile: 22.3 us at M=512 vs 19.8 on
         * 128 x 128, which the model does not see; on 32-row tiles its per-block decode is shared by half the
         * rows the model assumes (not timed: not offered) */
        if (rkind == ORKH_NF4 && (bn == 192 || bm <= 32)) continue;
        const long tiles = (long)cdiv(M, bm) * cdiv(NB, bn / 16);
        for (int ks = ks_force > 0 ? ks_force : 1; ks <= (ks_force > 0 ? ks_force : 8); ks *= (ks_force > 0 ? 8 : 2)) {
            const int kbs = cdiv(KB, ks);
            if (ks_force <= 0 && (cdiv(KB, kbs) != ks || (ks > 1 && kbs < 4))) continue;
            const long wgs = tiles * ks;
            /* the model underprices several rounds of the K-group tiles (W4A8 M=256 K=2048 N=6144 32x64: 18.2 us
             * measured, 14.3 modelled; int8 M=128 N=6144 32x32: 16.4 vs 12.2), so they are offered for one round */
            if (bm <= 32 && wgs > cu) continue;
            /* nor split 8 ways: both such picks ran 24-30% above the model (fp16 K=6144 N=2048 M=16 16 x 64: 12.05 us
             * measured, 9.18 modelled; M=32 32 x 64: 12.03 against 32 x 32 split 4 ways at 11.56), where splits of
             * up to 4 sit at 0.93-0.98 of it */
            if (bm <= 32 && ks > 4) continue;
            const double per = (double)((wgs + cu - 1) / cu);
            const double busy = (double)(wgs < cu ? wgs : cu) / cu;
            const double kib = ((double)bm * abpk * kbs + (double)bn / 16 * 1024 * kbs + (double)bm * bn * 4) / 1024;
            const double mmac = (double)bm * bn * kbs * kpb / 1e6;
            double t = 4.09 + per * (0.35 + (0.0104 + 0.0058 * busy) * kib + mac_rate(rkind, 1) * mmac);
            if (ks > 1) t += 2.11 + 0.456 * ks * (double)M * N * 4 / 1e6;
            if (best < 0 || t < best - 1e-9) {
                best = t;
                q->algo = ORKH_ALGO_TILED2;
                q->bm = bm;
                q->bn = bn;
                q->ksplit = ks;
                q->kbs = kbs;
            }
        }
    }
    return best;
}

static int plan_core(const ork_npu *c, int rkind, int M, int K, int N, int KB, orkh_plan *q, size_t *ws_bytes);

/* Groups of waves that split a stage's K-blocks on a tile of the LDS-ring kernel, each with its own sums: k_tiled2's wave
 * grid (t2_xg, t2_wn: 2 x 4 on the uniform-int4 64 x 192 tile, 2 x 2 on its 64 x 64 tile) */
static int tiled2_kgroups(int rkind, int bm, int bn) {
    const int xg = (rkind == ORKH_I4U && bm == 64) ? (bn == 192 ? 1 : bn == 64 ? 2 : 0) : 0;
    const int nbt = bn / 16, mb = xg ? 2 : (bm / 16 < 4 ? bm / 16 : 4);
    const int nb = xg == 2 ? 2 : (nbt < 4 ? nbt : (nbt % 4 == 0 ? 4 : 2));
    return 16 / (mb * nb);
}

/* A-stage layout of the LDS-ring kernel: whole 128-byte row lines (swizzled LDS image; a stage row of 1, 2 or 4
 * lines) or MFMA fragment order. Measured on MI355X, graph-timed, both layouts alternated three times in one run,
 * exact (us, fragment -> line):
 *   one line a stage row:  int8 64x64 K=2048 N=6144 M=128 8.25 -> 7.95, M=256 13.44 -> 11.73, K=N=2048 M=128 7.87 ->
 *                          7.68, M=512 7.88 -> 7.83; int8 64x192 M=256 12.62 -> 11.95, M=512 13.09 -> 12.91; int8
 *                          32x64 M=96 10.90 -> 10.51; int8 128x96 M=512 14.64 -> 12.36; fp16 64x64 K=N=2048 M=128
 *                          12.64 -> 13.05, M=512 12.41 -> 13.18, K=2048 N=6144 M=128 13.83 -> 13.27, M=256 22.92 ->
 *                          20.12; fp16 32x64 M=96 K=N=2048 11.29 -> 11.48, M=256 11.19 -> 11.39; NF4 64x64 M=128
 *                          9.57 -> 9.68, M=256 14.26 -> 14.69
 *   2-4 lines a stage row: W4A4 K=N=4096 64x64 M=256 11.98 -> 10.07, 32x32 M=64 8.19 -> 6.83, 16x32 M=32 6.17 ->
 *                          5.64; W4A8 K=2048 N=6144 64x64 M=128 8.01 -> 7.33, 64x192 M=512 11.78 -> 11.57, 32x64
 *                          M=64 5.84 -> 5.90 (W4A4 M=128 7.91 -> 8.06, M=96 8.40 -> 8.10); NF4 32x64 M=64 6.98 ->
 *                          7.04, M=96 12.43 -> 12.57, 16x64 M=48 11.57 -> 11.65, 32x32 K=N=2048 M=64 5.69 -> 5.55;
 *                          NF4 128x96 M=256 14.29 -> 14.26, M=512 14.96 -> 14.92; int8 32x32 K=N=2048 M=128 5.68 ->
 *                          5.55, 16x32 M=32 5.56 -> 5.34; fp16 32x32 M=128 8.06 -> 7.64, 16x32 M=48 7.35 -> 6.87,
 *                          16x64 M=64 9.49 -> 9.21
 * so lines except: fp16 32x64, and fp16 64x64 unless N > 4096; the nibble kinds' 32x64 tile; NF4's 64x64, 128x96
 * (no gain) and 16-row tiles. ORK_ALINE=0/1 forces it (tests, A/B timing). */
static int aline_rule(const ork_npu *c, int rkind, const orkh_plan *q, int N) {
    /* the kernel has the line layout only where a stage row is whole 128-byte lines: K-blocks per stage as
     * k_tiled2's t2_ks (1 for int4 kinds, 1 for 256 x 256, else 2; at least the tile's K groups of waves) */
    const int wk = tiled2_kgroups(rkind, q->bm, q->bn);
    const int base = (rkind == ORKH_I4U || rkind == ORKH_NF4) ? 1 : (q->bm * q->bn >= 65536 ? 1 : 2);
    const int ks = base > wk ? base : wk;
    const int row_bytes = ks * a_bytes_per_kb(rkind);
    if (row_bytes % 128) return 0;
    const char *e = knob(c, "ORK_ALINE");
    if (e) return atoi(e) != 0;
    if (rkind == ORKH_F16) {
        if (q->bm == 32 && q->bn == 64) return 0;
        if (q->bm == 64 && q->bn == 64) return N > 4096;
    }
    if ((rkind == ORKH_I4U || rkind == ORKH_NF4) && q->bm == 32 && q->bn == 64) return 0;
    if (rkind == ORKH_NF4 && ((q->bm == 64 && q->bn == 64) || q->bm == 16 || (q->bm == 128 && q->bn == 96))) return 0;
    return 1;
}

int orki_plan(const ork_npu *c, int rkind, int M, int K, int N, int KB, orkh_plan *q, size_t *ws_bytes) {
    const int rc = plan_core(c, rkind, M, K, N, KB, q, ws_bytes);
    if (q->algo == ORKH_ALGO_TILED2) q->aline = aline_rule(c, rkind, q, N);
    /* The LDS-ring kernel's two-slot ring (two workgroups per CU, where the kernel has it for the tile) on grids of
     * more than one round of the CUs: one workgroup's set-up, first stage and epilogue overlap the other's loop.
     * Measured against the 4-slot ring (graph-timed, us; K=2048 N=6144 unless given): int8 64x192 M=768 22.95 ->
     * 18.87, M=1024 24.76 -> 21.78; int8 128x128 K=N=4096 M=2048 50.34 -> 45.79, K=N=2048 M=4096 31.6 -> 26.32;
     * fp16 64x192 M=768 41.16 -> 33.48, 128x128 K=N=2048 M=4096 54.95 -> 45.98; uniform int4 128x128 M=2048
     * 43.14 -> 33.87. On one round it loses (int8 64x192 M=512 13.38 -> 14.72, 128x128 K=N=4096 M=1024 25.41 ->
     * 29.11). ORK_RING=0/2 forces either (tests, A/B). */
    if (q->algo == ORKH_ALGO_TILED2) {
        const char *fr = knob(c, "ORK_RING");
        const int cu = (c && c->cores > 0) ? c->cores : 256;
        long wgs = (long)cdiv(M, q->bm) * cdiv(N / 16, q->bn / 16) * (q->ksplit > 1 ? q->ksplit : 1);
        /* uniform int4's 64 x 192 tile has no two-slot form (41 KiB stages): where its grid and 128 x 128's both
         * exceed one round, 128 x 128 with two slots (us, W4A8 K=2048: N=6144 M=768 21.74 -> 19.96, M=1024 22.61
         * -> 20.36; N=12288 M=512 22.43 -> 20.06, M=768 32.23 -> 29.71) */
        const long w128 = (long)cdiv(M, 128) * cdiv(N / 16, 8);
        if (rkind == ORKH_I4U && !fr && !knob(c, "ORK_TILE") && q->bm == 64 && q->bn == 192 && q->ksplit <= 1 &&
            wgs > cu && w128 > cu && orkh_tiled2_ring2_ok(rkind, 128, 128)) {
            q->bm = q->bn = 128;
            q->aline = aline_rule(c, rkind, q, N);
            wgs = w128;
        }
        if (fr) q->ring = atoi(fr) == 2 ? 2 : 0;
        else if (wgs > cu && orkh_tiled2_ring2_ok(rkind, q->bm, q->bn)) q->ring = 2;
        /* C stored write-through (device scope) where the grid is one round of the CUs: every workgroup stores at
         * about the same time, after all the loads, and the L2s pass C on to memory as it comes instead of holding
         * up to 64 MB of it dirty for the end of the kernel. Graph-timed against write-back stores (us): int8 K=2048
         * N=6144 M=512 64 x 192 14.56 -> 13.45, M=256 12.89 -> 12.52; uniform int4 M=512 64 x 192 13.96 -> 12.60;
         * W4A4 K=N=4096 M=256 64 x 64 12.55 -> 12.21; fp16 K=N=2048 M=512 64 x 64 13.00 -> 12.65; int8 M=K=N=4096
         * 256 x 256 67.72 -> 66.35; int8 K=N=2048 M=128 32 x 32 5.66 -> 5.57; W4A8 M=64 32 x 64 6.25 -> 6.06. On
         * grids of several rounds the early writes compete with the later workgroups' loads: int8 M=1024 two-slot
         * 23.37 -> 25.80, fp16 M=768 32.84 -> 36.11. ORK_CWT=0/1 forces either. */
        const char *fc = knob(c, "ORK_CWT");
        q->cwt = fc ? atoi(fc) != 0 : wgs <= cu;
    }
    return rc;
}

static int plan_core(const ork_npu *c, int rkind, int M, int K, int N, int KB, orkh_plan *q, size_t *ws_bytes) {
    (void)K;
    memset(q, 0, sizeof *q);
    *ws_bytes = 0;
    const int cu = (c && c->cores > 0) ? c->cores : 256;
    const int NB = N / 16;
    const char *force = knob(c, "ORK_PLAN");
    const int f_stream = force && !strcmp(force, "stream"), f_tiled = force && !strcmp(force, "tiled");
    const char *fks = knob(c, "ORK_KSPLIT");
    int ks_force = fks ? atoi(fks) : 0;
    if (ks_force > KB) ks_force = KB;
    if (ks_force > 0) ks_force = cdiv(KB, cdiv(KB, ks_force)); /* as a split can realise it */

    const char *tf = knob(c, "ORK_TILE"); /* "BMxBN": that tile of the LDS-ring kernel (of k_tiled with ORK_PLAN=tiled) */
    int fbm, fbn;
    if (tf && sscanf(tf, "%dx%d", &fbm, &fbn) == 2) {
        const int ks = ks_force > 0 ? ks_force : 1;
        q->algo = f_tiled ? ORKH_ALGO_TILED : ORKH_ALGO_TILED2;
        q->bm = fbm;
        q->bn = fbn;
        q->kbs = cdiv(KB, ks);
        q->ksplit = cdiv(KB, q->kbs);
        if (q->ksplit > 1) *ws_bytes = (size_t)q->ksplit * M * N * 4;
        return 0;
    }

    if (rkind == ORKH_NF4 && M > 1 && !f_stream && !f_tiled && ks_force <= 0) {
        nf4_best(c, M, N, KB, cu, q);
        if (q->ksplit > 1) *ws_bytes = (size_t)q->ksplit * M * N * 4;
        return 0;
    }

    if (M <= 64 && !f_tiled) {
        int ks, half = 0;
        if (M == 1 || f_stream || ks_force > 0 || rkind == ORKH_NF4) {
            ks = ks_force > 0 ? ks_force : stream_rule_ks(c, rkind, M, KB, NB, cu);
        } else {
            /* both kernels priced, each at its best split (the streaming kernel also with half panels); the
             * streaming kernel wins ties */
            ks = 1;
            double ts = stream_us(c, rkind, M, N, KB, cu, 1, 0);
            for (int k = 1; k <= 8; k *= 2) {
                if (k > 1 && (cdiv(KB, cdiv(KB, k)) != k || cdiv(KB, k) < 4)) continue;
                for (int h = k == 1 ? 1 : 0; h <= stream_half_offered(rkind); h++) {
                    const double t = stream_us(c, rkind, M, N, KB, cu, k, h);
                    if (t >= 0 && t < ts - 1e-9) { ts = t; ks = k; half = h; }
                }
            }
            orkh_plan t2;
            memset(&t2, 0, sizeof t2);
            if (tiled2_best(rkind, M, N, KB, cu, 0, rkind == ORKH_I4U, &t2) < ts - 1e-9) {
                *q = t2;
                if (q->ksplit > 1) *ws_bytes = (size_t)q->ksplit * M * N * 4;
                return 0;
            }
        }
        /* M = 1 takes the VALU-dot GEMV (same grid and fields); ORK_PLAN=stream keeps the MFMA kernel. */
        q->algo = (M == 1 && !f_stream) ? ORKH_ALGO_GEMV : ORKH_ALGO_STREAM;
        stream_geom(c, rkind, M, KB, NB, cu, ks, q);
        if (q->algo == ORKH_ALGO_GEMV) gemv_half_geom(c, rkind, NB, cu, q);
        if (q->algo == ORKH_ALGO_STREAM) q->half = half && q->np == 1;
        const char *fh = knob(c, "ORK_STREAM_HALF"); /* testing / A-B: half panels on or off on the streaming kernel */
        if (q->algo == ORKH_ALGO_STREAM && q->np == 1 && fh) q->half = atoi(fh) != 0;
        if (q->ksplit > 1) *ws_bytes = (size_t)q->ksplit * M * N * 4;
        return 0;
    }

    /* (NF4 reaches here only with ORK_KSPLIT forced: k_tiled up to 128 rows, the LDS-ring kernel above) */
    if ((rkind != ORKH_NF4 || M > 128) && !f_tiled) {
        /* int8, fp16 and uniform int4: the per-tile fits (uniform int4 has no 256 x 256 fit: with the nibble decode
         * its registers spill, 20 B per lane); a forced split they were not timed at takes the shared model */
        if (rkind == ORKH_NF4 || mma_fit_best(rkind, M, N, KB, cu, ks_force, q) < 0)
            tiled2_best(rkind, M, N, KB, cu, ks_force, rkind == ORKH_I4U, q);
        if (q->ksplit > 1) *ws_bytes = (size_t)q->ksplit * M * N * 4;
        return 0;
    }

    /* k_tiled (NF4 up to 128 rows, or ORK_PLAN=tiled): each CU pulls its tiles' A and B rows through L2 at a roughly fixed
     * rate, so the time of a round of workgroups is about the operand bytes one workgroup loads. K is split
     * across workgroups when that cuts the per-workgroup bytes by more than the partial sums and the extra
     * reduce launch (~2 us) cost. Model units: us at ~48 KB/us per CU (measured order of magnitude),
     * 5 TB/s for the partials' HBM round trip. */
    static const int cfg[][2] = {{128, 96}, {128, 128}, {64, 64}};
    const int bpk = 64;                                                  /* B bytes per column per K-block, every kind */
    const int apk = (rkind == ORKH_I4U || rkind == ORKH_NF4) ? 128 : 64; /* A bytes per row per K-block */
    double best = -1;
    for (int i = 0; i < 3; i++) {
        const int bm = cfg[i][0], bn = cfg[i][1];
        const long tiles = (long)cdiv(M, bm) * cdiv(NB, bn / 16);
        for (int ks = ks_force > 0 ? ks_force : 1; ks <= (ks_force > 0 ? ks_force : 8); ks++) {
            const int kbs = cdiv(KB, ks);
            if (ks_force <= 0 && (cdiv(KB, kbs) != ks || (ks > 1 && kbs < 4))) continue;
            const long wgs = tiles * ks;
            const long rounds = (wgs + cu - 1) / cu;
            double t = rounds * (double)(bm * apk + bn * bpk) * kbs / 48e3;
            if (ks > 1) t += 2.0 + 2.0 * ks * (double)M * N * 4 / 5e6;
            if (best < 0 || t < best - 1e-9) {
                best = t;
                q->bm = bm;
                q->bn = bn;
                q->ksplit = ks;
                q->kbs = kbs;
            }
        }
    }
    q->algo = ORKH_ALGO_TILED;
    if (q->ksplit > 1) *ws_bytes = (size_t)q->ksplit * M * N * 4;
    return 0;
}

/* When a run takes the many-row kernel (k_big, ../hip/orkh_big.hip) instead of orki_plan's pick.
 * Above 64 rows both are priced, us, and the cheaper one runs:
 *   k_big, per tile     a + rounds * (b + c * KiB) + e * MB        (rounds of the CUs; KiB: the A and B bytes a workgroup
 *                                                                  loads; MB: C's megabytes, which the end of a round
 *                                                                  writes with nothing to overlap)
 *   orki_plan's pick    a + rounds * (b[tile] + c[tile] * KiB) + e * MB + [ks > 1] (d + f * ks * MB)
 *                                                                  (e: e1 on one round, else e2)
 * Each is a least-squares fit in relative error (non-negative terms) to launches timed on MI355X, every k_big tile and
 * orki_plan's pick at 31 (K, N) with K from 256 to 8192 and N from 512 to 16384 and row counts from 65 to 4096, per weight
 * kind (633 shapes a kind, tests/golden/big_plan_sweep.json); 3-8% rms. Total us over them, former picks, this rule, the
 * faster of the two everywhere: int8 12105, 11260, 11242; fp16 20187, 18886, 18819; uniform int4 11630, 10031, 10013; NF4
 * 15668, 13623, 13616. No shape runs 4% slower than its former pick (256 x 256: 11%). Fits without the costs per launch and
 * round, made from K = 2048 up, took tiles at K = 256 and 512 that ran up to 42% slower: fp16 K=256 N=6144 M=2689 33.4 us on
 * 256 x 256, 23.5 on 128 x 128. On 876 more shapes at 20 random (K, N), K from 160 to 7360: 12,126 us by the former picks,
 * 11,015 by this rule, 10,909 the faster of the two everywhere; the worst 4.7% slower than its pick (int8 K=288 N=1920
 * M=3442 9.23 -> 9.66). What the prices do not see is a memory-bound C: at K=896 N=9728, the worst timed, one tile or the
 * other is up to 14% ahead of the price's choice (int8 M=4096 62.7 -> 69.5 us, uniform int4 61.0 on k_big, 69.6 kept).
 * The margin keeps a pick whose price is that close. Some shapes, us: int8 K=N=4096 M=4096 65.0 -> 61.3, K=6144 N=2048
 * M=4096 63.3 -> 49.3; fp16 K=2048 N=6144 M=4096 140.6 -> 114.3; uniform int4 K=N=4096 M=4096 89.8 -> 52.3; NF4 112.0 ->
 * 67.3, K=2048 N=6144 M=1000 29.5 -> 24.2. At 512 rows and fewer the smaller tiles fill the CUs better and keep the run
 * (int8 K=2048 N=6144 M=500 11.9 against 16.6), except where N is large (N=12288 20.3 -> 17.6).
 * fp16: a tile is offered only where it keeps as many fp32 sums an output as the pick it would replace (the pick's K groups
 * of waves times its K split), each over that share of K: with one sum over all of K in place of two the error against
 * fp64 was 1.39 to 1.41 times the pick's (K=2048..8192); with two it is the pick's. k_big has two on its
 * 128-row tiles, one on the 256-row ones.
 * A context's planner overrides (ORK_PLAN, ORK_TILE and the others of orki_plan) turn the rule off, and ORK_PLAN=big with
 * ORK_TILE=BMxBN forces a k_big tile (ORK_CWT=0/1: its store policy). */
static const struct big_fit {
    int rkind, bm, bn;
    double a, b, c, e;
} big_fits[] = {
    {ORKH_I8, 256, 256, 0.0000, 5.8445, 0.0207, 0.1215},  {ORKH_I8, 256, 192, 0.0000, 5.0543, 0.0211, 0.1120},
    {ORKH_I8, 128, 256, 0.0000, 4.8374, 0.0161, 0.0988},  {ORKH_I8, 128, 192, 0.0841, 4.6869, 0.0167, 0.0681},
    {ORKH_F16, 256, 256, 0.0000, 5.1371, 0.0213, 0.1476}, {ORKH_F16, 256, 192, 0.0000, 4.6484, 0.0215, 0.1365},
    {ORKH_F16, 128, 256, 0.0000, 4.4193, 0.0163, 0.1458}, {ORKH_F16, 128, 192, 0.0000, 4.2182, 0.0171, 0.1170},
    {ORKH_I4U, 256, 256, 0.0000, 8.8331, 0.0253, 0.0537}, {ORKH_I4U, 256, 192, 0.6961, 4.8054, 0.0228, 0.1019},
    {ORKH_I4U, 128, 256, 0.0906, 5.3810, 0.0244, 0.0544}, {ORKH_I4U, 128, 192, 0.6025, 4.2765, 0.0214, 0.0620},
    {ORKH_NF4, 256, 256, 0.0000, 9.5851, 0.0337, 0.0481}, {ORKH_NF4, 256, 192, 0.7750, 5.3310, 0.0317, 0.0906},
    {ORKH_NF4, 128, 256, 0.3416, 5.4280, 0.0434, 0.0472}, {ORKH_NF4, 128, 192, 0.5835, 4.4760, 0.0394, 0.0468},
};
#define BIG_F16_SUMS(bm) ((bm) == 128 ? 2 : 1) /* BG::CH of the kernel */
static const struct pick_fit {
    int rkind;
    double margin, a, e1, e2, d, f;
} pick_fits[] = {
    {ORKH_I8, 0.99, 2.2018, 0.1412, 0.1751, 2.8660, 0.3011},
    {ORKH_F16, 0.96, 1.8442, 0.1792, 0.1781, 2.8651, 0.3646},
    {ORKH_I4U, 0.97, 2.4471, 0.0620, 0.1151, 1.8313, 0.4186},
    {ORKH_NF4, 0.99, 2.1421, 0.0546, 0.1092, 2.3528, 0.3783},
};
static const struct pick_rate { /* b and c of a tile; bm 0: a tile that no timed shape picked, at the kind's lowest rate */
    int rkind, algo, bm, bn, ring;
    double b, c;
} pick_rates[] = {
    {ORKH_I8, ORKH_ALGO_TILED2, 16, 64, 0, 0.0000, 0.0286},   {ORKH_I8, ORKH_ALGO_TILED2, 32, 32, 0, 0.4549, 0.0149},
    {ORKH_I8, ORKH_ALGO_TILED2, 32, 64, 0, 0.6428, 0.0206},   {ORKH_I8, ORKH_ALGO_TILED2, 64, 64, 0, 0.2054, 0.0161},
    {ORKH_I8, ORKH_ALGO_TILED2, 64, 192, 0, 0.3891, 0.0162},  {ORKH_I8, ORKH_ALGO_TILED2, 64, 192, 2, 0.0155, 0.0156},
    {ORKH_I8, ORKH_ALGO_TILED2, 128, 96, 0, 1.9867, 0.0143},  {ORKH_I8, ORKH_ALGO_TILED2, 128, 96, 2, 2.8802, 0.0133},
    {ORKH_I8, ORKH_ALGO_TILED2, 128, 128, 0, 0.2091, 0.0169}, {ORKH_I8, ORKH_ALGO_TILED2, 128, 128, 2, 0.0000, 0.0176},
    {ORKH_I8, 0, 0, 0, 0, 0.0000, 0.0133},
    {ORKH_F16, ORKH_ALGO_TILED2, 16, 64, 0, 0.0000, 0.0237},   {ORKH_F16, ORKH_ALGO_TILED2, 32, 32, 0, 0.7276, 0.0150},
    {ORKH_F16, ORKH_ALGO_TILED2, 32, 64, 0, 0.8455, 0.0198},   {ORKH_F16, ORKH_ALGO_TILED2, 64, 64, 0, 0.4332, 0.0171},
    {ORKH_F16, ORKH_ALGO_TILED2, 64, 192, 0, 1.2045, 0.0164},  {ORKH_F16, ORKH_ALGO_TILED2, 64, 192, 2, 0.2182, 0.0170},
    {ORKH_F16, ORKH_ALGO_TILED2, 128, 96, 0, 1.6126, 0.0156},  {ORKH_F16, ORKH_ALGO_TILED2, 128, 96, 2, 0.6610, 0.0157},
    {ORKH_F16, ORKH_ALGO_TILED2, 128, 128, 0, 0.0000, 0.0173}, {ORKH_F16, ORKH_ALGO_TILED2, 128, 128, 2, 0.0000, 0.0184},
    {ORKH_F16, 0, 0, 0, 0, 0.0000, 0.0150},
    {ORKH_I4U, ORKH_ALGO_TILED2, 16, 64, 0, 0.0000, 0.0324},   {ORKH_I4U, ORKH_ALGO_TILED2, 32, 32, 0, 0.5442, 0.0121},
    {ORKH_I4U, ORKH_ALGO_TILED2, 32, 64, 0, 0.5358, 0.0181},   {ORKH_I4U, ORKH_ALGO_TILED2, 64, 64, 0, 1.0193, 0.0132},
    {ORKH_I4U, ORKH_ALGO_TILED2, 64, 192, 0, 1.9941, 0.0175},  {ORKH_I4U, ORKH_ALGO_TILED2, 128, 96, 0, 2.3002, 0.0201},
    {ORKH_I4U, ORKH_ALGO_TILED2, 128, 128, 0, 0.8814, 0.0220}, {ORKH_I4U, ORKH_ALGO_TILED2, 128, 128, 2, 0.5425, 0.0210},
    {ORKH_I4U, 0, 0, 0, 0, 0.0000, 0.0121},
    {ORKH_NF4, ORKH_ALGO_TILED, 64, 64, 0, 3.8499, 0.0248},    {ORKH_NF4, ORKH_ALGO_TILED2, 32, 64, 0, 0.7575, 0.0299},
    {ORKH_NF4, ORKH_ALGO_TILED2, 64, 64, 0, 0.5283, 0.0328},   {ORKH_NF4, ORKH_ALGO_TILED2, 128, 96, 0, 2.7709, 0.0275},
    {ORKH_NF4, ORKH_ALGO_TILED2, 128, 128, 0, 1.8063, 0.0284}, {ORKH_NF4, 0, 0, 0, 0, 0.0000, 0.0248},
};

/* A and B KiB that one workgroup of a bm x bn tile loads over kbs K-blocks */
static double tile_kib(int rkind, int bm, int bn, int kbs) {
    return ((double)bm * a_bytes_per_kb(rkind) + bn * 64.0) * kbs / 1024;
}

/* Price of orki_plan's pick q over its wgs workgroups, times the kind's margin; mb: C's megabytes. From K = 256
 * (the timed range) a 256 x 256 pick moves wherever a k_big tile is offered, so k_tiled2's runs below that and where an fp16
 * pick has four sums: over the 143 timed int8 and fp16 shapes with that pick the rule's k_big tile was more than 4% slower
 * at three (int8 K=256 N=12288 M=3300 40.2 -> 41.8 us, K=896 N=9728) and up to 15% faster where the fits call them level
 * (int8 K=256 N=12288 M=4096 54.0 -> 46.1, fp16 K=1024 N=8192 M=3300 79.1 -> 70.8). */
static double pick_us(int rkind, const orkh_plan *q, long wgs, int KB, double mb, int cu) {
    const struct pick_fit *p = pick_fits;
    while (p->rkind != rkind) p++;
    const struct pick_rate *r = pick_rates;
    while (r->rkind != rkind ||
           (r->bm && (r->algo != q->algo || r->bm != q->bm || r->bn != q->bn || r->ring != q->ring)))
        r++;
    const int ks = q->ksplit > 1 ? q->ksplit : 1;
    if (q->bm == 256 && q->bn == 256 && KB * kpb_of(rkind) >= 256) return 1e30;
    const double rounds = (double)((wgs + cu - 1) / cu);
    double t = p->a + rounds * (r->b + r->c * tile_kib(rkind, q->bm, q->bn, ks > 1 ? q->kbs : KB)) + (wgs <= cu ? p->e1 : p->e2) * mb;
    if (ks > 1) t += p->d + p->f * ks * mb;
    return t * p->margin;
}

static double big_us(const struct big_fit *g, long wgs, int KB, double mb, int cu) {
    return g->a + (double)((wgs + cu - 1) / cu) * (g->b + g->c * tile_kib(g->rkind, g->bm, g->bn, KB)) + g->e * mb;
}

/* any planner override of orki_plan in the environment of a context that honours them */
static int overridden(const ork_npu *c) {
    static const char *const names[] = {"ORK_PLAN", "ORK_TILE", "ORK_KSPLIT", "ORK_ALINE", "ORK_RING", "ORK_CWT"};
    if (!c || !c->plan_knobs) return 0;
    for (size_t i = 0; i < sizeof names / sizeof names[0]; i++)
        if (getenv(names[i])) return 1;
    return 0;
}

/* Workgroups of a launch of bm x bn tiles over n matmuls of N[i] columns. Each matmul of a joint launch has tiles of its own
 * and starts on the first XCD (workgroup b runs on XCD b % 8), so it fills whole rows of eight: the first XCD has that many
 * to run, whatever the others have (int8 K=2048 N=2048+1024+1024 M=1281 on 128 x 192: 253 tiles, 34 of them on the first
 * XCD's 32 CUs, two rounds). */
static long tiles_of(int M, const int *N, int n, int bm, int bn) {
    if (n == 1) return (long)cdiv(M, bm) * cdiv(N[0], bn);
    long w = 0;
    for (int i = 0; i < n; i++) w += ((long)cdiv(M, bm) * cdiv(N[i], bn) + 7) / 8 * 8;
    return w;
}

static void take_big(const ork_npu *c, int bm, int bn, int M, const int *N, int n, int KB, orkh_plan *q) {
    const int cu = (c && c->cores > 0) ? c->cores : 256;
    memset(q, 0, sizeof *q);
    q->algo = ORKH_ALGO_BIG;
    q->bm = bm;
    q->bn = bn;
    q->ksplit = 1;
    q->kbs = KB;
    const char *fc = knob(c, "ORK_CWT");
    q->cwt = fc ? atoi(fc) != 0 : tiles_of(M, N, n, bm, bn) <= cu; /* write-through C on one round, as orki_plan's tiles */
}

/* The k_big tile priced below `limit` us for n matmuls of N[i] columns, with at least `sums` fp32 sums an output; 0: none. */
static const struct big_fit *big_best(int rkind, int M, const int *N, int n, int KB, double mb, int cu, int sums, double limit) {
    const struct big_fit *best = NULL;
    for (size_t j = 0; j < sizeof big_fits / sizeof big_fits[0]; j++) {
        const struct big_fit *g = &big_fits[j];
        if (g->rkind != rkind || (rkind == ORKH_F16 && BIG_F16_SUMS(g->bm) < sums)) continue;
        const double t = big_us(g, tiles_of(M, N, n, g->bm, g->bn), KB, mb, cu);
        if (t < limit) {
            limit = t;
            best = g;
        }
    }
    return best;
}

/* ORK_PLAN=big with ORK_TILE=BMxBN */
static int forced_big(int *bm, int *bn) {
    const char *f = getenv("ORK_PLAN"), *t = getenv("ORK_TILE");
    return f && !strcmp(f, "big") && t && sscanf(t, "%dx%d", bm, bn) == 2;
}

int orki_plan_mm(const ork_npu *c, int rkind, int M, int K, int N, int KB, orkh_plan *q, size_t *ws_bytes) {
    const int rc = orki_plan(c, rkind, M, K, N, KB, q, ws_bytes);
    if (rc || M <= 64) return rc;
    int bm, bn;
    if (overridden(c)) {
        if (!forced_big(&bm, &bn)) return 0;
        take_big(c, bm, bn, M, &N, 1, KB, q);
        *ws_bytes = 0;
        return 0;
    }
    if (q->algo != ORKH_ALGO_TILED2 && q->algo != ORKH_ALGO_TILED) return 0;
    const int cu = (c && c->cores > 0) ? c->cores : 256, ks = q->ksplit > 1 ? q->ksplit : 1;
    const double mb = (double)M * N * 4 / 1e6;
    const double us = pick_us(rkind, q, tiles_of(M, &N, 1, q->bm, q->bn) * ks, KB, mb, cu);
    const int sums = rkind == ORKH_F16 ? tiled2_kgroups(rkind, q->bm, q->bn) * ks : 1;
    const struct big_fit *g = big_best(rkind, M, &N, 1, KB, mb, cu, sums, us);
    if (!g) return 0;
    take_big(c, g->bm, g->bn, M, &N, 1, KB, q);
    *ws_bytes = 0;
    return 0;
}

/* The joint launch of n matmuls of one input (the multi-matmul submit): the LDS-ring tile that orki_plan picks for their
 * summed columns, unsplit, or a k_big tile. Each task has tiles of its own, so both are priced at the tiles launched, not at
 * the summed columns' (us, the tile priced at the summed columns, then this rule: int8 K=2048 N=2048+1024+1024 M=1281 264
 * tiles of 128 x 192 30.1, 22.2 on 64 x 192; K=4096 3 x N=4096 M=769 82.0, 61.1; uniform int4 K=2048 3 x N=2048 M=1793 48.1,
 * 36.2; NF4 K=2048 2 x N=1024 M=2689 45.3, 32.3); the joint LDS-ring launch always has the 4-slot ring. Timed at 15
 * lists of widths and 15 row counts, us, orki_plan's tile, this rule: int8 4596, 3837; uniform int4 6773, 5330; NF4 8185,
 * 6685 (one shape over 1% slower: NF4 K=896 2 x N=4864 M=1537, 4.4%). Where orki_plan's pick is no joint launch (K split)
 * the tasks run one by one: no k_big tile was ahead at the 54 such shapes (NF4 K=8192 2 x N=1024 M=1024 50.6 us, 75.8). */
int orki_plan_group(const ork_npu *c, int rkind, int M, int K, const int *N, int n, int KB, orkh_plan *q) {
    int nsum = 0, bm, bn;
    size_t ws = 0;
    for (int i = 0; i < n; i++) nsum += N[i];
    if (orki_plan(c, rkind, M, K, nsum, KB, q, &ws)) return 0;
    const int joint = q->algo == ORKH_ALGO_TILED2 && q->ksplit <= 1;
    if (M <= 64) return joint;
    if (overridden(c)) {
        if (!forced_big(&bm, &bn)) return joint;
        take_big(c, bm, bn, M, N, n, KB, q);
        return 1;
    }
    if (!joint) return 0;
    const int cu = (c && c->cores > 0) ? c->cores : 256;
    const double mb = (double)M * nsum * 4 / 1e6;
    orkh_plan ring4 = *q;
    ring4.ring = 0;
    const double us = pick_us(rkind, &ring4, tiles_of(M, N, n, q->bm, q->bn), KB, mb, cu);
    const int sums = rkind == ORKH_F16 ? tiled2_kgroups(rkind, q->bm, q->bn) : 1;
    const struct big_fit *g = big_best(rkind, M, N, n, KB, mb, cu, sums, us);
    if (g) take_big(c, g->bm, g->bn, M, N, n, KB, q);
    return 1;
}

/* Grouped-scale runs (ork_*_mm_run_grouped). The groups must close in ascending order inside one workgroup, so
 * K is never split. Few rows: k_grouped streams each 16-column panel (and re-reads A per panel, 64 rows at a time above
 * 16). With more rows, int8 and uniform int4 take k_tiled2g at the tile that the prices below make cheapest:
 *   from 32 rows where every group is whole 128-k spans (W4A4 K=N=4096 G=128 M=32: 16.0 us k_grouped, 12.0 64 x 64);
 *   from 17 where groups are one MFMA step (G = 32 or 64), K >= 1024 and N >= 512 (M=17, K=N=4096, W4A4 G=64: 25.9 ->
 *   15.4 us, int8 G=32: 49.1 -> 24.2; they meet at K=1024, N=1536: int8 G=64 6.8 and 6.3; at 16 rows k_grouped wins,
 *   12.2 to 15.4);
 *   from 128 otherwise (a run-time count of steps per group: int8 K=3072 N=512 G=192 M=64 11.4 k_grouped, 12.1 64 x 64,
 *   M=256 12.8 and 12.1).
 * The kernel's index divisions are exact below 2^24, hence the bound on K.
 * NF4 stays on k_grouped (its codebook decode would repeat in every wave row).
 * ORK_PLAN=stream|tiled forces either (tests, A/B), ORK_TILE=BMxBN one of the tiles. */
#define ORKI_GROUPED_TILED_M 32
#define ORKI_GROUPED_TILED_M_STEP 17
#define ORKI_GROUPED_TILED_M_PARTIAL 128
/* A k_tiled2g tile's time in us: a + rounds * (b + K / 1024 * (c + d * 64 / G)), rounds of one workgroup a CU: c is the
 * operands' delivery, d the closing of groups. Fitted to 13 row counts from 32 to 2048 at five (K, N) from 1024 to 6144
 * and seven G from 32 to 512; over them the cheapest by price is within 8% of the fastest, 0.03% in the mean, e.g. (us)
 * W4A4 K=N=4096 G=128: 12.8 on 64 x 64 at M=256 (25.6 on 64 x 192), 24.8 on it and 30.5 on 128 x 128 at M=512, 31.3 on
 * 128 x 128 at M=1000 (48.0 on 64 x 64), 56.5 on 128 x 256 at M=2048 (62.6 on 128 x 128). */
static const struct grouped_fit { int rkind, bm, bn; double a, b, c, d; } grouped_fits[] = {
    {ORKH_I4U, 64, 64, 0.80, 2.41, 1.59, 2.08},  {ORKH_I4U, 64, 128, 0.38, 3.13, 2.94, 3.23},
    {ORKH_I4U, 64, 192, 0.00, 3.74, 3.56, 4.78}, {ORKH_I4U, 128, 128, 0.00, 4.16, 3.94, 6.21},
    {ORKH_I4U, 128, 256, 0.00, 5.53, 7.55, 9.97},
    {ORKH_I8, 64, 64, 0.89, 2.32, 2.05, 1.60},   {ORKH_I8, 64, 128, 0.15, 3.18, 2.64, 3.11},
    {ORKH_I8, 64, 192, 0.12, 3.54, 4.19, 3.84},  {ORKH_I8, 128, 128, 0.00, 3.74, 4.92, 5.03},
    {ORKH_I8, 128, 256, 0.00, 5.16, 7.56, 7.85},
};
void orki_plan_grouped(const ork_npu *c, int rkind, int M, int K, int N, int KB, int G, orkh_plan *q) {
    memset(q, 0, sizeof *q);
    const int cu = (c && c->cores > 0) ? c->cores : 256;
    const char *force = knob(c, "ORK_PLAN");
    int tiled = M >= (G % 128 == 0                       ? ORKI_GROUPED_TILED_M
                      : G <= 64 && K >= 1024 && N >= 512 ? ORKI_GROUPED_TILED_M_STEP
                                                         : ORKI_GROUPED_TILED_M_PARTIAL);
    if (force && !strcmp(force, "stream")) tiled = 0;
    if (force && !strcmp(force, "tiled")) tiled = 1;
    if (tiled && rkind != ORKH_NF4 && K < 1 << 24) {
        const char *tf = knob(c, "ORK_TILE");
        int fbm, fbn;
        if (!tf || sscanf(tf, "%dx%d", &fbm, &fbn) != 2) fbm = fbn = 0;
        double best = -1;
        for (size_t i = 0; i < sizeof grouped_fits / sizeof grouped_fits[0]; i++) {
            const struct grouped_fit *f = &grouped_fits[i];
            if (f->rkind != rkind || (f->bn == 256 && G % 64)) continue;
            const long w = (long)cdiv(M, f->bm) * cdiv(N, f->bn);
            const double t = f->a + (double)((w + cu - 1) / cu) * (f->b + K / 1024.0 * (f->c + f->d * 64 / G));
            const int forced = f->bm == fbm && f->bn == fbn;
            if (best >= 0 && t >= best - 1e-9 && !forced) continue;
            best = t;
            q->bm = f->bm;
            q->bn = f->bn;
            if (forced) break;
        }
        q->algo = ORKH_ALGO_TILED2;
        q->ksplit = 1;
        q->kbs = KB;
        /* write-through C stores on a grid of one round, as for the plain runs */
        const char *fc = knob(c, "ORK_CWT");
        q->cwt = fc ? atoi(fc) != 0 : (long)cdiv(M, q->bm) * cdiv(N / 16, q->bn / 16) <= cu;
        return;
    }
    /* one row: the half-panel VALU kernel (k_grouped_gemv) where the groups' partials fit its LDS (K/G <= 512), runs
     * as the GEMV's (ORK_PLAN=stream keeps k_grouped). Graph-timed against k_grouped (us): W4A4 K=N=4096 G=128
     * 9.6 -> 4.4; int8 K=2048 N=6144 G=128 7.9 -> 4.7; int8 K=2048 N=16384 G=512 8.1 -> 7.5 */
    if (M == 1 && K / G <= 512 && !(force && !strcmp(force, "stream"))) {
        q->algo = ORKH_ALGO_GEMV;
        q->mt = 1;
        q->ksplit = 1;
        q->kbs = KB;
        q->half = 1;
        const int need = cdiv(KB, rkind == ORKH_NF4 ? 4 : 8);
        q->wpg = need <= 2 ? 2 : need <= 4 ? 4 : 8;
        q->kbw = cdiv(KB, q->wpg);
        return;
    }
    q->algo = ORKH_ALGO_STREAM;
    q->mt = M > 16 ? 4 : 1;
    q->ksplit = 1;
    q->kbs = KB;
}
