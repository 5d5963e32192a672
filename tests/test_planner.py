"""The planner's picks against measurements, on the CPU: single runs (orki_plan, and orki_plan_mm above 64 rows), chains'
joint launches and grouped-scale runs, each against its sweep under tests/golden.

tests/planner/plan_names.c prints the planner's choice (plan.c alone, a 256-CU device) for each shape of
tests/golden/nf4_plan_sweep.json, which holds graph-timed MI355X launches of every NF4 kernel, tile and K split on
offer at 45 shapes (tests/golden/nf4_plan_sweep.py made it). Each pick must be a timed candidate, within 15% of the
fastest at its shape, and the picks must total within 2% of the fastest candidates' total. The planner's fits
were made on these launches, so this pins the fits as implemented in C against the data, not their accuracy on
other shapes.
"""
import json
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CLANG = "/opt/rocm/llvm/bin/clang"   # _Float16 in the public header needs clang on x86


@pytest.fixture(scope="module")
def planner(tmp_path_factory):
    if not os.path.exists(CLANG):
        pytest.skip("ROCm clang not installed")
    exe = str(tmp_path_factory.mktemp("planner") / "plan_names")
    hs = os.path.join(ROOT, "ork-driver_amd", "csrc", "host")
    r = subprocess.run([CLANG, "-O1", "-std=gnu11", "-Wall", "-Werror", "-ffp-contract=off",
                        "-I" + os.path.join(ROOT, "include"), "-I" + hs,
                        "-I" + os.path.join(ROOT, "ork-driver_amd", "csrc", "hip"),
                        os.path.join(ROOT, "tests", "planner", "plan_names.c"), os.path.join(hs, "plan.c"),
                        "-o", exe, "-lm"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]

    def pick(cases, mm=False, chain=False, grouped=False):
        args = ["mm"] * mm + ["chain"] * chain + ["grouped"] * grouped + [str(x) for c in cases for x in c]
        out = subprocess.run([exe] + args, capture_output=True, text=True, timeout=60, env={}).stdout.split("\n")
        return [ln.split()[4] for ln in out if ln.strip()]
    return pick


def test_nf4_picks_against_the_sweep(planner):
    data = json.load(open(os.path.join(ROOT, "tests", "golden", "nf4_plan_sweep.json")))
    shapes = data["shapes"]
    assert len(shapes) == 45
    picks = planner([(2, s["M"], s["K"], s["N"]) for s in shapes])
    tot_pick = tot_best = 0.0
    for s, p in zip(shapes, picks):
        best = min(s["us"].values())
        assert p in s["us"], (s["K"], s["N"], s["M"], p)
        assert s["us"][p] <= 1.15 * best, (s["K"], s["N"], s["M"], p, s["us"][p], best)
        tot_pick += s["us"][p]
        tot_best += best
    assert tot_pick <= 1.02 * tot_best, (tot_pick, tot_best)


def test_fixed_picks(planner):
    """The benchmark's two halves and the NF4 decode row keep their kernels (the committed rocprof summaries under
    profiles/ are of these): the half-panel GEMV at M=1, the 128 x 96 LDS-ring tile with line-loaded A at M=512 (int8
    K=2048 N=6144), the GEMV for NF4 at M=1."""
    got = planner([(0, 1, 2048, 6144), (0, 512, 2048, 6144), (2, 1, 2048, 6144)])
    assert got[0].startswith("gemvh_i8_") and got[1] == "tiled2_i8_128x96_al" and got[2].startswith("gemvh_nf4_"), got


def test_stream_half_panels_offered(planner):
    """Half panels on the streaming kernel: taken for fp16 and int8 where the halves still fit one round of the CUs
    (C2 fp16 K=N=2048 M=16: 4.98 -> 4.41 us measured; int8 K=6144 N=2048 M=16), not where they would need a second
    round (int8 K=N=4096 M=16), not with paired panels (C1 M=16), never for the nibble kinds."""
    got = planner([(3, 16, 2048, 2048), (0, 16, 6144, 2048), (0, 16, 4096, 4096), (0, 16, 2048, 6144),
                   (1, 16, 2048, 2048), (2, 16, 2048, 2048)])
    assert got[0].startswith("stream_f16_") and got[0].endswith("_h"), got
    assert got[1].startswith("stream_i8_") and got[1].endswith("_h"), got
    assert not got[2].endswith("_h") and got[3].endswith("_p2"), got
    assert not got[4].endswith("_h") and not got[5].endswith("_h"), got


def test_two_slot_ring_picks(planner):
    """The LDS-ring kernel's two-slot ring: taken on grids of more than one round where the tile has it (int8
    K=2048 N=6144 M=768 and 1024 on 64 x 192; fp16 K=N=2048 M=4096 and uniform int4 K=2048 N=6144 M=2048 on
    128 x 128), not on one round (M=512), never on 256 x 256 nor for NF4."""
    got = planner([(0, 768, 2048, 6144), (0, 1024, 2048, 6144), (3, 4096, 2048, 2048), (1, 2048, 2048, 6144),
                   (0, 512, 2048, 6144), (0, 4096, 4096, 4096), (2, 1024, 2048, 6144)])
    assert all(g.endswith("_r2") for g in got[:4]), got
    assert not any(g.endswith("_r2") for g in got[4:]), got
    # uniform int4, whose 64 x 192 tile has no two-slot form, moves to 128 x 128 with two slots where both grids
    # exceed one round (K=2048 N=6144 M=768: 21.74 -> 19.96 us), not where 64 x 192 fills one (K=N=4096 M=512)
    got = planner([(1, 768, 2048, 6144), (1, 512, 4096, 4096)])
    assert got[0] == "tiled2_i4u_128x128_al_r2" and got[1].startswith("tiled2_i4u_64x192") and "_r2" not in got[1], got


@pytest.mark.parametrize("kind", ["int8", "i4u", "fp16"])
def test_mma_picks_against_the_sweep(planner, kind):
    """int8, fp16 and uniform int4 above 64 rows (tests/golden/mma_plan_sweep.json: graph-timed launches of every
    LDS-ring tile and K split on offer at 36-39 shapes per kind): each pick is a timed candidate within 20% of the
    fastest at its shape (the worst: fp16 K=N=4096 M=256, 23.9 us on 64 x 64 against 20.9 on 128 x 128 split 4 ways,
    where both fits are off by ~10%), and the picks total within 2% of the fastest candidates' total."""
    data = json.load(open(os.path.join(ROOT, "tests", "golden", "mma_plan_sweep.json")))
    shapes = [s for s in data["shapes"] if s["kind"] == kind]
    if not shapes:
        pytest.skip(f"no {kind} launches in the sweep")
    rk = {"int8": 0, "i4u": 1, "fp16": 3}[kind]
    picks = planner([(rk, s["M"], s["K"], s["N"]) for s in shapes])
    tot_pick = tot_best = 0.0
    worst = []
    for s, p in zip(shapes, picks):
        best = min(s["us"].values())
        assert p in s["us"], (s["K"], s["N"], s["M"], p)
        worst.append((s["us"][p] / best, s["K"], s["N"], s["M"], p))
        tot_pick += s["us"][p]
        tot_best += best
    assert max(worst)[0] <= 1.20, max(worst)
    assert tot_pick <= 1.02 * tot_best, (tot_pick, tot_best, sorted(worst)[-3:])


@pytest.mark.parametrize("kind", ["int8", "i4u", "nf4", "fp16"])
def test_run_picks_against_the_sweep(planner, kind):
    """What a run above 64 rows takes (orki_plan_mm: orki_plan's pick or a tile of the many-row kernel) against graph-timed
    launches of both at 633 shapes a kind, K from 256 to 8192 and M from 65 to 4096 (tests/golden/big_plan_sweep.json): no
    shape over 4% slower than orki_plan's pick (11% where that is 256 x 256, which moves at every K here), and
    the total within 1% of the faster of the two everywhere (fp16: of the tiles with the pick's fp32 sums). The bounds are
    the rule's worst on these launches (K=896 N=9728); before it was fitted below K = 2048 the worst was 42%."""
    data = json.load(open(os.path.join(ROOT, "tests", "golden", "big_plan_sweep.json")))
    runs = [r for r in data["runs"] if r[0] == kind]
    assert len(runs) == 633
    rk = {"int8": 0, "i4u": 1, "nf4": 2, "fp16": 3}[kind]
    cases = [(rk, M, K, N) for _, K, N, M, *_ in runs]
    tot_pick = tot_best = tot_former = 0.0
    for (_, K, N, M, former, us, *big), old, p in zip(runs, planner(cases), planner(cases, mm=True)):
        assert old == former, (K, N, M, old, former)
        kn = {"int8": "i8", "fp16": "f16"}.get(kind, kind)
        times = {"big_%s_%s" % (kn, t): x for t, x in zip(("256x256", "256x192", "128x256", "128x192"), big)}
        if kind == "fp16":
            times = {t: x for t, x in times.items() if _f16_sums(t) >= _f16_sums(former)}
        times[former] = us
        assert times[p] <= (1.11 if "256x256" in former else 1.04) * us, (K, N, M, former, us, p, times[p])
        tot_pick += times[p]
        tot_best += min(times.values())
        tot_former += us
    assert tot_pick <= 1.01 * tot_best and tot_pick < 0.94 * tot_former, (tot_pick, tot_best, tot_former)


@pytest.mark.parametrize("kind", ["int8", "i4u", "nf4"])
def test_chain_picks_against_the_sweep(planner, kind):
    """The joint launch of a chain's matmuls against graph-timed launches (tests/golden/big_plan_sweep.json: 15 lists of
    widths, M from 65 to 2689) on every many-row tile and on the LDS-ring tiles: where orki_plan's pick for the summed
    columns is one of those, the joint launch is at most 5% slower than on it, and the total within 1% of the faster of
    the two everywhere. Each task has tiles of its own: a tile priced at the summed columns' count ran up to 52% slower."""
    data = json.load(open(os.path.join(ROOT, "tests", "golden", "big_plan_sweep.json")))
    rows = [r for r in data["chains"] if r[0] == kind]
    rk, kn = {"int8": (0, "i8"), "i4u": (1, "i4u"), "nf4": (2, "nf4")}[kind]
    former = planner([(rk, M, K, sum(Ns)) for _, K, Ns, M, *_ in rows])
    picks = planner([(rk, M, K, len(Ns), *Ns) for _, K, Ns, M, *_ in rows], chain=True)
    tiles = ["big_%s_%s" % (kn, t) for t in ("256x256", "256x192", "128x256", "128x192")] + \
            ["tiled2_%s_%s" % (kn, t) for t in ("128x128", "128x96", "64x192", "64x64")]
    tot_pick = tot_best = n = 0
    for (_, K, Ns, M, *us), f, p in zip(rows, former, picks):
        times = {t: x for t, x in zip(tiles, us) if x}
        f, p = ("_".join(x.split("_")[:3]) if "_ks" not in x else x for x in (f, p))
        if f not in times:
            continue
        assert times[p] <= 1.05 * times[f], (K, Ns, M, f, times[f], p, times[p])
        tot_pick += times[p]
        tot_best += min(v for t, v in times.items() if t == f or t.startswith("big_"))
        n += 1
    assert n > 100 and tot_pick <= 1.01 * tot_best, (n, tot_pick, tot_best)


@pytest.mark.parametrize("kind", ["int8", "i4u"])
def test_grouped_picks_against_the_sweep(planner, kind):
    """Grouped-scale runs against graph-timed launches of the panel-streaming kernel and every tile of k_tiled2g
    (tests/golden/grouped_plan_sweep.json: 13 (K, N), eleven group sizes from 32 to 768, M from 17 to 2048): where the plan is
    a tile, its total is within 0.5% of the fastest tile's or kernel's everywhere and no shape over 10% slower (int4
    K=2048 N=6144 M=768 G=64 8.5%; K=1024 runs of 5 us where the streaming kernel is 3 to 6% ahead). Where it keeps the
    streaming kernel, from 17 rows with groups of whole 128-k spans and from 17 to 127 with G = 96, 192 and 320, a tile is
    often ahead; those are not asserted."""
    runs = [r for r in json.load(open(os.path.join(ROOT, "tests", "golden", "grouped_plan_sweep.json")))["runs"] if r[0] == kind]
    assert len(runs) == 1192
    rk = {"int8": 0, "i4u": 1}[kind]
    picks = planner([(rk, M, K, N, G) for _, K, N, G, M, *_ in runs], grouped=True)
    names = ("stream", "64x64", "64x128", "64x192", "128x128", "128x256")
    tot_pick = tot_best = tiles = 0
    for (_, K, N, G, M, *us), p in zip(runs, picks):
        times = {n: x for n, x in zip(names, us) if x}
        if p == "stream":
            continue
        best = min(times.values())
        assert times[p] <= 1.10 * best, (K, N, G, M, p, times)
        tot_pick += times[p]
        tot_best += best
        tiles += 1
    assert tiles > 900 and tot_pick <= 1.005 * tot_best, (tiles, tot_pick, tot_best)


def _f16_sums(name):
    """fp32 sums an output has under a plan: K groups of waves (k_tiled2's 16 waves over its tile; k_big's 128-row tiles:
    2) times the K split"""
    bm, bn = map(int, name.split("_")[2].split("x"))
    if name.startswith("big_"):
        return 2 if bm == 128 else 1
    mb, nb = min(bm // 16, 4), bn // 16
    nb = nb if nb < 4 else 4 if nb % 4 == 0 else 2
    return 16 // (mb * nb) * int(name.split("_ks")[1].split("_")[0] if "_ks" in name else 1)


def test_f16_sums_not_longer(planner):
    """fp16 above 64 rows: a run on the many-row kernel keeps at least as many fp32 sums an output (each over that share
    of K) as the LDS-ring pick it replaces, over 5,000 shapes; both kinds of move (one sum, two sums) occur."""
    cases = [(3, M, K, N) for K in (256, 1024, 2048, 3072, 4096, 6144, 8192, 16384) for N in (512, 1024, 2048, 4096, 6144, 8192, 12288)
             for M in list(range(65, 600, 31)) + list(range(600, 4200, 53))]
    moved = {}
    for lo in range(0, len(cases), 1000):
        part = cases[lo:lo + 1000]
        for c, a, b in zip(part, planner(part), planner(part, mm=True)):
            if b.startswith("big_"):
                assert _f16_sums(b) >= _f16_sums(a), (c, a, b)
                moved[_f16_sums(a)] = moved.get(_f16_sums(a), 0) + 1
            else:
                assert a == b, (c, a, b)
    assert moved.get(1) and moved.get(2), moved
