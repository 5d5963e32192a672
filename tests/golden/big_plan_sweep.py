"""Graph-timed launches behind the planner's choice between the many-row kernel (k_big) and the smaller tiles above 64 rows
(plan.c, orki_plan_cols): at each shape every k_big tile and orki_plan's own pick, for single runs of each weight kind and
for the multi-matmul submit's joint launches (ork_i8_mm_run_chain: several weights, one input). Writes big_plan_sweep.json
beside this file (read by tests/test_planner.py).

On one MI355X, from the repository root, with the library built:
    python3 tests/golden/big_plan_sweep.py KIND [KIND ...] > LOG    # int8 i4u nf4 fp16, chain
    python3 tests/golden/big_plan_sweep.py --reduce LOG [LOG ...]   # write the fixture from the JSON lines, fit
uniform int4 runs as W4A4 (ork_i4_mm_run): the same kernels as W4A8; in chains as W4A8. Times are the least of two, us per
launch, weights rotated over up to 24 copies; results are checked by the tests of these tiles, not here.

The fits are the forms plan.c evaluates, least squares on the relative error with non-negative terms:
    k_big, per tile     a + rounds * (b + c * KiB) + e * MB
    orki_plan's pick    a + rounds * (b[tile] + c[tile] * KiB) + e * MB + [ks > 1] (d + f * ks * MB)
                        (e: e1 on one round of the CUs, else e2)
KiB being the A and B bytes one workgroup loads and MB C's megabytes; a k_big tile's fit takes the shapes where it ran within
1.6 times the fastest.
"""
import json
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
OUT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "big_plan_sweep.json")
PAIRS = ((256, 2048), (256, 6144), (256, 12288), (512, 4096), (512, 12288), (1024, 1024), (1024, 3072), (1024, 8192), (2048, 512),
         (2048, 2048), (2048, 4096), (2048, 6144), (2048, 12288), (4096, 1024), (4096, 4096), (4096, 11008), (6144, 2048), (8192, 4096),
         (896, 4864), (896, 9728), (1536, 1536), (2048, 8192), (2048, 16384), (2560, 9728), (3072, 5120), (4096, 512), (4096, 2560),
         (6144, 1024), (8192, 512), (8192, 1024), (8192, 2560))
ROWS = (65, 96, 128, 160, 200, 257, 320, 384, 448, 512, 641, 769, 900, 1024, 1280, 1537, 1793, 2048, 2689, 3300, 4096)
CHAINS = ((2048, (2048, 1024, 1024)), (2048, (6144, 6144)), (2048, (2048, 2048, 2048)), (2048, (1024, 1024)), (2048, (2048, 512, 512)),
          (4096, (4096, 2048)), (4096, (4096, 4096, 4096)), (1024, (3072, 1024, 1024)), (4096, (11008, 11008)), (512, (4096, 4096)),
          (896, (4864, 4864)), (2048, (8192, 8192)), (8192, (2048, 512)), (8192, (1024, 1024)), (6144, (1024, 512, 512)))
CHAIN_ROWS = (65, 128, 200, 256, 384, 500, 641, 769, 897, 1024, 1281, 1537, 1793, 2048, 2689)
BIG = ("256x256", "256x192", "128x256", "128x192")
CHAIN_TILES = ("128x128", "128x96", "64x192", "64x64")   # the smaller tiles of a joint launch
RKIND = {"int8": 0, "i4u": 1, "nf4": 2, "fp16": 3}
MAX_MACS = 4096 ** 3
CU = 256
STEPS = 48


def cdiv(a, b):
    return -(-a // b)


def kblocks(kind, K):
    return cdiv(K, {"int8": 64, "fp16": 32}.get(kind, 128))


class Env:
    def __init__(self, **kv):
        self.kv = kv

    def __enter__(self):
        os.environ.update(self.kv)

    def __exit__(self, *a):
        for k in self.kv:
            os.environ.pop(k, None)


def setup():
    sys.path[:0] = [os.path.join(ROOT, "ork-driver_amd"), ROOT]
    os.environ["ORK_PLAN_DEBUG"] = "1"
    import bench
    import ork
    bench.WARM_S = 0.01
    return bench, ork


def packer(npu, np, kind, K, N, rng):
    """packs one random weight, again each call"""
    if kind == "fp16":
        B = (rng.standard_normal((K, N), np.float32) * 0.02).astype(np.float16)
        return lambda: npu.pack_f16(B)
    if kind in ("int8", "i4u"):
        lo = -128 if kind == "int8" else -8
        B = rng.integers(lo, -lo, size=(K, N), dtype=np.int8)
        return lambda: (npu.pack_i8 if kind == "int8" else npu.pack_i4)(B)
    W = rng.standard_normal((N, K), np.float32) * np.float32(0.02)

    def pack():
        with Env(**({"ORK_NF4": "1"} if kind == "nf4" else {})):
            return npu.pack_i4a8(W)[0]
    return pack


def copies(kind, n):
    """copies of a weight of n codes, so that rotating over them reads most of it from HBM"""
    return int(min(24, max(2, 400e6 // (n * {"fp16": 2, "int8": 1}.get(kind, 0.5)))))


def pick_env(npu, w, M, N):
    """an override that leaves orki_plan's pick as it is and turns the many-row rule off: its own store policy"""
    with Env(ORK_CWT="1"):
        name = npu.plan_name(w, M)
    bm, bn = map(int, name.split("_")[2].split("x"))
    ks = int(name.split("_ks")[1].split("_")[0]) if "_ks" in name else 1
    return {"ORK_CWT": "1" if cdiv(M, bm) * cdiv(N // 16, bn // 16) * ks <= CU else "0"}, name


def sweep(kinds):
    bench, ork = setup()
    import numpy as np
    rng = np.random.default_rng(5)
    hip, L = bench.Hip(), ork.lib()
    with ork.Npu() as npu:
        L.ork_npu_set_async(npu.h, 1)
        for kind in [k for k in kinds if k in RKIND]:
            entry = {"fp16": "ork_f16_mm_run", "i4u": "ork_i4_mm_run"}.get(kind, "ork_i8_mm_run")
            for K, N in PAIRS:
                pack = packer(npu, np, kind, K, N, rng)
                ws = [pack() for _ in range(copies(kind, K * N))]
                assert all(ws)
                Ms = [M for M in ROWS if M * K * N <= MAX_MACS]
                A = rng.standard_normal((Ms[-1], K)).astype(np.float16) if kind == "fp16" else \
                    rng.integers(-7, 8, size=(Ms[-1], K), dtype=np.int8)
                dA, dC = L.ork_dev_alloc(npu.h, A.nbytes), L.ork_dev_alloc(npu.h, Ms[-1] * N * 4)
                assert dA and dC and L.ork_dev_upload(npu.h, dA, ork.ptr(A), A.nbytes) == 0
                for M in Ms:
                    env, pick = pick_env(npu, ws[0], M, N)
                    us = {}
                    for name, e in [(pick, env)] + [("big_" + t, {"ORK_PLAN": "big", "ORK_TILE": t}) for t in BIG]:
                        with Env(**e):
                            us[name] = round(min(bench.measure(npu, hip, ws, M, dA, dC, STEPS, 4, entry)[0] for _ in range(2)) * 1e3, 2)
                    print(json.dumps({"kind": kind, "K": K, "N": N, "M": M, "pick": pick, "us": us}), flush=True)
                for w in ws:
                    L.ork_mm_free(npu.h, w)
                L.ork_dev_free(npu.h, dA)
                L.ork_dev_free(npu.h, dC)
        if "chain" in kinds:
            for kind in ("int8", "i4u", "nf4"):
                for K, Ns in CHAINS:
                    chains(npu, ork, hip, bench, np, kind, K, Ns, rng)


def chains(npu, ork, hip, bench, np, kind, K, Ns, rng):
    L = ork.lib()
    Ms = [M for M in CHAIN_ROWS if M * K * sum(Ns) <= 2 * MAX_MACS]
    A = rng.integers(-7, 8, size=(Ms[-1], K), dtype=np.int8)
    dA = L.ork_dev_alloc(npu.h, A.nbytes)
    assert dA and L.ork_dev_upload(npu.h, dA, ork.ptr(A), A.nbytes) == 0

    packs = [packer(npu, np, "i4a8" if kind == "i4u" else kind, K, N, rng) for N in Ns]
    sets = [[p() for p in packs] for _ in range(copies(kind, K * sum(Ns)))]
    dC = [L.ork_dev_alloc(npu.h, Ms[-1] * N * 4) for N in Ns]
    for M in Ms:
        tasks = [ork.tasks(ork.TaskI8, [(w, M, dA, c) for w, c in zip(s, dC)]) for s in sets]
        us = {}
        cands = [("default", {})] + [("big_" + t, {"ORK_PLAN": "big", "ORK_TILE": t}) for t in BIG] + \
                [("tiled2_" + t, {"ORK_TILE": t}) for t in CHAIN_TILES if not (kind == "nf4" and t == "64x192")]
        for name, e in cands:
            with Env(**e):
                us[name] = round(min(bench.measure(npu, hip, tasks, M, dA, dC, 24, 2, call=lambda t: L.ork_i8_mm_run_chain(npu.h, len(Ns), t))[0]
                                     for _ in range(2)) * 1e3, 2)
        print(json.dumps({"kind": kind, "K": K, "Ns": list(Ns), "M": M, "us": us}), flush=True)
    for w in [w for s in sets for w in s]:
        L.ork_mm_free(npu.h, w)
    for d in dC + [dA]:
        L.ork_dev_free(npu.h, d)


def tile_of(name):
    """(kernel, bm, bn, K split, two-slot ring) of a tiled plan's name"""
    bm, bn = map(int, name.split("_")[2].split("x"))
    ks = int(name.split("_ks")[1].split("_")[0]) if "_ks" in name else 1
    return name.split("_")[0], bm, bn, ks, name.endswith("_r2")


def kib(kind, bm, bn, kb):
    return (bm * (128 if kind in ("i4u", "nf4") else 64) + bn * 64) * kb / 1024


def nnls_rel(X, t):
    """non-negative least squares on the relative error: coefficients, rms"""
    import numpy as np
    from scipy.optimize import nnls
    X, t = np.array(X, float), np.array(t)
    coef, _ = nnls(X / t[:, None], np.ones(len(t)))
    return [round(float(x), 4) for x in coef], round(float(np.sqrt(np.mean((X @ coef / t - 1) ** 2))), 3)


def fits(kind, rows):
    out = {"big": {}, "tiles": {}}
    for tile in BIG:
        bm, bn = map(int, tile.split("x"))
        X, t = [], []
        for r in rows:
            if r["us"]["big_" + tile] <= 1.6 * min(r["us"].values()):
                rounds = cdiv(cdiv(r["M"], bm) * cdiv(r["N"], bn), CU)
                X.append([1.0, rounds, rounds * kib(kind, bm, bn, kblocks(kind, r["K"])), r["M"] * r["N"] * 4e-6])
                t.append(r["us"]["big_" + tile])
        coef, rms = nnls_rel(X, t)
        out["big"][tile] = {"abce": coef, "rms": rms, "n": len(t)}
    tiles = sorted({tile_of(r["pick"])[:3] + tile_of(r["pick"])[4:] for r in rows})
    X, t = [], []
    for r in rows:
        algo, bm, bn, ks, r2 = tile_of(r["pick"])
        mb, w = r["M"] * r["N"] * 4e-6, cdiv(r["M"], bm) * cdiv(r["N"], bn) * ks
        f = [1.0, mb * (w <= CU), mb * (w > CU), float(ks > 1), ks * mb * (ks > 1)] + [0.0] * (2 * len(tiles))
        j, rounds = 5 + 2 * tiles.index((algo, bm, bn, r2)), cdiv(w, CU)
        f[j], f[j + 1] = rounds, rounds * kib(kind, bm, bn, cdiv(kblocks(kind, r["K"]), ks))
        X.append(f)
        t.append(r["us"][r["pick"]])
    coef, rms = nnls_rel(X, t)
    out["pick"] = {"a_e1_e2_d_f": coef[:5], "rms": rms, "n": len(t)}
    for j, tl in enumerate(tiles):
        out["tiles"]["%s_%dx%d%s" % (tl[0], tl[1], tl[2], "_r2" * tl[3])] = coef[5 + 2 * j:7 + 2 * j]
    return out


def reduce(logs):
    rows = [json.loads(x) for f in logs for x in open(f) if x.startswith("{")]
    runs = [r for r in rows if "N" in r]
    data = {"units": "us per launch, graph-timed on one MI355X, weights rotated over up to 24 copies",
            "made_by": "tests/golden/big_plan_sweep.py",
            "runs_fields": "kind, K, N, M, orki_plan's pick, its us, us of k_big on " + ", ".join(BIG),
            "chains_fields": "kind, K, N of each task, M, us of k_big on " + ", ".join(BIG) + ", of k_tiled2m on " +
                             ", ".join(CHAIN_TILES) + " (null: not built for the kind)",
            "fits": {k: fits(k, [r for r in runs if r["kind"] == k]) for k in RKIND if any(r["kind"] == k for r in runs)}}
    rows_of = {"runs": [[r["kind"], r["K"], r["N"], r["M"], r["pick"], r["us"][r["pick"]]] + [r["us"]["big_" + t] for t in BIG]
                        for r in runs],
               "chains": [[r["kind"], r["K"], r["Ns"], r["M"]] + [r["us"]["big_" + t] for t in BIG] +
                          [r["us"].get("tiled2_" + t) for t in CHAIN_TILES] for r in rows if "Ns" in r]}
    with open(OUT, "w") as f:
        f.write(json.dumps(data, indent=1)[:-2])
        for k, rs in rows_of.items():
            f.write(',\n "%s": [\n' % k + ",\n".join(json.dumps(r, separators=(",", ":")) for r in rs) + "\n ]")
        f.write("\n}\n")
    print(json.dumps(data["fits"], indent=1))


if __name__ == "__main__":
    if sys.argv[1:2] == ["--reduce"]:
        reduce(sys.argv[2:])
    else:
        sweep(sys.argv[1:])
