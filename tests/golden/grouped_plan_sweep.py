"""Graph-timed launches behind the planner's choice for grouped-scale runs (plan.c, orki_plan_grouped): the panel-streaming
kernel (k_grouped) and every tile of k_tiled2g. Writes grouped_plan_sweep.json beside this file (read by
tests/test_planner.py).

On one MI355X, from the repository root, with the library built:
    python3 tests/golden/grouped_plan_sweep.py KIND > LOG              # int8, i4u (W4A4); --default: the default plan only
    python3 tests/golden/grouped_plan_sweep.py --reduce LOG [LOG ...]  # write the fixture from the JSON lines
Times are the least of two, us per launch, weights rotated over up to 16 copies; results are checked by the tests of these
kernels, not here.
"""
import json
import os
import sys

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import big_plan_sweep as S  # noqa: E402

OUT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "grouped_plan_sweep.json")
PAIRS = ((1024, 512), (1024, 1536), (1024, 4096), (2048, 512), (2048, 2048), (2048, 6144), (3072, 512), (3072, 3072), (4096, 512),
         (4096, 1024), (4096, 4096), (6144, 2048), (3840, 2560))
GROUPS = (32, 64, 96, 128, 192, 256, 320, 384, 512, 640, 768)
ROWS = (17, 20, 24, 32, 48, 64, 96, 128, 200, 256, 384, 512, 768, 1024, 2048)
TILES = ("64x64", "64x128", "64x192", "128x128", "128x256")
MAX_MACS = 4096 * 4096 * 1024


def sweep(kinds, only):
    bench, ork = S.setup()
    import numpy as np
    rng = np.random.default_rng(6)
    hip, L = bench.Hip(), ork.lib()
    with ork.Npu() as npu:
        L.ork_npu_set_async(npu.h, 1)
        for kind in kinds:
            lo = -128 if kind == "int8" else -8
            entry = "ork_i8_mm_run_grouped" if kind == "int8" else "ork_i4_mm_run_grouped"
            for K, N in PAIRS:
                B = rng.integers(lo, -lo, size=(K, N), dtype=np.int8)
                Ms = [M for M in ROWS if M * K * N <= MAX_MACS]
                A = rng.integers(-7, 8, size=(Ms[-1], K), dtype=np.int8)
                dA, dC = L.ork_dev_alloc(npu.h, A.nbytes), L.ork_dev_alloc(npu.h, Ms[-1] * N * 4)
                assert dA and dC and L.ork_dev_upload(npu.h, dA, ork.ptr(A), A.nbytes) == 0
                for G in GROUPS:
                    if K % G:
                        continue
                    aS = rng.uniform(1e-3, 1e-2, size=(Ms[-1], K // G)).astype(np.float32)
                    bS = rng.uniform(1e-3, 1e-2, size=(K // G, N)).astype(np.float32)
                    daS, dbS = (L.ork_dev_alloc(npu.h, x.nbytes) for x in (aS, bS))
                    for d, x in ((daS, aS), (dbS, bS)):
                        assert d and L.ork_dev_upload(npu.h, d, ork.ptr(x), x.nbytes) == 0
                    ws = []
                    for _ in range(min(16, S.copies(kind, K * N))):
                        if kind == "int8":
                            w = npu.pack_i8(B)
                            assert w and L.ork_w_set_group(w, G) == 0
                        else:
                            w = L.ork_i4_mm_pack_grouped(npu.h, K, N, ork.ptr(B), G)
                        assert w
                        ws.append(w)
                    for M in Ms:
                        us = {}
                        cands = [("default", {})]
                        if not only:
                            cands += [("stream", {"ORK_PLAN": "stream"})] + \
                                     [(t, {"ORK_PLAN": "tiled", "ORK_TILE": t}) for t in TILES if t != "128x256" or G % 64 == 0]
                        if M <= 16 or (M > 256 and len(cands) > 1):
                            cands = [c for c in cands if c[0] != "stream"]
                        for name, e in cands:
                            with S.Env(**e):
                                us[name] = round(min(bench.measure(npu, hip, ws, M, dA, dC, 32, 2, entry, (daS, dbS))[0]
                                                     for _ in range(2)) * 1e3, 2)
                        print(json.dumps({"kind": kind, "K": K, "N": N, "G": G, "M": M, "plan": npu.grouped_plan_name(ws[0], M),
                                          "us": us}), flush=True)
                    for w in ws:
                        L.ork_mm_free(npu.h, w)
                    for d in (daS, dbS):
                        L.ork_dev_free(npu.h, d)
                L.ork_dev_free(npu.h, dA)
                L.ork_dev_free(npu.h, dC)


def reduce(logs):
    rows = [json.loads(x) for f in logs for x in open(f) if x.startswith("{")]
    with open(OUT, "w") as f:
        f.write(json.dumps({"units": "us per launch, graph-timed on one MI355X, weights rotated over up to 16 copies",
                            "made_by": "tests/golden/grouped_plan_sweep.py",
                            "fields": "kind, K, N, G, M, us of k_grouped (null: not timed), of k_tiled2g on " + ", ".join(TILES) +
                                      " (null: not built)"}, indent=1)[:-2])
        f.write(',\n "runs": [\n' + ",\n".join(json.dumps([r["kind"], r["K"], r["N"], r["G"], r["M"]] + [r["us"].get(t) for t in ("stream",) + TILES],
                                                         separators=(",", ":")) for r in rows) + "\n ]\n}\n")


if __name__ == "__main__":
    if sys.argv[1:2] == ["--reduce"]:
        reduce(sys.argv[2:])
        sys.exit()
    sweep([k for k in sys.argv[1:] if not k.startswith("--")], "--default" in sys.argv)
