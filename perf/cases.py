"""The calls that a user of this library spends their time in, as cases that can be prepared, run and checked one by one.

Every case goes through the public C API (the ctypes bindings of ork-driver_amd) on one device context, as a program
does: weights are packed once and stay resident, activations and results live in device buffers of the context, and
device-resident runs are asynchronous. Two kinds of calls take host data by their nature: packing a model's weights, and
the reference's own calling convention (host A, host C, C valid on return).

  mm        one matmul on a resident weight: ork_i8_mm_run (int8, uniform int4 and NF4 weights), ork_f16_mm_run,
            ork_i4_mm_run
  chain     the projections that share one input (q / k / v, gate / up) as one ork_i8_mm_run_chain
  grouped   a grouped-scale matmul: ork_i4_mm_run_grouped / ork_i8_mm_run_grouped
  host      ork_i8_mm_run with host operands
  pack      ork_i8_mm_pack_f32 / ork_i4a8_mm_pack_im of one linear layer
  prefill   q3_prefill of a Qwen3-shaped decoder (a few layers of it), and the logits of the last position
  generate  a short prompt and greedy decode steps of the same decoder
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "ork-driver_amd"))

import ork  # noqa: E402
import qwen3  # noqa: E402

MAX_FLOPS = 2.0 * 4096 ** 3  # the largest listed matmul
MAX_OPERANDS = 192e6         # bytes of a drawn matmul's A, B (as fp32) and C, so that preparing it stays quick

# Qwen3-1.7B widths (the decoder of bench.py and the tests), a few layers deep
WIDTHS = dict(qwen3.QWEN3_1P7B)

_npu = None


def npu():
    """One context for the process, as a program has."""
    global _npu
    if _npu is None:
        torch.cuda.init()
        _npu = ork.Npu()
    return _npu


# ---- what a program holds: device buffers, weights, models --------------------------------------------------------------

TYPESTR = {torch.int8: "|i1", torch.int32: "<i4", torch.float32: "<f4", torch.float16: "<f2", torch.uint8: "|u1"}


class _Memory:
    """A span of device memory; `own`: an ork_dev_alloc buffer, given back with this object."""

    def __init__(self, ptr, shape, dtype, own):
        self.ptr, self.own = ptr, own
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": TYPESTR[dtype], "data": (ptr, False), "version": 2}

    def __del__(self):
        if self.own:
            ork.lib().ork_dev_free(npu().h, self.ptr)


def device_buffer(shape, dtype, like=None):
    """A tensor in a device buffer of the context (with the values of `like`)."""
    n = math.prod(shape) * torch.empty((), dtype=dtype).element_size()
    ptr = ork.lib().ork_dev_alloc(npu().h, n)
    if not ptr:
        raise RuntimeError("out of memory: ork_dev_alloc(%d)" % n)
    t = torch.as_tensor(_Memory(ptr, shape, dtype, True), device="cuda")
    if like is None:
        t.zero_()
    else:
        t.copy_(like)
    return t


class Weight:
    def __init__(self, h):
        if not h:
            raise RuntimeError("a pack failed (out of memory?)")
        self.h = h

    def __del__(self):
        ork.lib().ork_mm_free(npu().h, self.h)


class Decoder:
    def __init__(self, cfg):
        self.m = qwen3.Model(npu(), cfg)

    def __del__(self):
        self.m.close()
        ork.lib().ork_npu_set_async(npu().h, 1)


def generator(seed):
    return torch.Generator("cuda").manual_seed(seed)


def ints(g, shape, lo, hi):
    """int8 values in [lo, hi]."""
    return torch.randint(lo, hi + 1, shape, generator=g, device="cuda", dtype=torch.int8)


def weights_f32(g, N, K):
    """f32[N][K] ~ N(0, 0.02), a linear layer as a checkpoint holds it."""
    return torch.randn((N, K), generator=g, device="cuda", dtype=torch.float32).mul_(0.02)


def importance(g, K):
    return torch.rand((K,), generator=g, device="cuda", dtype=torch.float32).mul_(1.5).add_(0.5)


NF4 = [-1.0, -0.6961928009986877, -0.5250730514526367, -0.39491748809814453, -0.28444138169288635, -0.18477343022823334,
       -0.09105003625154495, 0.0, 0.07958029955625534, 0.16093020141124725, 0.24611230194568634, 0.33791524171829224,
       0.44070982933044434, 0.5626170039176941, 0.7229568362236023, 1.0]


def nf4_env(on):
    """ork_i4a8_mm_pack(_im) packs the NF4 codebook where ORK_NF4 is set."""
    if on:
        os.environ["ORK_NF4"] = "1"
    else:
        os.environ.pop("ORK_NF4", None)


def matmul_inputs(case, seed):
    """(A, B): the activations and the weight in the form that its pack takes."""
    g = generator(seed)
    kind, M, K, N = case["kind"], case["M"], case["K"], case["N"]
    if kind == "f16":
        A = torch.randn((M, K), generator=g, device="cuda").half()
        return A, torch.randn((K, N), generator=g, device="cuda").mul_(0.02).half()
    if kind == "i4":
        A = ints(g, (M, K), -8, 7)
        return A, ints(g, (K, N), -8, 7)
    A = ints(g, (M, K), -127, 127)
    return A, weights_f32(g, N, K)


def pack(kind, B, im=None):
    if kind == "i8":
        return Weight(npu().pack_i8_f32(B.cpu().numpy())[0])
    if kind in ("u4", "nf4"):
        nf4_env(kind == "nf4")
        try:
            return Weight(npu().pack_i4a8(B.cpu().numpy(), None if im is None else im.cpu().numpy())[0])
        finally:
            nf4_env(False)
    if kind == "f16":
        return Weight(npu().pack_f16(B.cpu().numpy()))
    return Weight(npu().pack_i4(B.cpu().numpy()))


RUN = {"i8": "ork_i8_mm_run", "u4": "ork_i8_mm_run", "nf4": "ork_i8_mm_run", "f16": "ork_f16_mm_run", "i4": "ork_i4_mm_run"}


# ---- the cases -----------------------------------------------------------------------------------------------------------

def listed():
    return [
        # one decode step's projection (w8a8, FFN width): the smallest call, where the launch counts
        dict(name="gemv_i8", op="mm", kind="i8", M=1, K=2048, N=6144),
        # the reference's calling convention: host rows in, host rows out, a small batch
        dict(name="host_i8_m16", op="host", M=16, K=2048, N=6144),
        # a batch of decode streams on 4-bit weights
        dict(name="u4_m64", op="mm", kind="u4", M=64, K=2048, N=6144),
        # a prompt on fp16 weights
        dict(name="f16_m512", op="mm", kind="f16", M=512, K=2048, N=2048),
        # a prompt on int8 weights, FFN width
        dict(name="i8_m512", op="mm", kind="i8", M=512, K=2048, N=6144),
        # the largest: a batch of long prompts on int8 weights
        dict(name="i8_m4096", op="mm", kind="i8", M=4096, K=4096, N=4096),
        # W4A4
        dict(name="i4_m256", op="mm", kind="i4", M=256, K=4096, N=4096),
        # a ragged long prompt on NF4 weights
        dict(name="nf4_m1000", op="mm", kind="nf4", M=1000, K=2048, N=6144),
        # grouped scales (GPTQ / AWQ-style checkpoints: one scale per 128 k) on a prompt
        dict(name="grouped_i4_m256", op="grouped", kind="i4", M=256, K=4096, N=4096, G=128),
        # loading a model: one FFN projection quantised to int8 and made resident
        dict(name="pack_i8", op="pack", kind="i8", K=2048, N=6144),
        # a long ragged prompt through decoder layers: norms, projections, attention, SwiGLU
        dict(name="prefill_500", op="prefill", M=500, layers=2, vocab=4096, ffn_nf4=0),
        # a chat turn: a short prompt, then greedy decode steps
        dict(name="generate_32", op="generate", M=16, steps=32, layers=4, vocab=151936, ffn_nf4=0),
    ]


def log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["mm"] * 9 + ["chain"] * 2 + ["grouped"] * 3 + ["host", "pack", "prefill", "prefill", "generate"])
    if op == "prefill":
        return dict(op=op, M=log_int(rng, 20, 1000), layers=rng.randint(1, 3), vocab=4096, ffn_nf4=rng.choice([0, 0, 1, 2]))
    if op == "generate":
        return dict(op=op, M=rng.randint(4, 16), steps=rng.randint(8, 32), layers=rng.randint(2, 4), vocab=4096, ffn_nf4=rng.choice([0, 1, 2]))
    if op == "pack":
        return dict(op=op, kind=rng.choice(["i8", "i8", "u4", "nf4"]), K=32 * log_int(rng, 8, 128), N=64 * log_int(rng, 4, 64))
    while True:
        M = log_int(rng, 1, 4096)
        K, N = rng.choice([(2048, 6144), (2048, 2048), (6144, 2048), (4096, 4096), (2048, 1024), (2048, 12288), None, None]) or (
            32 * log_int(rng, 8, 256), 64 * log_int(rng, 4, 192))
        if op == "chain":  # q / k / v or gate / up
            c = dict(op=op, kind=rng.choice(["i8", "i8", "u4"]), M=M, K=K, N=N // 64 * 64, N2=rng.choice([N, max(64, N // 128 * 64)]), tasks=rng.randint(2, 3))
            cols = c["N"] + (c["tasks"] - 1) * c["N2"]
        elif op == "grouped":
            kind = rng.choice(["i4", "i4", "i8"])
            G = rng.choice([g for g in (32, 64, 128, 128, 256, 512) if K % g == 0])
            c, cols = dict(op=op, kind=kind, M=M, K=K, N=N, G=G), N
        elif op == "host":
            M = min(M, 512)
            c, cols = dict(op=op, M=M, K=K, N=N), N
        else:
            c, cols = dict(op=op, kind=rng.choice(["i8", "i8", "f16", "u4", "nf4", "i4"]), M=M, K=K, N=N), N
        if 2.0 * M * K * cols <= MAX_FLOPS and M * K + 4 * K * cols + 4 * M * cols <= MAX_OPERANDS:
            return c


# ---- prepare -------------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    ctx = npu()
    ork.lib().ork_npu_set_async(ctx.h, 1)
    make = {"mm": prepare_mm, "chain": prepare_chain, "grouped": prepare_grouped, "host": prepare_host, "pack": prepare_pack,
            "prefill": prepare_decoder, "generate": prepare_decoder}
    state = make[case["op"]](case, seed)
    state["case"] = case
    torch.cuda.synchronize()  # inputs made on torch's stream, used on the context's
    return state


def prepare_mm(case, seed):
    A, B = matmul_inputs(case, seed)
    w = pack(case["kind"], B)
    out = torch.float32 if case["kind"] == "f16" else torch.int32
    return dict(w=w, A=device_buffer(A.shape, A.dtype, A), C=device_buffer((case["M"], case["N"]), out))


def chain_inputs(case, seed):
    g = generator(seed)
    A = ints(g, (case["M"], case["K"]), -127, 127)
    return A, [weights_f32(g, case["N"] if i == 0 else case["N2"], case["K"]) for i in range(case["tasks"])]


def prepare_chain(case, seed):
    A, Bs = chain_inputs(case, seed)
    A = device_buffer(A.shape, A.dtype, A)
    ws = [pack(case["kind"], B) for B in Bs]
    Cs = [device_buffer((case["M"], B.shape[0]), torch.int32) for B in Bs]
    tasks = ork.tasks(ork.TaskI8, [(w.h, case["M"], A.data_ptr(), C.data_ptr()) for w, C in zip(ws, Cs)])
    return dict(w=ws, A=A, C=Cs, tasks=tasks)


def grouped_inputs(case, seed):
    g = generator(seed)
    M, K, N, G = case["M"], case["K"], case["N"], case["G"]
    hi = 7 if case["kind"] == "i4" else 127
    A, B = ints(g, (M, K), -hi, hi), ints(g, (K, N), -hi, hi)
    scale = lambda shape, s: torch.rand(shape, generator=g, device="cuda").mul_(s).add_(s / 2)  # noqa: E731
    return A, B, scale((M, K // G), 0.02), scale((K // G, N), 0.004)


def prepare_grouped(case, seed):
    A, B, aS, bS = grouped_inputs(case, seed)
    K, N, G = case["K"], case["N"], case["G"]
    B = np.ascontiguousarray(B.cpu().numpy())
    if case["kind"] == "i4":
        w = Weight(ork.lib().ork_i4_mm_pack_grouped(npu().h, K, N, ork.ptr(B), G))
    else:
        w = Weight(npu().pack_i8(B))
        if ork.lib().ork_w_set_group(w.h, G):
            raise RuntimeError("ork_w_set_group")
    put = lambda t: device_buffer(t.shape, t.dtype, t)  # noqa: E731
    return dict(w=w, A=put(A), aS=put(aS), bS=put(bS), C=device_buffer((case["M"], N), torch.float32))


def prepare_host(case, seed):
    A, B = matmul_inputs(dict(case, kind="i8"), seed)
    return dict(w=pack("i8", B), A=A.cpu().numpy(), C=np.zeros((case["M"], case["N"]), np.int32))


def pack_inputs(case, seed):
    g = generator(seed)
    B = weights_f32(g, case["N"], case["K"])
    return B, importance(g, case["K"]) if case["kind"] != "i8" else None


def prepare_pack(case, seed):
    B, im = pack_inputs(case, seed)
    return dict(B=B.cpu().numpy(), im=None if im is None else im.cpu().numpy(), w=None)


def decoder_cfg(case):
    return qwen3.make_cfg(max_ctx=1024 if case["op"] == "prefill" else 512, max_rows=case["M"], ffn_nf4=case["ffn_nf4"],
                          **dict(WIDTHS, layers=case["layers"], vocab=case["vocab"]))


def decoder_inputs(case, seed):
    """The prompt, and the weights one by one (they need not all be held at once)."""
    g = generator(seed)
    cfg = decoder_cfg(case)
    prompt = torch.randint(0, cfg.vocab, (case["M"],), generator=g, device="cuda", dtype=torch.int32)

    def parts():
        yield "linear", -1, 0, weights_f32(g, *qwen3.lin_shape(cfg, -1, 0))
        yield "norm", -1, qwen3.N_ATTN, 1 + weights_f32(g, 1, cfg.hidden)[0]
        for l in range(cfg.layers):
            for i in qwen3.LINEARS:
                yield "linear", l, i, weights_f32(g, *qwen3.lin_shape(cfg, l, i))
            for i, n in ((qwen3.N_ATTN, cfg.hidden), (qwen3.N_FFN, cfg.hidden), (qwen3.N_Q, cfg.head_dim), (qwen3.N_K, cfg.head_dim)):
                yield "norm", l, i, 1 + weights_f32(g, 1, n)[0]

    return cfg, prompt, parts


def prepare_decoder(case, seed):
    cfg, prompt, parts = decoder_inputs(case, seed)
    d = Decoder(cfg)
    for what, l, i, t in parts():
        t = t.cpu().numpy()
        rc = d.m.set_linear(l, i, t) if what == "linear" else d.m.set_norm(l, i, t)
        if rc:
            raise RuntimeError("setting a weight failed: %d" % rc)
    return dict(m=d, prompt=prompt.cpu().numpy())


# ---- run -----------------------------------------------------------------------------------------------------------------

def check(rc):
    if rc:
        raise RuntimeError("the run failed: %d" % rc)


def run(s):
    case, L, h = s["case"], ork.lib(), npu().h
    op = case["op"]
    if op == "mm":
        check(getattr(L, RUN[case["kind"]])(h, s["w"].h, case["M"], s["A"].data_ptr(), s["C"].data_ptr()))
        return s["C"]
    if op == "chain":
        check(L.ork_i8_mm_run_chain(h, case["tasks"], s["tasks"]))
        return s["C"]
    if op == "grouped":
        fn = L.ork_i4_mm_run_grouped if case["kind"] == "i4" else L.ork_i8_mm_run_grouped
        check(fn(h, s["w"].h, case["M"], s["A"].data_ptr(), s["aS"].data_ptr(), s["bS"].data_ptr(), s["C"].data_ptr()))
        return s["C"]
    if op == "host":
        rc, C = npu().run_i8(s["w"].h, s["A"], s["C"])
        check(rc)
        return C
    if op == "pack":
        return run_pack(s, case)
    m = s["m"].m
    check(m.prefill(s["prompt"]))
    if op == "generate":
        check(m.decode(case["steps"]))
        return {"logits": m.last_logits(), "tokens": m.tokens()}
    return {"logits": m.last_logits()}


def run_pack(s, case):
    s["w"] = None  # the weight of the pass before
    if case["kind"] == "i8":
        h, bs = npu().pack_i8_f32(s["B"])
    else:
        nf4_env(case["kind"] == "nf4")
        try:
            h, bs = npu().pack_i4a8(s["B"], s["im"])
        finally:
            nf4_env(False)
    s["w"] = Weight(h)
    panels, KB, kind, lut = ctypes.c_void_p(), ctypes.c_int(), ctypes.c_int(), (ctypes.c_uint32 * 4)()
    check(ork.lib().ork_w_device_panels(h, ctypes.byref(panels), ctypes.byref(KB), ctypes.byref(kind), lut))
    n = case["N"] // 16 * KB.value * 1024
    return {"bscale": bs, "panels": torch.as_tensor(_Memory(panels.value, (n,), torch.uint8, False), device="cuda")}


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------

B_BYTES = {"i8": 1.0, "f16": 2.0, "u4": 0.5, "nf4": 0.5, "i4": 0.5}


def layer_macs(ffn=WIDTHS["ffn"]):
    H, QD, KVD = WIDTHS["hidden"], WIDTHS["heads"] * WIDTHS["head_dim"], WIDTHS["kv_heads"] * WIDTHS["head_dim"]
    return H * QD + 2 * H * KVD + QD * H, 3 * H * ffn


def work(case):
    op = case["op"]
    if op in ("mm", "host"):
        kind, M, K, N = case.get("kind", "i8"), case["M"], case["K"], case["N"]
        a = 2 if kind == "f16" else 1
        return {"bytes": a * M * K + B_BYTES[kind] * K * N + 4 * M * N, "flops": 2.0 * M * K * N}
    if op == "chain":
        M, K, cols = case["M"], case["K"], case["N"] + (case["tasks"] - 1) * case["N2"]
        return {"bytes": M * K + B_BYTES[case["kind"]] * K * cols + 4 * M * cols, "flops": 2.0 * M * K * cols}
    if op == "grouped":
        M, K, N, Sk = case["M"], case["K"], case["N"], case["K"] // case["G"]
        return {"bytes": M * K + B_BYTES[case["kind"]] * K * N + 4 * M * N + 4 * Sk * (M + N), "flops": 2.0 * M * K * N}
    if op == "pack":
        K, N = case["K"], case["N"]
        return {"bytes": 4 * K * N + B_BYTES[case["kind"]] * K * N + 4 * N, "flops": 2.0 * K * N}
    att, ffn = layer_macs()
    ffn_b = ffn * (0.5 if case["ffn_nf4"] else 1.0)
    L, V, H = case["layers"], case["vocab"], WIDTHS["hidden"]
    QD, KVD = WIDTHS["heads"] * WIDTHS["head_dim"], WIDTHS["kv_heads"] * WIDTHS["head_dim"]
    M = case["M"]
    weights = L * (att + ffn_b) + V * H
    flops = 2.0 * (M * L * (att + ffn) + V * H) + L * 4.0 * QD * M * (M + 1) / 2
    total = weights + L * 2 * 4 * M * KVD + 2 * M * H + 4 * V
    if op == "generate":
        S = case["steps"]
        keys = sum(M + i + 1 for i in range(S))
        total += S * (weights + 4 * V) + L * 2 * 4 * KVD * keys
        flops += 2.0 * S * (L * (att + ffn) + V * H) + L * 4.0 * QD * keys
    return {"bytes": float(total), "flops": flops}


# ---- how exactly -----------------------------------------------------------------------------------------------------------

def tolerance(case):
    op = case["op"]
    if op == "mm" and case["kind"] == "f16":
        return {"rel": 2e-6, "max": 2e-5}  # fp16 products summed in fp32: the order of the sums
    if op == "grouped":
        return {"rel": 2e-6, "max": 2e-5}  # exact int32 groups, scaled and summed in fp32
    if op in ("prefill", "generate"):
        # Rows are quantised to int8 before every matmul: a last bit that moves one code moves many in the next row, a
        # whole step each. Against 64 bits one layer's logits are 1.5e-5 off where no code moved and 0.02 to 0.03 where
        # one did, two layers' 0.02 to 0.045: the bound is the order of one layer's.
        return {"rel": 0.03, "max": 0.3}
    return "exact"                         # integers, codes and their scales


def quant_rows(y):
    """Per-row int8: a = clamp(rint(y / s)), s = max|y| / 127 (1 for a zero row)."""
    s = y.abs().amax(-1, keepdim=True) / 127
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(y / s), -127, 127), s


def quant_i8(B):
    """(codes f64[N][K], scale f32[N]) of ork_i8_mm_pack_f32: q = clamp(rint(w * (127 / mx))), in fp32."""
    mx = B.abs().amax(1).clamp_min(1e-9)
    q = torch.clamp(torch.round(B * (127.0 / mx)[:, None]), -127, 127)
    return q.double(), mx / 127.0


def quant_4(B, nf4):
    """(codes that the weight multiplies with f64[N][K], scale f32[N]) of ork_i4a8_mm_pack without an importance vector."""
    mx = B.abs().amax(1).clamp_min(1e-9)
    if not nf4:
        sc = mx / 7.0
        return torch.clamp(torch.round(B * (1.0 / sc)[:, None]), -7, 7).double(), sc
    lev = torch.tensor(NF4, device=B.device, dtype=torch.float32)
    wn = B * (1.0 / mx)[:, None]
    hi = torch.searchsorted(lev, wn.clamp(-1, 1).contiguous()).clamp(0, 15)
    lo = (hi - 1).clamp_min(0)
    t = torch.where(hi > lo, (wn - lev[lo]) / (lev[hi] - lev[lo]).clamp_min(1e-30), torch.zeros_like(wn))
    return torch.round(lev * 127)[torch.where(t >= 0.5, hi, lo)].double(), mx / 127.0


def codes(kind, B):
    """f64[K][N] that the resident weight multiplies with."""
    if kind == "i8":
        return quant_i8(B)[0].t()
    if kind in ("u4", "nf4"):
        return quant_4(B, kind == "nf4")[0].t()
    return B.double()


def exact(case, seed):
    op = case["op"]
    if op in ("mm", "host"):
        c = dict(case, kind=case.get("kind", "i8"))
        A, B = matmul_inputs(c, seed)
        r = A.double() @ codes(c["kind"], B)
        return r if c["kind"] == "f16" else r.cpu().numpy().astype(np.int32) if op == "host" else r.to(torch.int32)
    if op == "chain":
        A, Bs = chain_inputs(case, seed)
        return [(A.double() @ codes(case["kind"], B)).to(torch.int32) for B in Bs]
    if op == "grouped":
        A, B, aS, bS = grouped_inputs(case, seed)
        G = case["G"]
        C = torch.zeros((case["M"], case["N"]), dtype=torch.float64, device="cuda")
        for g in range(case["K"] // G):
            P = A[:, g * G:(g + 1) * G].double() @ B[g * G:(g + 1) * G].double()
            C += P * aS[:, g:g + 1].double() * bS[g].double()
        return C
    if op == "pack":
        if case["kind"] != "i8":
            return None  # the clip search over the importance vector
        B, _ = pack_inputs(case, seed)
        q, bs = quant_i8(B)
        return {"bscale": bs.double().cpu().numpy(), "panels": i8_panels(q, case["K"], case["N"])}
    if op == "generate":
        return None  # greedy: a near-tie anywhere changes every token after it
    return exact_prefill(case, seed)


def i8_panels(q, K, N):
    """Resident int8 panels: 1 KiB per (16 columns, 64 k); lane l: column l % 16, k-group l / 16; byte i: k = 16 group + i."""
    KB = -(-K // 64)
    p = torch.zeros((N, KB * 64), dtype=torch.int8, device=q.device)
    p[:, :K] = q.to(torch.int8)
    return p.view(N // 16, 16, KB, 4, 16).permute(0, 2, 3, 1, 4).contiguous().view(-1).view(torch.uint8)


def exact_prefill(case, seed):
    cfg, prompt, parts = decoder_inputs(case, seed)
    H, NH, NKV, HD, eps = cfg.hidden, cfg.heads, cfg.kv_heads, cfg.head_dim, cfg.eps
    M = case["M"]
    lin, norm = {}, {}
    for what, l, i, t in parts():
        if what == "norm":
            norm[l, i] = t.double()
        elif l >= 0 and i in (qwen3.WG, qwen3.WU, qwen3.WD) and cfg.ffn_nf4:
            lin[l, i] = quant_4(t, cfg.ffn_nf4 == 1)
        else:
            lin[l, i] = quant_i8(t)
            if l < 0:
                emb = t.half()[prompt.long()]

    def rms(x, w):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w

    def mul(a, s, l, i):
        q, ws = lin[l, i]
        return (a @ q.t()) * s * ws.double()

    inv = cfg.rope_theta ** (-2.0 * torch.arange(HD // 2, dtype=torch.float64, device="cuda") / HD)
    ang = torch.arange(M, dtype=torch.float64, device="cuda")[:, None] * inv
    cos, sin = ang.cos().float().double()[:, None], ang.sin().float().double()[:, None]

    def rope(v):
        a, b = v[..., :HD // 2], v[..., HD // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    x = emb.double()
    mask = torch.ones((M, M), dtype=torch.bool, device="cuda").triu(1)
    for l in range(cfg.layers):
        a, s = quant_rows(rms(x, norm[l, qwen3.N_ATTN]))
        q = rope(rms(mul(a, s, l, qwen3.WQ).view(M, NH, HD), norm[l, qwen3.N_Q]))
        k = rope(rms(mul(a, s, l, qwen3.WK).view(M, NKV, HD), norm[l, qwen3.N_K]))
        v = mul(a, s, l, qwen3.WV).view(M, NKV, HD)
        out = torch.empty((M, NH, HD), dtype=torch.float64, device="cuda")
        for hd in range(NH):
            g = hd // (NH // NKV)
            sc = (q[:, hd] @ k[:, g].t().contiguous()) / math.sqrt(HD)
            out[:, hd] = torch.softmax(sc.masked_fill(mask, -math.inf), -1) @ v[:, g]
        a, s = quant_rows(out.view(M, NH * HD))
        x = x + mul(a, s, l, qwen3.WO)
        a, s = quant_rows(rms(x, norm[l, qwen3.N_FFN]))
        gt, up = mul(a, s, l, qwen3.WG), mul(a, s, l, qwen3.WU)
        a, s = quant_rows(gt / (1 + torch.exp(-gt)) * up)
        x = x + mul(a, s, l, qwen3.WD)
    a, s = quant_rows(rms(x[-1:], norm[-1, qwen3.N_ATTN]))
    return {"logits": mul(a, s, -1, 0)[0].cpu().numpy()}
