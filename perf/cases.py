"""The quantized matmul path's performance cases: what a program does with this library, per entry
point and regime, with inputs in the formats of bybylang_amd/synth.py.

Kinds
  q4      byhip_q4_matmul on resident weights: the decode vector, a prefill chunk of fp16
          activations, the session's fp32 activations, and weights with a zero point per group.
  layer   the decoder layer's four Q4 projections (QKV, O, gate+up, down) for a batch of sequences.
  fused   the same layer for one token through sessionMatmulQ4Fused (norm and residual inside).
  vm_q4   a micro-VM program of one OP_Q4_COOP_GEMM (or OP_Q4_GEMV) over the slots.
  fp4km   sessionFp4GemmTensorCore: fp32 activations, FP4-KM weights, a 272-float decode table.
  f16     sessionF16GemmTile: fp32 activations, half weights.
  mxfp4   byhip_mxfp4_gemm: both operands MXFP4, bf16 output.

Buffers are torch tensors whose pointers go to the C ABI; the outputs are the state's own.
"""
import ctypes as C
import math

import numpy as np
import torch

from bybylang_amd import _abi
from bybylang_amd import device as dev
from bybylang_amd import gpubackend as gb

F32, F16, BF16 = _abi.F32, _abi.F16, _abi.BF16
CODE = {"f32": F32, "f16": F16, "bf16": BF16}
TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
SIZE = {"f32": 4, "f16": 2, "bf16": 2}
E2M1 = [0, .5, 1, 1.5, 2, 3, 4, 6, -0.0, -.5, -1, -1.5, -2, -3, -4, -6]
EPS = 1e-5


def listed():
    return [
        # one token, one projection: the smallest call a decode loop makes (benchmark config 1)
        {"name": "q4_decode_f16", "kind": "q4", "M": 1, "K": 4096, "N": 14336, "group": 32, "x": "f16", "y": "f16", "zeros": "one"},
        # one token through a whole layer of resident weights, at the session's fp32
        {"name": "q4_fused_layer", "kind": "fused", "K": 4096, "kv": 1024, "F": 14336, "group": 32},
        # one decode step of 32 sequences: the layer's four projections (benchmark config 4)
        {"name": "q4_layer_batch", "kind": "layer", "M": 32, "K": 4096, "kv": 1024, "F": 14336, "group": 32},
        # a compiled micro-kernel's Q4 op, fp32 in and out (benchmark config 0)
        {"name": "vm_q4_coop", "kind": "vm_q4", "M": 16, "K": 4096, "N": 4096, "group": 32, "op": "coop"},
        # a prompt chunk through a projection, fp16 (benchmark config 2)
        {"name": "q4_prefill_f16", "kind": "q4", "M": 512, "K": 4096, "N": 4096, "group": 32, "x": "f16", "y": "f16", "zeros": "one"},
        # the same at the session's fp32, a prompt of no round length
        {"name": "q4_prefill_f32", "kind": "q4", "M": 509, "K": 4096, "N": 14336, "group": 32, "x": "f32", "y": "f32", "zeros": "one"},
        # asymmetric checkpoints: group 128 with a zero point per group
        {"name": "q4_zeros_f16", "kind": "q4", "M": 251, "K": 4096, "N": 11008, "group": 128, "x": "f16", "y": "f16", "zeros": "group"},
        # FP4-KM decode with an E2M1 / E8M0 table, as MXFP4 checkpoints have it
        {"name": "fp4km_decode", "kind": "fp4km", "M": 1, "K": 4096, "N": 14336, "table": "mx"},
        # FP4-KM prefill with the table of the reference's tests
        {"name": "fp4km_prefill", "kind": "fp4km", "M": 512, "K": 4096, "N": 4096, "table": "ref"},
        # half weights, a short prompt
        {"name": "f16_tile", "kind": "f16", "M": 130, "K": 4096, "N": 6144},
        # MXFP4 activations and weights: a batch of decode rows, N of no whole tile
        {"name": "mxfp4_batch", "kind": "mxfp4", "M": 47, "K": 8192, "N": 8200},
        # MXFP4 prefill, the largest product of the benchmark (config 3)
        {"name": "mxfp4_prefill", "kind": "mxfp4", "M": 2048, "K": 8192, "N": 8192},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _n(rng, lo, hi):
    """Output columns: mostly multiples of 64, now and then any number."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.3 else max(lo, n // 64 * 64)


def draw(rng):
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= 1.2e8:  # the layer cases are the largest listed in bytes
            return case


def _draw(rng):
    kind = rng.choice(["q4", "q4", "q4", "fused", "layer", "vm_q4", "fp4km", "fp4km", "f16", "mxfp4"])
    group = rng.choice([32, 32, 64, 128])
    k = 128 * _log(rng, 8, 112)  # 1024 .. 14336
    if kind == "fused":
        hid = 256 * rng.randint(8, 24)
        return {"kind": kind, "K": hid, "kv": rng.choice([hid, hid // 4, hid // 8]), "F": 128 * rng.randint(hid // 50, hid // 36), "group": group}
    if kind == "layer":
        hid = 256 * rng.randint(8, 20)
        return {"kind": kind, "M": _log(rng, 2, 64), "K": hid, "kv": rng.choice([hid, hid // 4]), "F": 128 * rng.randint(hid // 50, hid // 36), "group": group}
    if kind == "vm_q4":
        op = rng.choice(["coop", "gemv"])
        return {"kind": kind, "M": 1 if op == "gemv" else _log(rng, 2, 64), "K": k if k <= 8192 else 8192, "N": _n(rng, 512, 8192), "group": group, "op": op}
    n = _n(rng, 512, 14336)
    if kind == "q4":
        x = rng.choice(["f16", "f16", "f32"])
        m = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 1024)])
        y = "f32" if x == "f32" else rng.choice(["f16", "f16", "bf16"])
        zeros = "group" if m > 8 and rng.random() < 0.3 else "one"
        while 2 * m * k * n > 5.5e10:
            m = max(1, m // 2)
        return {"kind": kind, "M": m, "K": k, "N": n, "group": group, "x": x, "y": y, "zeros": zeros}
    if kind == "mxfp4":
        m = rng.choice([_log(rng, 1, 64), _log(rng, 65, 2048)])
        return {"kind": kind, "M": m, "K": min(k, 8192), "N": min(n, 8192)}
    m = rng.choice([1, _log(rng, 2, 32), _log(rng, 33, 512)])
    while 2 * m * k * n > 1.7e10:
        m = max(1, m // 2)
    if kind == "fp4km":
        return {"kind": kind, "M": m, "K": k, "N": n, "table": rng.choice(["mx", "ref"])}
    return {"kind": kind, "M": m, "K": k, "N": min(n, 8192)}


# ── inputs ──────────────────────────────────────────────────────────────────────────────────


class Gen:
    """Seeded inputs on the GPU, in the distributions of bybylang_amd/synth.py."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)

    def normal(self, *shape, dtype="f32"):
        return torch.randn(*shape, generator=self.g, device="cuda").to(TORCH[dtype])

    def ints(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.uint8)

    def q4(self, K, N, group, zeros="one"):
        """Nibble rows (two codes per byte, even k low), fp16-valued scales and zeros as fp32."""
        ng = K // group
        q = {"wq": self.ints(0, 256, N, K // 2), "K": K, "N": N, "group": group}
        q["s"] = (self.normal(N, ng).mul_(0.02).abs_() + 1e-4).half().float()
        if zeros == "one":
            q["z"] = torch.full((N, ng), 8.0, device="cuda")
        else:
            q["z"] = (8 + 1.5 * self.normal(N, ng)).round_().clamp_(0, 15)
        return q

    def fp4(self, R, K, ref_table=False):
        """R rows of an FP4-KM operand: nibbles [R, K/2], then one scale byte per 32 values."""
        nib = self.ints(0, 256, R, K // 2)
        sb = self.ints(0, 256, R, K // 32) if ref_table else self.ints(123, 130, R, K // 32)
        return torch.cat([nib.reshape(-1), sb.reshape(-1)])


def table(kind):
    """The decode table: E2M1, then the scales: 2^(e - 127), or (1 + i mod 13) / 64."""
    i = np.arange(256)
    with np.errstate(over="ignore"):
        s = np.ldexp(np.float32(1), i - 127) if kind == "mx" else (1 + i % 13) / 64
    return np.concatenate([np.array(E2M1), s]).astype(np.float32)


class Weights:
    """Resident Q4 weights; freed with the object."""

    def __init__(self, q):
        torch.cuda.synchronize()  # the library copies on its own stream
        h = C.c_void_p()
        _abi.check(_abi.load().byhip_q4_resident_from_device(
            q["wq"].data_ptr(), 0, q["s"].data_ptr(), q["z"].data_ptr(), q["K"], q["N"], q["group"],
            q["K"] // q["group"], C.byref(h)))
        self.handle = h.value

    def __del__(self):
        if getattr(self, "handle", None):
            _abi.load().byhip_q4_resident_free(self.handle)


class Table:
    """A decode table uploaded through the session; freed with the object."""

    def __init__(self, t):
        self.h = gb.sessionUpload(gb.gbHip, t)

    def __del__(self):
        if getattr(self, "h", None):
            gb.sessionFree(gb.gbHip, self.h)


def _handle(t):
    return gb.SessionHandle(gb.gbHip, t.data_ptr(), t.numel() * t.element_size())


def _resident(q):
    w = Weights(q)
    return w, gb.ResidentWeightHandle(gb.gbHip, q["K"], q["N"], q["group"], q["K"] // q["group"], 0, w.handle)


def _layer_shapes(c):
    """(K, N) of QKV, O, gate+up and down."""
    return [(c["K"], c["K"] + 2 * c["kv"]), (c["K"], c["K"]), (c["K"], 2 * c["F"]), (c["F"], c["K"])]


def _inputs(c, seed):
    """The case's host-side picture: plain tensors, without anything of the library."""
    g = Gen(seed)
    k = c["kind"]
    if k == "q4":
        return {"x": g.normal(c["M"], c["K"], dtype=c["x"]), "w": g.q4(c["K"], c["N"], c["group"], c["zeros"])}
    if k == "layer":
        return {"x": [g.normal(c["M"], kk, dtype="f16") for kk, _ in _layer_shapes(c)],
                "w": [g.q4(kk, n, c["group"]) for kk, n in _layer_shapes(c)]}
    if k == "fused":
        H, F, kv, gr = c["K"], c["F"], c["kv"], c["group"]
        names = {"q": (H, H), "k": (H, kv), "v": (H, kv), "o": (H, H), "gate": (H, F), "up": (H, F), "down": (F, H)}
        return {"x": g.normal(H), "att": g.normal(H), "g1": 1 + 0.1 * g.normal(H), "g2": 1 + 0.1 * g.normal(H),
                "w": {n: g.q4(a, b, gr) for n, (a, b) in names.items()}}
    if k == "vm_q4":
        return {"x": g.normal(c["M"], c["K"]), "w": g.q4(c["K"], c["N"], c["group"])}
    if k == "fp4km":
        return {"x": g.normal(c["M"], c["K"]), "w": g.fp4(c["N"], c["K"], c["table"] == "ref"), "t": table(c["table"])}
    if k == "f16":
        return {"x": g.normal(c["M"], c["K"]), "w": g.normal(c["N"], c["K"]).mul_(0.05).half()}
    return {"x": g.fp4(c["M"], c["K"]), "w": g.fp4(c["N"], c["K"])}


def prepare(case, seed):
    c = dict(case)
    dev.init(0)
    torch.cuda.init()
    s = {"c": c, "kind": c["kind"], "lib": _abi.load()}
    i = _inputs(c, seed)
    empty = lambda *shape, dtype="f32": torch.empty(*shape, device="cuda", dtype=TORCH[dtype])  # noqa: E731
    k = c["kind"]
    if k == "q4":
        s["x"], s["w"], s["y"] = i["x"], Weights(i["w"]), empty(c["M"], c["N"], dtype=c["y"])
        s["call"] = (s["x"].data_ptr(), CODE[c["x"]], s["w"].handle, s["y"].data_ptr(), CODE[c["y"]], c["M"])
    elif k == "layer":
        s["x"], s["w"] = i["x"], [Weights(q) for q in i["w"]]
        s["y"] = [empty(c["M"], n, dtype="f16") for _, n in _layer_shapes(c)]
        s["calls"] = [(x.data_ptr(), F16, w.handle, y.data_ptr(), F16, c["M"]) for x, w, y in zip(s["x"], s["w"], s["y"])]
    elif k == "fused":
        s["w"] = {n: _resident(q) for n, q in i["w"].items()}
        s["t"] = {n: i[n] for n in ("x", "att", "g1", "g2")}
        s["y"] = {n: empty(m) for n, m in (("q", c["K"]), ("k", c["kv"]), ("v", c["kv"]), ("h", c["K"]), ("act", c["F"]), ("unused", c["F"]), ("out", c["K"]))}
        s["h"] = {n: _handle(t) for n, t in list(s["t"].items()) + list(s["y"].items())}
    elif k == "vm_q4":
        N, K, ng = c["N"], c["K"], c["K"] // c["group"]
        s["x"], s["y"] = i["x"], empty(c["M"], N)
        pad = (-(N * (K // 2))) % 4
        s["blob"] = torch.cat([i["w"]["wq"].reshape(-1), torch.zeros(pad, dtype=torch.uint8, device="cuda"),
                               i["w"]["s"].reshape(-1).view(torch.uint8), i["w"]["z"].reshape(-1).view(torch.uint8)])
        op = 0xAA if c["op"] == "coop" else 0xAB
        s["words"] = np.array([op, c["M"], K, N, c["group"], ng, 0x01], dtype=np.uint32)
        s["h"] = (_handle(s["y"]), _handle(s["blob"]), _handle(s["blob"]), _handle(s["x"]))
    elif k == "fp4km":
        s["x"], s["blob"], s["y"] = i["x"], i["w"], empty(c["M"], c["N"])
        s["t"] = Table(i["t"])
        s["h"] = (_handle(s["x"]), _handle(s["blob"]), s["t"].h, _handle(s["y"]))
    elif k == "f16":
        s["x"], s["w"], s["y"] = i["x"], i["w"], empty(c["M"], c["N"])
        s["h"] = (_handle(s["x"]), _handle(s["w"]), _handle(s["y"]))
    else:
        s["x"], s["w"], s["y"] = i["x"], i["w"], empty(c["M"], c["N"], dtype="bf16")
        s["call"] = (s["x"].data_ptr(), s["w"].data_ptr(), s["y"].data_ptr(), BF16, c["M"], c["K"], c["N"])
    torch.cuda.synchronize()  # the inputs are made on torch's stream, the library has its own
    return s


def _done(ok):
    if not ok:
        raise RuntimeError("not taken: " + gb.sessionGetLastError(gb.gbHip))


def run(s):
    k, c = s["kind"], s["c"]
    if k == "q4":
        _abi.check(s["lib"].byhip_q4_matmul(*s["call"]))
    elif k == "layer":
        for call in s["calls"]:
            _abi.check(s["lib"].byhip_q4_matmul(*call))
    elif k == "fused":
        h, w = s["h"], {n: v[1] for n, v in s["w"].items()}
        f = gb.sessionMatmulQ4Fused
        _done(f(gb.gbHip, 0, h["x"], [w["q"], w["k"], w["v"]], [h["q"], h["k"], h["v"]], None, False, h["g1"], EPS, True))
        _done(f(gb.gbHip, 0, h["att"], [w["o"]], [h["h"]], h["x"], True))
        _done(f(gb.gbHip, 1, h["h"], [w["gate"], w["up"]], [h["act"], h["unused"]], None, False, h["g2"], EPS, True))
        _done(f(gb.gbHip, 0, h["act"], [w["down"]], [h["out"]], h["h"], True))
        return {n: s["y"][n] for n in ("q", "k", "v", "h", "act", "out")}
    elif k == "vm_q4":
        _done(gb.sessionEncTileProgram(gb.gbHip, s["words"], *s["h"]))
    elif k == "fp4km":
        _done(gb.sessionFp4GemmTensorCore(gb.gbHip, *s["h"], c["M"], c["K"], c["N"]))
    elif k == "f16":
        _done(gb.sessionF16GemmTile(gb.gbHip, *s["h"], c["M"], c["K"], c["N"]))
    else:
        _abi.check(s["lib"].byhip_mxfp4_gemm(*s["call"]))
    return s["y"]


# ── work and tolerance ──────────────────────────────────────────────────────────────────────


def _q4_work(M, K, N, group, xs, ys, zeros="one", slot=False):
    """Nibbles, a scale per group (fp16 as the checkpoint's, fp32 in a slot), zeros where there is
    one per group, activations and outputs."""
    ng = N * (K // group)
    b = N * K // 2 + ng * (4 if slot else 2) + (ng * 4 if slot or zeros == "group" else 0) + M * K * xs + M * N * ys
    return b, 2 * M * K * N


def work(c):
    k = c["kind"]
    if k == "q4":
        b, f = _q4_work(c["M"], c["K"], c["N"], c["group"], SIZE[c["x"]], SIZE[c["y"]], c["zeros"])
    elif k == "layer":
        parts = [_q4_work(c["M"], kk, n, c["group"], 2, 2) for kk, n in _layer_shapes(c)]
        b, f = sum(p[0] for p in parts), sum(p[1] for p in parts)
    elif k == "fused":
        # the layer's matrices, x, att, h and act in, both gammas, q, k, v, h, act and out
        H, F, kv = c["K"], c["F"], c["kv"]
        parts = [_q4_work(1, kk, n, c["group"], 0, 0) for kk, n in _layer_shapes(c)]
        b, f = sum(p[0] for p in parts) + 4 * (2 * H + 2 * H + H + 2 * kv + H + F + H), sum(p[1] for p in parts)
    elif k == "vm_q4":
        b, f = _q4_work(c["M"], c["K"], c["N"], c["group"], 4, 4, slot=True)
    else:
        M, K, N = c["M"], c["K"], c["N"]
        f = 2 * M * K * N
        fp4 = K // 2 + K // 32
        b = {"fp4km": N * fp4 + 1088 + 4 * M * K + 4 * M * N, "f16": 2 * N * K + 4 * M * K + 4 * M * N,
             "mxfp4": (M + N) * fp4 + 2 * M * N}[k]
    return {"bytes": b, "flops": f}


def tolerance(c):
    """About four times the error against exact() that the formats show: an fp16 output with the
    weights rounded once to fp16 2.8e-4, a bf16 output 1.8e-3, fp32 sums 2e-7 to 1.3e-6, the fused
    layer, whose last outputs carry the errors of the first, 2e-6."""
    k = c["kind"]
    if k == "layer" or (k == "q4" and c["y"] == "f16"):
        return {"rel": 1.1e-3}
    if k == "mxfp4" or (k == "q4" and c["y"] == "bf16"):
        return {"rel": 7e-3}
    return {"rel": 8e-6 if k == "fused" else 5e-6}


# ── the exact results, in 64 bits ───────────────────────────────────────────────────────────


def _q4_exact(q):
    N, K, group = q["N"], q["K"], q["group"]
    codes = torch.stack([q["wq"] & 15, q["wq"] >> 4], dim=2).reshape(N, K // group, group).double()
    return ((codes - q["z"].double()[:, :, None]) * q["s"].double()[:, :, None]).reshape(N, K)


def _fp4_exact(blob, R, K, t):
    t = torch.from_numpy(t).cuda().double()
    nib = blob[: R * (K // 2)].reshape(R, K // 32, 16)
    sb = blob[R * (K // 2):].reshape(R, K // 32).long()
    codes = torch.cat([nib & 15, nib >> 4], dim=2).long()
    return (t[codes] * t[16 + sb][:, :, None]).reshape(R, K)


def exact(case, seed):
    c = dict(case)
    i = _inputs(c, seed)
    k = c["kind"]
    if k == "layer":
        return [x.double() @ _q4_exact(w).T for x, w in zip(i["x"], i["w"])]
    if k == "fused":
        w = {n: _q4_exact(q) for n, q in i["w"].items()}
        d = {n: i[n].double() for n in ("x", "att", "g1", "g2")}
        norm = lambda v, g: v * g / torch.sqrt((v * v).mean() + EPS)  # noqa: E731
        a = norm(d["x"], d["g1"])
        h = w["o"] @ d["att"] + d["x"]
        b = norm(h, d["g2"])
        gate = w["gate"] @ b
        act = gate / (1 + torch.exp(-gate)) * (w["up"] @ b)
        return {"q": w["q"] @ a, "k": w["k"] @ a, "v": w["v"] @ a, "h": h, "act": act, "out": w["down"] @ act + h}
    if k in ("q4", "vm_q4"):
        return i["x"].double() @ _q4_exact(i["w"]).T
    if k == "fp4km":
        return i["x"].double() @ _fp4_exact(i["w"], c["N"], c["K"], i["t"]).T
    if k == "f16":
        return i["x"].double() @ i["w"].double().T
    t = table("mx")
    return _fp4_exact(i["x"], c["M"], c["K"], t) @ _fp4_exact(i["w"], c["N"], c["K"], t).T
