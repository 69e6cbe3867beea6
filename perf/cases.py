"""Timing cases: the quantized matrix products and decodes that a user of
flatrun_amd runs, through its public entry points.

Five kinds of call:
  matvec   device.gemv: `rows` activations against one resident weight (one
           row: a decode step; a few: several sequences or drafted tokens
           together; many: a prompt), fp32 activations and results
  block    layer.DecoderProjections: the seven projections and the SwiGLU
           activation of one decoder block (one row: decode; many: prefill)
  gemm     device.gemm_bf16_group: weights that share bf16 activations
  dequant  device.dequant / device.dequant_f16: a whole weight decoded
  host     NativeBackend.matmul_*: activations and results in host arrays,
           the weight uploaded once

Weights are GGUF blocks with codes concentrated near zero, as quantized
normal weights have them; activations have a per-channel spread with a few
large channels.
"""

from __future__ import annotations

import math

import numpy as np
import torch

import flatrun_amd
from flatrun_amd import device
from flatrun_amd.layer import DecoderProjections

BLOCK = {"Q8_0": (34, 32), "Q4_K": (144, 256), "Q5_K": (176, 256), "Q6_K": (210, 256), "Q1_0": (18, 128)}
UNIT = {"Q8_0": 128, "Q4_K": 256, "Q5_K": 256, "Q6_K": 256, "Q1_0": 128}      # k of every kind of call


def listed() -> list[dict]:
    return [
        # The smallest calls: one projection of a 0.5B model in Q8_0 for one
        # token, and a 1-bit model's square projection; launch and latency.
        dict(name="decode_small_q8_0", kind="matvec", qtype="Q8_0", n=4864, k=896, rows=1),
        dict(name="decode_q1_0", kind="matvec", qtype="Q1_0", n=4096, k=4096, rows=1),
        # One token through a 7B model's MLP output projection: the headline.
        dict(name="decode_q4_k", kind="matvec", qtype="Q4_K", n=3584, k=18944, rows=1),
        # The same step in a file kept at 5 bits.
        dict(name="decode_q5_k", kind="matvec", qtype="Q5_K", n=14336, k=4096, rows=1),
        # The vocabulary projection of every generated token.
        dict(name="lm_head_q6_k", kind="matvec", qtype="Q6_K", n=152064, k=3584, rows=1),
        # Sixteen sequences decoded together (or drafted tokens verified).
        dict(name="batch16_q4_k", kind="matvec", qtype="Q4_K", n=4096, k=14336, rows=16),
        # A short prompt on a 5-bit file, an odd number of tokens.
        dict(name="prompt_q5_k", kind="matvec", qtype="Q5_K", n=14336, k=4096, rows=97),
        # A whole 8B decoder block for one token, 4-bit with 6-bit v and down.
        dict(name="block_decode", kind="block", hidden=4096, inter=14336, q_n=4096, kv_n=1024, main="Q4_K",
             more="Q6_K", rows=1),
        # The same for a prompt on a 7B block, fp32 activations.
        dict(name="block_prefill", kind="block", hidden=3584, inter=18944, q_n=3584, kv_n=512, main="Q4_K",
             more="Q6_K", rows=333),
        # Gate and up of a prompt with bf16 activations.
        dict(name="prefill_bf16", kind="gemm", qtypes="Q4_K,Q4_K", ns="14336,14336", k=4096, rows=512),
        # A weight decoded to half precision for a caller that multiplies itself.
        dict(name="dequant_q4_k_f16", kind="dequant", qtype="Q4_K", n=18944, k=3584, drop=0, out="f16"),
        # The drop-in call of a Python runtime: host activations and results.
        dict(name="host_q4_k", kind="host", qtype="Q4_K", n=4096, k=4096, rows=1),
    ]


MAX_FLOPS, MAX_BYTES = 1.5e11, 4.4e8         # below the largest listed cases


def _log(rng, lo: float, hi: float) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _rows(rng, most: int) -> int:
    band = rng.choice([(1, 1), (1, 1), (2, 8), (9, 64), (65, 512)])
    return max(1, min(most, _log(rng, *band)))


def draw(rng) -> dict:
    kind = rng.choice(["matvec"] * 6 + ["block"] * 2 + ["gemm", "dequant", "host"])
    if kind in ("matvec", "host"):
        q = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q6_K", "Q8_0", "Q1_0"])
        k = UNIT[q] * max(1, _log(rng, 512, 24576) // UNIT[q])
        n = min(_log(rng, 200, 65536), int(MAX_BYTES / (k * BLOCK[q][0] / BLOCK[q][1])))
        if kind == "host":
            return dict(kind=kind, qtype=q, n=min(n, 32768), k=k, rows=rng.choice([1, 1, 3, 17]))
        return dict(kind=kind, qtype=q, n=n, k=k, rows=_rows(rng, max(1, int(MAX_FLOPS / (2.0 * n * k)))))
    if kind == "block":
        hidden = 256 * max(4, _log(rng, 1024, 5120) // 256)
        inter = 256 * (_log(rng, 2 * hidden, 5.3 * hidden) // 256)
        main, more = rng.choice([("Q4_K", "Q6_K"), ("Q4_K", "Q4_K"), ("Q5_K", "Q6_K"), ("Q8_0", "Q8_0")])
        per_row = 2.0 * hidden * (2.5 * hidden + 3 * inter)
        return dict(kind=kind, hidden=hidden, inter=inter, q_n=hidden, kv_n=64 * rng.randint(2, hidden // 64),
                    main=main, more=more, rows=_rows(rng, min(512, max(1, int(MAX_FLOPS / per_row)))))
    if kind == "gemm":
        count = rng.randint(1, 4)
        qs = [rng.choice(["Q4_K", "Q4_K", "Q6_K", "Q8_0"]) for _ in range(count)]
        k = 256 * max(2, _log(rng, 512, 16384) // 256)
        ns = [_log(rng, 256, 16384) for _ in range(count)]
        rows = min(_log(rng, 32, 1024), max(1, int(1.2e11 / (2.0 * k * sum(ns)))))
        return dict(kind=kind, qtypes=",".join(qs), ns=",".join(map(str, ns)), k=k, rows=rows)
    q = rng.choice(list(BLOCK))
    out = rng.choice(["f16", "f32"])
    k = UNIT[q] * max(1, _log(rng, 512, 16384) // UNIT[q])
    n = max(1, min(_log(rng, 64, 65536), int(MAX_BYTES / (k * (BLOCK[q][0] / BLOCK[q][1] + (2 if out == "f16" else 4))))))
    return dict(kind=kind, qtype=q, n=n, k=k, drop=rng.choice([0, 0, rng.randint(1, 31)]), out=out)


# ------------------------------------------------------------------ inputs

def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _bell(g, shape, bits: int) -> torch.Tensor:
    """Integers 0 .. 2^bits - 1, concentrated in the middle."""
    h = 1 << (bits - 1)
    a = torch.randint(0, h, shape, generator=g, device="cuda", dtype=torch.uint8)
    a += torch.randint(0, h, shape, generator=g, device="cuda", dtype=torch.uint8)
    a += torch.randint(0, 2, shape, generator=g, device="cuda", dtype=torch.uint8)
    return a


def _half(g, nb: int, lo: float, hi: float) -> torch.Tensor:
    v = torch.empty(nb, device="cuda").uniform_(lo, hi, generator=g)
    return v.to(torch.float16)


def _bytes16(v: torch.Tensor) -> torch.Tensor:
    return v.contiguous().view(torch.uint8).view(-1, 2)


def blocks(q: str, n: int, k: int, g) -> torch.Tensor:
    """(n, k) weight in format q: raw block bytes on the GPU."""
    bb, be = BLOCK[q]
    nb = n * (k // be)
    b = torch.empty((nb, bb), dtype=torch.uint8, device="cuda")
    u8 = dict(generator=g, device="cuda", dtype=torch.uint8)
    if q == "Q8_0":
        b[:, :2] = _bytes16(_half(g, nb, 2e-4, 6e-4))
        b[:, 2:] = _bell(g, (nb, 32), 8) + 128                     # signed, centred at 0
    elif q == "Q1_0":
        b[:, :2] = _bytes16(_half(g, nb, 1e-2, 3e-2))
        b[:, 2:] = torch.randint(0, 256, (nb, 16), **u8)
    elif q in ("Q4_K", "Q5_K"):
        d = _half(g, nb, 8e-5, 2e-4) if q == "Q4_K" else _half(g, nb, 4e-5, 1e-4)
        b[:, 0:2] = _bytes16(d)
        b[:, 2:4] = _bytes16((d.float() * (7.5 if q == "Q4_K" else 15.5)).to(torch.float16))
        sc = torch.randint(24, 62, (nb, 8), **u8)
        m = sc + torch.randint(0, 5, (nb, 8), **u8) - 2
        m.clamp_(max=63)
        b[:, 4:8] = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
        b[:, 8:12] = (m[:, :4] & 63) | ((m[:, 4:] >> 4) << 6)
        b[:, 12:16] = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
        if q == "Q5_K":
            c = _bell(g, (nb, 8, 32), 5)
            b[:, 16:48] = 0
            for j in range(8):
                b[:, 16:48] |= (c[:, j] >> 4) << j
            c = (c & 15).view(nb, 4, 2, 32)
        else:
            c = _bell(g, (nb, 4, 2, 32), 4)
        b[:, bb - 128:] = (c[:, :, 0] | (c[:, :, 1] << 4)).view(nb, 128)
    elif q == "Q6_K":
        c = _bell(g, (nb, 2, 4, 32), 6)
        b[:, :128] = ((c[:, :, 0:2] & 15) | ((c[:, :, 2:4] & 15) << 4)).view(nb, 128)
        h = c >> 4
        b[:, 128:192] = (h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)).view(nb, 64)
        s = torch.randint(40, 120, (nb, 16), **u8)
        b[:, 192:208] = torch.where(torch.randint(0, 2, (nb, 16), **u8) > 0, s, 0 - s)
        b[:, 208:210] = _bytes16(_half(g, nb, 1e-5, 4e-5))
    else:
        raise ValueError(q)
    return b.view(-1)


def acts(rows: int, k: int, g) -> torch.Tensor:
    """Activations (rows, k): a scale per channel, one channel in 300 large."""
    ch = torch.exp(0.5 * torch.randn(k, generator=g, device="cuda"))
    ch = torch.where(torch.rand(k, generator=g, device="cuda") < 1 / 300, 20 * ch, ch)
    return torch.randn((rows, k), generator=g, device="cuda") * ch


class _View:
    """A device buffer of the package as a torch tensor (no copy)."""

    def __init__(self, buf, shape):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f4", "data": (buf.ptr, False),
                                         "version": 2}


def _view(buf, shape) -> torch.Tensor:
    return torch.as_tensor(_View(buf, shape), device="cuda")


PROJ = ("q", "k", "v", "o", "gate", "up", "down")


def _block_specs(case) -> dict:
    h, i, qn, kv = case["hidden"], case["inter"], case["q_n"], case["kv_n"]
    main, more = case["main"], case["more"]
    return {"q": (main, qn, h), "k": (main, kv, h), "v": (more, kv, h), "o": (main, h, qn), "gate": (main, i, h),
            "up": (main, i, h), "down": (more, h, i)}


def _gemm_parts(case) -> list:
    return list(zip(case["qtypes"].split(","), map(int, case["ns"].split(","))))


def _inputs(case, seed) -> dict:
    """The raw inputs, from the seed alone."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "block":
        r = case["rows"]
        w = {p: blocks(q, n, k, g) for p, (q, n, k) in _block_specs(case).items()}
        return {"w": w, "x": acts(r, case["hidden"], g), "attn": acts(r, case["q_n"], g),
                "xn": acts(r, case["hidden"], g)}
    if kind == "gemm":
        w = [blocks(q, n, case["k"], g) for q, n in _gemm_parts(case)]
        return {"w": w, "x": acts(case["rows"], case["k"], g).to(torch.bfloat16)}
    w = blocks(case["qtype"], case["n"], case["k"], g)
    return {"w": w} if kind == "dequant" else {"w": w, "x": acts(case["rows"], case["k"], g)}


def prepare(case, seed):
    st = _inputs(case, seed)
    kind = case["kind"]
    f32 = dict(device="cuda", dtype=torch.float32)
    st["case"] = case
    if kind == "block":
        r, i = case["rows"], case["inter"]
        specs = _block_specs(case)
        st["proj"] = p = DecoderProjections({m: (q, st["w"][m], n, k, st["w"][m].numel())
                                             for m, (q, n, k) in specs.items()}, max_seq=r)
        st["out"] = {"qkv": _view(p.qkv, (r, p.qkv_n)), "o": _view(p.o_out, (r, case["hidden"])),
                     "gateup": _view(p.gateup, (r, 2 * i)), "act": _view(p.act, (r, i)),
                     "mlp": _view(p.mlp_out, (r, case["hidden"]))}
    elif kind == "gemm":
        parts = _gemm_parts(case)
        total, off = sum(n for _, n in parts), 0
        st["y"] = torch.empty((case["rows"], total), **f32)
        st["parts"] = []
        for (q, n), w in zip(parts, st["w"]):
            st["parts"].append((q, w, n, st["y"].data_ptr() + 4 * off, w.numel()))
            off += n
        st["total"] = total
    elif kind == "dequant":
        st["elems"] = case["n"] * case["k"] - case["drop"]
        st["y"] = torch.empty(st["elems"], device="cuda", dtype=torch.float16 if case["out"] == "f16" else torch.float32)
    elif kind == "host":
        st["backend"] = flatrun_amd.NativeBackend()
        st["weight"] = st["backend"].upload(st.pop("w").cpu().numpy())
        x = st.pop("x").cpu().numpy()
        st["x"] = x[0].copy() if case["rows"] == 1 else x
        st["call"] = getattr(st["backend"], {"Q4_K": "matmul_q4k", "Q5_K": "matmul_q5_k", "Q6_K": "matmul_q6_k",
                                             "Q8_0": "matmul_q8_0", "Q1_0": "matmul_q1_0"}[case["qtype"]])
    else:
        st["y"] = torch.empty((case["rows"], case["n"]), **f32)
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "matvec":
        device.gemv(case["qtype"], state["w"], state["x"], state["y"], case["n"], case["k"], batch=case["rows"],
                    w_bytes=state["w"].numel())
        return state["y"]
    if kind == "block":
        p, r = state["proj"], case["rows"]
        p.qkv_proj(state["x"], r)
        p.o_proj(state["attn"], r)
        p.mlp(state["xn"], r)
        return state["out"]
    if kind == "gemm":
        device.gemm_bf16_group(state["parts"], state["x"], case["rows"], case["k"], y_stride=state["total"])
        return state["y"]
    if kind == "dequant":
        fn = device.dequant_f16 if case["out"] == "f16" else device.dequant
        fn(case["qtype"], state["w"], state["y"], state["elems"], w_bytes=state["w"].numel())
        return state["y"]
    return state["call"](state["x"], state["weight"], case["n"], case["k"])


# ---------------------------------------------------------- work and truth

def _raw(q: str, n: int, k: int) -> int:
    return n * (k // BLOCK[q][1]) * BLOCK[q][0]


def work(case) -> dict:
    kind = case["kind"]
    if kind == "block":
        r, specs = case["rows"], _block_specs(case)
        w = sum(_raw(q, n, k) for q, n, k in specs.values())
        elems = sum(n * k for _, n, k in specs.values())
        io = 2 * case["hidden"] + case["q_n"] + sum(n for _, n, _ in specs.values()) + case["inter"]
        return {"bytes": w + 4 * r * io, "flops": 2 * r * elems}
    if kind == "gemm":
        r, k, parts = case["rows"], case["k"], _gemm_parts(case)
        total = sum(n for _, n in parts)
        return {"bytes": sum(_raw(q, n, k) for q, n in parts) + 2 * r * k + 4 * r * total, "flops": 2 * r * k * total}
    n, k = case["n"], case["k"]
    if kind == "dequant":
        e = n * k - case["drop"]
        return {"bytes": _raw(case["qtype"], n, k) + e * (2 if case["out"] == "f16" else 4), "flops": 2 * e}
    r = case["rows"]
    return {"bytes": _raw(case["qtype"], n, k) + 4 * r * (n + k), "flops": 2 * r * n * k}


def tolerance(case):
    if case["kind"] == "dequant":
        return "exact"                       # the same bits as the reference decoders
    if case["kind"] == "gemm":
        return {"rel": 6e-3}                 # weights rounded to bf16: 1.7e-3 from 64 bits
    if case["kind"] == "block":
        return {"rel": 2.5e-6}               # fp32 sums of fp32 results: up to 6.3e-7 from 64 bits
    return {"rel": 1.3e-6}                   # fp32 products and sums: up to 3.4e-7


def _f64(b: torch.Tensor) -> torch.Tensor:
    return b.contiguous().view(torch.float16).double()


def weights64(q: str, raw: torch.Tensor, n: int, k: int) -> torch.Tensor:
    """The (n, k) weight that raw stands for, in 64 bits."""
    b = raw.view(-1, BLOCK[q][0])
    nb = b.shape[0]
    if q == "Q8_0":
        w = _f64(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).double()
    elif q == "Q1_0":
        bits = (b[:, 2:].unsqueeze(-1) >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1
        w = _f64(b[:, :2]) * (2.0 * bits.view(nb, 128).double() - 1.0)
    elif q in ("Q4_K", "Q5_K"):
        s0, s1, s2 = b[:, 4:8], b[:, 8:12], b[:, 12:16]
        sc = torch.cat([s0 & 63, (s2 & 15) | ((s0 >> 6) << 4)], 1).double()
        m = torch.cat([s1 & 63, (s2 >> 4) | ((s1 >> 6) << 4)], 1).double()
        qs = b[:, -128:].view(nb, 4, 32)
        c = torch.stack([qs & 15, qs >> 4], 2).view(nb, 8, 32)
        if q == "Q5_K":
            sh = torch.arange(8, device="cuda", dtype=torch.uint8).view(1, 8, 1)
            c = c | (((b[:, 16:48].unsqueeze(1) >> sh) & 1) << 4)
        d, dm = _f64(b[:, 0:2]), _f64(b[:, 2:4])
        w = (d * sc).unsqueeze(-1) * c.double() - (dm * m).unsqueeze(-1)
    else:
        ql, qh = b[:, :128].view(nb, 2, 2, 32), b[:, 128:192].view(nb, 2, 32)
        c = torch.empty((nb, 2, 4, 32), device="cuda", dtype=torch.float64)
        for j in range(4):
            c[:, :, j] = (((ql[:, :, j & 1] >> (4 * (j >> 1))) & 15) | (((qh >> (2 * j)) & 3) << 4)).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (_f64(b[:, 208:210]) * sc).unsqueeze(-1) * c.view(nb, 16, 16)
    return w.reshape(n, k)


def _mul64(q: str, raw, x64: torch.Tensor, n: int, k: int) -> torch.Tensor:
    y = torch.empty((x64.shape[0], n), dtype=torch.float64, device="cuda")
    rb, step = _raw(q, 1, k), max(1, (1 << 26) // k)
    for i in range(0, n, step):
        j = min(n, i + step)
        y[:, i:j] = x64 @ weights64(q, raw[i * rb:j * rb], j - i, k).t()
    return y


def exact(case, seed):
    st = _inputs(case, seed)
    kind = case["kind"]
    if kind == "block":
        specs, w = _block_specs(case), st["w"]
        x, attn, xn = (st[p].double() for p in ("x", "attn", "xn"))
        y = {p: _mul64(specs[p][0], w[p], xn if p in ("gate", "up") else attn if p == "o" else x, *specs[p][1:])
             for p in PROJ[:6]}
        act = y["gate"] * torch.sigmoid(y["gate"]) * y["up"]
        return {"qkv": torch.cat([y["q"], y["k"], y["v"]], 1), "o": y["o"],
                "gateup": torch.cat([y["gate"], y["up"]], 1), "act": act,
                "mlp": _mul64(specs["down"][0], w["down"], act, *specs["down"][1:])}
    if kind == "gemm":
        x = st["x"].double()
        return torch.cat([_mul64(q, w, x, n, case["k"]) for (q, n), w in zip(_gemm_parts(case), st["w"])], 1)
    n, k = case["n"], case["k"]
    if kind == "dequant":
        return weights64(case["qtype"], st["w"], n, k).reshape(-1)[:n * k - case["drop"]]
    y = _mul64(case["qtype"], st["w"], st["x"].double(), n, k)
    if kind == "host":
        y = y.cpu().numpy()
        return np.ascontiguousarray(y[0]) if case["rows"] == 1 else y
    return y
