"""The work a program does with this library, as timed cases.

Five kinds, each through the public wrappers of pulsar_amd.kernels:

  matvec   a decode step's dense projections: every matrix of a stack takes
           the same 1-16 tokens (q8_K quantize + matmul_kq), captured once
           into a graph and replayed, as a decode loop does
  gemm     one dense projection of a prompt chunk (quantize + matmul_kq)
  decode   the routed-MoE layers of a decode step at batch 1, fused entry
           points, captured once and replayed
  chunk    one routed-MoE layer on a token chunk: router, routing, gate / up,
           mid quantize, down, slot sum, grouped on the device
  prefill  the expert FFN of one MoE layer on a long prompt chunk whose
           (token, slot) pairs the host has grouped by expert (CSR)

Weights are random blocks of the GGUF formats, scaled so that a row's dot
with N(0, 1) activations is about N(0, 1), as in a trained layer.
"""
import math
import re
from pathlib import Path

import numpy as np
import torch

from pulsar_amd import kernels as K
from pulsar_amd import runtime
from pulsar_amd.formats import (QUANT_IQ2_XXS, QUANT_IQ4_XS, QUANT_MXFP4, QUANT_Q2_K, QUANT_Q3_K, QUANT_Q4_K,
                                QUANT_Q5_K, QUANT_Q6_K, q8k_blocks, row_bytes)

FMT = {"Q2_K": QUANT_Q2_K, "Q3_K": QUANT_Q3_K, "Q4_K": QUANT_Q4_K, "Q5_K": QUANT_Q5_K, "Q6_K": QUANT_Q6_K,
       "IQ4_XS": QUANT_IQ4_XS, "IQ2_XXS": QUANT_IQ2_XXS, "MXFP4": QUANT_MXFP4}
DEV = "cuda:0"


def listed():
    return [
        # smallest call: one projection after another at batch 1, the decode
        # loop of a dense layer (each launch a few microseconds)
        dict(name="matvec_q4k_1", kind="matvec", quant="Q4_K", rows=4096, cols=4096, tokens=1, stack=32),
        # the output head of a 151936-token vocabulary at batch 1
        dict(name="matvec_q6k_head", kind="matvec", quant="Q6_K", rows=151936, cols=4096, tokens=1, stack=1),
        # speculative / batched decode: 16 tokens per projection
        dict(name="matvec_q6k_16", kind="matvec", quant="Q6_K", rows=8192, cols=4096, tokens=16, stack=10),
        # prompt processing, the common 4-bit format, a whole 512-token chunk
        dict(name="gemm_q4k_512", kind="gemm", quant="Q4_K", rows=14336, cols=4096, tokens=512),
        # prompt processing, a ragged chunk of a codebook format
        dict(name="gemm_iq4xs_250", kind="gemm", quant="IQ4_XS", rows=8192, cols=2816, tokens=250),
        # MoE decode at batch 1 with a shared expert, 4-bit / 6-bit mix
        dict(name="decode_q4k_q6k", kind="decode", gate="Q4_K", down="Q6_K", hidden=2048, experts=256, ffn=512,
             top=8, shared=True, biases=False, act=0, layers=6),
        # MoE decode at batch 1 with biases, MXFP4 experts of wide rows
        dict(name="decode_mxfp4", kind="decode", gate="MXFP4", down="MXFP4", hidden=2880, experts=32, ffn=2880, top=4,
             shared=False, biases=True, act=2, layers=8),
        # a short chunk that touches most experts once or twice
        dict(name="chunk_q2k_16", kind="chunk", gate="Q2_K", down="Q2_K", hidden=4096, experts=128, ffn=1536, top=8,
             tokens=16, shared=False, biases=False, act=0),
        # a ragged chunk of the 2-bit codebook format, ~6 pairs per expert
        dict(name="chunk_iq2xxs_100", kind="chunk", gate="IQ2_XXS", down="IQ2_XXS", hidden=4096, experts=128,
             ffn=1536, top=8, tokens=100, shared=False, biases=False, act=0),
        # a chunk of an MXFP4 layer, ~8 pairs per expert
        dict(name="chunk_mxfp4_64", kind="chunk", gate="MXFP4", down="MXFP4", hidden=2880, experts=32, ffn=2880,
             top=4, tokens=64, shared=False, biases=True, act=2),
        # the largest chunk that groups on the device: 256 tokens, top-8
        dict(name="chunk_q4k_q6k_256", kind="chunk", gate="Q4_K", down="Q6_K", hidden=2048, experts=128, ffn=768,
             top=8, tokens=256, shared=False, biases=False, act=0),
        # a long prompt chunk, ~96 pairs per expert
        dict(name="prefill_q4k_q6k_1536", kind="prefill", gate="Q4_K", down="Q6_K", hidden=2048, experts=128,
             ffn=768, top=8, tokens=1536, shared=False, biases=False, act=0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "gemm", "gemm", "decode", "chunk", "chunk", "prefill"])
    if kind in ("matvec", "gemm"):
        quant = rng.choice(["Q2_K", "Q3_K", "Q4_K", "Q5_K", "Q6_K", "IQ4_XS", "IQ2_XXS"])
        rows, cols = _log(rng, 1000, 16000), 256 * _log(rng, 4, 32)
        if kind == "matvec":
            stack = max(2, min(32, 200_000_000 // (rows * row_bytes(FMT[quant], cols))))
            return dict(kind=kind, quant=quant, rows=rows, cols=cols, tokens=_log(rng, 1, 16), stack=stack)
        most = min(2048, 30_000_000_000 // (rows * cols))
        return dict(kind=kind, quant=quant, rows=rows, cols=cols, tokens=_log(rng, 17, most))
    shape = rng.choice([
        dict(gate="Q4_K", down="Q6_K", hidden=2048, experts=256, ffn=512, top=8, shared=True, biases=False, act=0),
        dict(gate="Q4_K", down="Q6_K", hidden=2048, experts=128, ffn=768, top=8, shared=False, biases=False, act=0),
        dict(gate="Q5_K", down="Q5_K", hidden=2048, experts=128, ffn=768, top=8, shared=False, biases=False, act=0),
        dict(gate="Q3_K", down="Q5_K", hidden=2048, experts=64, ffn=1024, top=6, shared=False, biases=False, act=0),
        dict(gate="IQ4_XS", down="IQ4_XS", hidden=2048, experts=128, ffn=768, top=8, shared=False, biases=False, act=0),
        dict(gate="Q2_K", down="Q2_K", hidden=4096, experts=128, ffn=1536, top=8, shared=False, biases=False, act=0),
        dict(gate="IQ2_XXS", down="IQ2_XXS", hidden=4096, experts=128, ffn=1536, top=8, shared=False, biases=False,
             act=0),
        dict(gate="MXFP4", down="MXFP4", hidden=2880, experts=32, ffn=2880, top=4, shared=False, biases=True, act=2),
    ])
    case = dict(kind=kind, **shape)
    if kind == "decode":
        case["layers"] = rng.randint(3, 8)
        case["top"] = rng.randint(2, case["top"])
        return case
    slots = case["top"] + (1 if case["shared"] else 0)
    if kind == "chunk":
        case["tokens"] = _log(rng, 5, 2048 // slots)
    else:
        # pairs of a long chunk, bounded so that a pass costs no more than the listed ones
        per_pair = 3 * case["hidden"] * case["ffn"]
        case["shared"] = False
        case["tokens"] = _log(rng, 64, min(2048, 55_000_000_000 // (per_pair * case["top"])))
    return case


# ------------------------------------------------------------------ inputs --

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _f16(blocks, off, lo, hi, g):
    """f16 values uniform in [lo, hi] at byte `off` of every block."""
    v = (torch.rand(blocks.shape[0], generator=g, device=DEV) * (hi - lo) + lo).half()
    blocks[:, off:off + 2] = v.view(torch.uint8).view(-1, 2)


# bytes per 256 values, byte offset of d, rms of w / d over random blocks;
# byte offset of dmin and the ratio dmin / d that centres the codes
_BLOCK = {"Q2_K": (84, 80, 13.0, 82, 1.5), "Q3_K": (110, 108, 42.0, None, 0), "Q4_K": (144, 0, 250.0, 2, 7.5),
          "Q5_K": (176, 0, 500.0, 2, 15.5), "Q6_K": (210, 208, 1370.0, None, 0), "IQ4_XS": (136, 0, 1200.0, None, 0),
          "IQ2_XXS": (66, 0, 55.0, None, 0)}


def _weights(fmt, rows, cols, g):
    """uint8 [rows * row_bytes]: random blocks of the format."""
    n = rows * row_bytes(FMT[fmt], cols)
    raw = torch.empty((n + 3) // 4, dtype=torch.int32, device=DEV).random_(-2**31, 2**31 - 1, generator=g)
    raw = raw.view(torch.uint8)[:n]
    if fmt == "MXFP4":
        # a code's rms is ~2.9 half-steps; e8m0 exponents of a trained layer's range
        raw.view(-1, 17)[:, 0] = torch.randint(117, 122, (n // 17,), dtype=torch.uint8, device=DEV, generator=g)
        return raw
    size, d_at, rms, dmin_at, ratio = _BLOCK[fmt]
    blocks = raw.view(-1, size)
    d = 1.0 / (rms * math.sqrt(cols))
    _f16(blocks, d_at, 0.5 * d, 1.5 * d, g)
    if dmin_at is not None:
        _f16(blocks, dmin_at, 0.5 * d * ratio, 1.5 * d * ratio, g)
    return raw


def _randn(shape, g, scale=1.0):
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * scale


def _layer(c, g):
    """One MoE layer's weights: banks [experts][rows][row_bytes] and the rest."""
    E, H, F = c["experts"], c["hidden"], c["ffn"]
    w = dict(gate=_weights(c["gate"], E * F, H, g), up=_weights(c["gate"], E * F, H, g),
             down=_weights(c["down"], E * H, F, g), router=_randn((E, H), g, 1 / math.sqrt(H)))
    if c["biases"]:
        w.update(router_b=_randn((E,), g, 0.02), gate_b=_randn((E, F), g, 0.02), up_b=_randn((E, F), g, 0.02),
                 down_b=_randn((E, H), g, 0.02))
    if c["shared"]:
        w.update(sh_gate=_weights(c["gate"], F, H, g), sh_up=_weights(c["gate"], F, H, g),
                 sh_down=_weights(c["down"], H, F, g))
    return w


def _inputs(c, seed):
    g = _gen(seed)
    if c["kind"] in ("matvec", "gemm"):
        n = c.get("stack", 1)
        return dict(w=[_weights(c["quant"], c["rows"], c["cols"], g) for _ in range(n)],
                    x=_randn((c["tokens"], c["cols"]), g))
    n, T = c.get("layers", 1), c.get("tokens", 1)
    got = dict(layers=[_layer(c, g) for _ in range(n)], x=_randn((n, T, c["hidden"]), g))
    if c["kind"] == "prefill":  # the router's answer: uneven expert loads
        pop = _randn((c["experts"],), g, 0.5)
        top = torch.topk(_randn((T, c["experts"]), g) + pop, c["top"], dim=1)
        got["ids"], got["wts"] = top.indices.int(), torch.softmax(top.values, 1).contiguous()
    return got


def _empty(shape, dtype=torch.float32):
    return torch.zeros(shape, dtype=dtype, device=DEV)


def _bank(c, w):
    grb, drb = row_bytes(FMT[c["gate"]], c["hidden"]), row_bytes(FMT[c["down"]], c["ffn"])
    ptr = lambda k: w[k].data_ptr() if k in w else None  # noqa: E731
    return K.ExpertBank(ptr("gate"), ptr("up"), ptr("down"), ptr("gate_b"), ptr("up_b"), ptr("down_b"),
                        c["ffn"] * grb, c["ffn"] * grb, c["hidden"] * drb, c["ffn"], c["ffn"], c["hidden"])


def prepare(case, seed):
    c, s = case, _inputs(case, seed)
    s["case"] = c
    if c["kind"] in ("matvec", "gemm"):
        s["xq"] = _empty(c["tokens"] * q8k_blocks(c["cols"]) * 292, torch.uint8)
        s["out"] = _empty((len(s["w"]), c["tokens"], c["rows"]))
    else:
        T, n = c.get("tokens", 1), len(s["layers"])
        slots = c["top"] + (1 if c["shared"] else 0)
        E, H, F = c["experts"], c["hidden"], c["ffn"]
        s["xq"] = _empty(T * q8k_blocks(H) * 292, torch.uint8)
        s["midq"] = _empty(T * slots * q8k_blocks(F) * 292, torch.uint8)
        s["mid"], s["out"] = _empty((n, T * slots, F)), _empty((n, T, H))
        s["partial"] = _empty((T * slots, H))
        s["bank"] = [_bank(c, w) for w in s["layers"]]
        if c["kind"] == "prefill":
            _group(c, s)
        else:
            s["logits"], s["sel"] = _empty((n, T, E)), _empty((n, T, c["top"]), torch.int32)
            s["rw"], s["sw"] = _empty((T, c["top"])), _empty((T, slots))
            s["ptrs"], s["active"] = _empty(T * slots * 48, torch.uint8), _empty(2 + E, torch.int32)
            s["no_bias"] = _empty(E)
            s["shared"] = [[(w["sh_gate"].data_ptr(), w["sh_up"].data_ptr(), w["sh_down"].data_ptr())]
                           if c["shared"] else [] for w in s["layers"]]
    torch.cuda.synchronize()
    if c["kind"] in ("matvec", "decode"):
        step = _matvec if c["kind"] == "matvec" else _decode
        s["graph"] = runtime.Graph.capture(lambda: step(s))
    return s


def _group(c, s):
    """The host's CSR of (token, slot) pairs by expert, as a program builds it from the router's ids."""
    bank = s["bank"][0]
    ids = s["ids"].cpu().numpy()
    order = np.argsort(ids.reshape(-1), kind="stable")
    found, count = np.unique(ids, return_counts=True)
    top = c["top"]
    pairs = ((order // top) << 4 | (order % top)).astype(np.uint32)
    starts = np.concatenate([[0], np.cumsum(count)]).astype(np.uint32)
    g = K.expert_ptrs([(bank.gate + int(e) * bank.gate_stride, bank.up + int(e) * bank.up_stride,
                        bank.down + int(e) * bank.down_stride)
                       + ((bank.gate_b + 4 * int(e) * bank.gate_b_stride, bank.up_b + 4 * int(e) * bank.up_b_stride,
                           bank.down_b + 4 * int(e) * bank.down_b_stride) if c["biases"] else ()) for e in found])
    up = lambda a: torch.from_numpy(a.view(np.uint8).copy()).to(DEV)  # noqa: E731
    s["gptrs"], s["starts"], s["pairs"], s["groups"] = up(g), up(starts), up(pairs), len(found)
    if c["biases"]:
        slot = np.searchsorted(found, ids.reshape(-1))
        s["ptrs"] = up(np.ascontiguousarray(g[slot]))


# -------------------------------------------------------------------- run --

def _matvec(s):
    c = s["case"]
    K.quantize_q8_k(s["xq"], s["x"], c["cols"], c["tokens"])
    for w, out in zip(s["w"], s["out"]):
        K.matmul_kq(out, w, s["xq"], c["cols"], c["rows"], c["tokens"], row_bytes(FMT[c["quant"]], c["cols"]),
                    FMT[c["quant"]])


def _decode(s):
    c = s["case"]
    H, F, E, top = c["hidden"], c["ffn"], c["experts"], c["top"]
    gq, dq = FMT[c["gate"]], FMT[c["down"]]
    slots = top + (1 if c["shared"] else 0)
    for i, w in enumerate(s["layers"]):
        K.router_logits_q8(s["logits"][i], s["xq"], s["x"][i], w["router"], w.get("router_b"), H, E, 1)
        K.moe_pair_routed(s["mid"][i], s["ptrs"], s["sw"], s["sel"][i], s["rw"], s["logits"][i], s["no_bias"], E, top,
                          1.0, 1, s["bank"][i], s["shared"][i], s["xq"], H, F, 1, row_bytes(gq, H), gq, c["act"])
        if slots * q8k_blocks(F) <= 24:
            K.moe_down_f32(s["out"][i], s["ptrs"], s["sw"], s["mid"][i], F, H, slots, 1, row_bytes(dq, F), dq,
                           c["biases"])
        else:  # wide mids: one quantize launch beats a quantize in every block
            K.quantize_q8_k(s["midq"], s["mid"][i], F, slots)
            if c["biases"]:
                K.moe_down_biased(s["out"][i], s["ptrs"], s["sw"], s["midq"], F, H, slots, 1, row_bytes(dq, F), dq)
            else:
                K.moe_down(s["out"][i], s["ptrs"], s["midq"], F, H, slots, 1, row_bytes(dq, F), dq)


def _chunk(s):
    c, w, bank, sh = s["case"], s["layers"][0], s["bank"][0], s["shared"][0]
    H, F, E, top, T = c["hidden"], c["ffn"], c["experts"], c["top"], c["tokens"]
    gq, dq = FMT[c["gate"]], FMT[c["down"]]
    slots = top + len(sh)
    K.router_logits_q8(s["logits"], s["xq"], s["x"], w["router"], w.get("router_b"), H, E, T)
    K.moe_route(s["sel"], s["rw"], s["ptrs"], s["sw"], s["active"], s["logits"], s["no_bias"], E, top, 1.0, 1, bank,
                sh, T)
    K.moe_pair_swiglu_experts(s["mid"], s["sel"], s["active"], s["sw"], s["xq"], bank, E, sh, T, top, H, F,
                              row_bytes(gq, H), gq, c["act"])
    K.quantize_q8_k(s["midq"], s["mid"], F, T * slots)
    K.moe_down_experts(s["partial"], s["sel"], s["active"], s["midq"], bank, E, sh, T, top, F, H, row_bytes(dq, F), dq)
    if c["biases"]:
        K.moe_slot_sum_bias(s["out"], s["partial"], s["ptrs"], s["sw"], H, slots, T)
    else:
        K.moe_slot_sum(s["out"], s["partial"], H, slots, T)


def _prefill(s):
    c = s["case"]
    H, F, top, T = c["hidden"], c["ffn"], c["top"], c["tokens"]
    gq, dq = FMT[c["gate"]], FMT[c["down"]]
    K.quantize_q8_k(s["xq"], s["x"], H, T)
    K.moe_pair_swiglu_grouped(s["mid"], s["gptrs"], s["starts"], s["pairs"], s["wts"], s["xq"], H, F, top,
                              s["groups"], row_bytes(gq, H), gq, c["act"])
    K.quantize_q8_k(s["midq"], s["mid"], F, T * top)
    K.moe_down_grouped(s["partial"], s["gptrs"], s["starts"], s["pairs"], s["midq"], F, H, top, s["groups"],
                       row_bytes(dq, F), dq)
    if c["biases"]:
        K.moe_slot_sum_bias(s["out"], s["partial"], s["ptrs"], s["wts"], H, top, T)
    else:
        K.moe_slot_sum(s["out"], s["partial"], H, top, T)


def run(s):
    kind = s["case"]["kind"]
    if "graph" in s:
        s["graph"].launch()
    elif kind == "gemm":
        _matvec(s)
    elif kind == "chunk":
        _chunk(s)
    else:
        _prefill(s)
    if kind in ("matvec", "gemm"):
        return s["out"]
    if kind == "prefill":
        return dict(mid=s["mid"], out=s["out"])
    return dict(logits=s["logits"], selected=s["sel"], mid=s["mid"], out=s["out"])


# ------------------------------------------------------- work, tolerances --

def work(c):
    if c["kind"] in ("matvec", "gemm"):
        n, T = c.get("stack", 1), c["tokens"]
        rb = row_bytes(FMT[c["quant"]], c["cols"])
        return {"bytes": n * c["rows"] * (rb + 4 * T) + 4 * T * c["cols"],
                "flops": 2 * n * T * c["rows"] * c["cols"]}
    n, T, E, H, F = c.get("layers", 1), c.get("tokens", 1), c["experts"], c["hidden"], c["ffn"]
    slots = c["top"] + (1 if c["shared"] else 0)
    touched = E * (1 - (1 - c["top"] / E) ** T) + (1 if c["shared"] else 0)
    expert = 2 * F * row_bytes(FMT[c["gate"]], H) + H * row_bytes(FMT[c["down"]], F)
    if c["biases"]:
        expert += 4 * (2 * F + H)
    router = 0 if c["kind"] == "prefill" else 1
    return {"bytes": n * (touched * expert + router * 4 * E * H + T * 8 * H),
            "flops": n * T * (slots * 6 * H * F + router * 2 * E * H)}


def tolerance(c):
    if c["kind"] in ("matvec", "gemm"):
        # exact int32 sums per 256 values, f32 over the super-blocks
        return {"rel": 2e-6}
    # the mids are rounded to 8 bits again: one f32 ulp can move a code by one
    return {"rel": 2e-3, "max": 0.1, "differ": 0.005}


# ------------------------------------------------------------------- exact --

def _half(b, off):
    return b[..., off:off + 2].contiguous().view(torch.float16)[..., 0].double()


def _kscales(b):
    """The 8 six-bit scales and mins of the 12 packed bytes at 4 of a block."""
    q = b[..., 4:16].int()
    lo, mid, hi = q[..., 0:4], q[..., 4:8], q[..., 8:12]
    sc = torch.cat([lo & 63, (hi & 15) | (lo >> 6) << 4], -1)
    mn = torch.cat([mid & 63, (hi >> 4) | (mid >> 6) << 4], -1)
    return sc.double(), mn.double()


_IQ4NL = [-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113]
_E2M1 = [0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6]


def _iq2xxs_tables():
    text = (Path(__file__).resolve().parent.parent / "include" / "pulsar_iq2xxs_grid.h").read_text()
    codes = [int(v) for v in re.findall(r"\d+", text.split("GRID_CODES")[1].split("#endif")[0])]
    grid = [[(8, 25, 43)[code // 3 ** j % 3] for j in range(8)] for code in codes]
    sign = [[-1 if (i | (bin(i).count("1") & 1) << 7) >> j & 1 else 1 for j in range(8)] for i in range(128)]
    return (torch.tensor(v, dtype=torch.float64, device=DEV) for v in (grid, sign))


def _dequant(fmt, raw, rows, cols):
    """float64 [rows][cols] of the format's blocks, from their layout."""
    if fmt == "MXFP4":
        b = raw.view(rows, -1, 17)
        code = torch.cat([b[..., 1:] & 15, b[..., 1:] >> 4], -1).long()
        w = torch.tensor(_E2M1, dtype=torch.float64, device=DEV)[code]
        return (w * torch.exp2(b[..., :1].double() - 127)).reshape(rows, cols)
    b = raw.view(rows, cols // 256, _BLOCK[fmt][0])
    sh2 = torch.tensor([0, 2, 4, 6], device=DEV, dtype=torch.uint8).view(4, 1)
    if fmt in ("Q4_K", "Q5_K"):
        q = b[..., -128:].reshape(*b.shape[:2], 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], -2).reshape(*b.shape[:2], 8, 32)
        if fmt == "Q5_K":
            bit = torch.arange(8, device=DEV, dtype=torch.uint8).view(8, 1)
            q = q + ((b[..., None, 16:48] >> bit & 1) << 4)
        sc, mn = _kscales(b)
        w = (_half(b, 0)[..., None] * sc)[..., None] * q.double() - (_half(b, 2)[..., None] * mn)[..., None]
    elif fmt == "Q2_K":
        q = b[..., 16:80].reshape(*b.shape[:2], 2, 1, 32) >> sh2 & 3
        q = q.reshape(*b.shape[:2], 16, 16).double()
        s = b[..., :16]
        w = (_half(b, 80)[..., None] * (s & 15).double())[..., None] * q
        w = w - (_half(b, 82)[..., None] * (s >> 4).double())[..., None]
    elif fmt == "Q3_K":
        q = b[..., 32:96].reshape(*b.shape[:2], 2, 1, 32) >> sh2 & 3
        bit = torch.arange(8, device=DEV, dtype=torch.uint8).view(8, 1)
        high = (b[..., None, :32] >> bit & 1).reshape(*b.shape[:2], 2, 4, 32)
        q = (q + 4 * high).double().reshape(*b.shape[:2], 16, 16) - 4
        s = b[..., 96:108].int()
        lo = torch.cat([s[..., :8] & 15, s[..., :8] >> 4], -1)
        hi = torch.cat([s[..., 8:12] >> 2 * k & 3 for k in range(4)], -1)
        w = (_half(b, 108)[..., None] * ((lo | hi << 4) - 32).double())[..., None] * q
    elif fmt == "Q6_K":
        ql = b[..., :128].reshape(*b.shape[:2], 2, 1, 64)
        ql = torch.cat([ql & 15, ql >> 4], -2).reshape(*b.shape[:2], 2, 4, 32)
        qh = b[..., 128:192].reshape(*b.shape[:2], 2, 1, 32) >> sh2 & 3
        q = (ql.double() + 16 * qh.double() - 32).reshape(*b.shape[:2], 16, 16)
        w = (_half(b, 208)[..., None] * b[..., 192:208].contiguous().view(torch.int8).double())[..., None] * q
    elif fmt == "IQ4_XS":
        q = b[..., 8:].reshape(*b.shape[:2], 8, 16).long()
        q = torch.tensor(_IQ4NL, dtype=torch.float64, device=DEV)[torch.cat([q & 15, q >> 4], -1)]
        lo = torch.stack([b[..., 4 + k // 2].int() >> 4 * (k & 1) & 15 for k in range(8)], -1)
        h = b[..., 2].int() | b[..., 3].int() << 8
        hi = torch.stack([h >> 2 * k & 3 for k in range(8)], -1)
        w = (_half(b, 0)[..., None] * ((lo | hi << 4) - 32).double())[..., None] * q
    else:  # IQ2_XXS
        grid, sign = _iq2xxs_tables()
        a = b[..., 2:].contiguous().view(torch.int32).long().reshape(*b.shape[:2], 8, 2) & 0xffffffff
        g = torch.stack([grid[a[..., 0] >> 8 * j & 255] * sign[a[..., 1] >> 7 * j & 127] for j in range(4)], -2)
        w = (_half(b, 0)[..., None] * (2 * (a[..., 1] >> 28) + 1).double() * 0.125)[..., None, None] * g
    return w.reshape(rows, cols)


def _q8(x):
    """float64 [n][cols]: f32 rows through the q8_K quantizer (codes of 256-value
    blocks in steps of amax / 127, halves away from zero) and back."""
    n, cols = x.shape
    pad = -cols % 256
    b = torch.nn.functional.pad(x.float(), (0, pad)).reshape(n, -1, 256)
    amax = b.abs().amax(-1, keepdim=True)
    # divided tensor by tensor: a division by a number is a product with its reciprocal here
    top = torch.full_like(amax, 127.0)
    v = b * torch.where(amax > 0, top / amax, torch.zeros_like(amax))
    q = torch.sign(v) * torch.floor(v.double().abs() + 0.5)
    return (q.clamp(-127, 127) * (amax / top).double()).reshape(n, -1)[:, :cols]


def _glu(g, u, act):
    if act == 2:
        g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0) + 1
        return g * torch.sigmoid(1.702 * g) * u
    return g * torch.sigmoid(g) * u


def _experts(c, w, x, ids, wts):
    """mid of one layer in 64 bits: x [T][H], ids / wts [T][slots]; id -1: the shared expert."""
    E, H, F = c["experts"], c["hidden"], c["ffn"]
    T, slots = ids.shape
    xq = _q8(x)
    mid = torch.zeros((T * slots, F), dtype=torch.float64, device=DEV)
    flat = ids.reshape(-1)
    for e in flat.unique().tolist():
        at = (flat == e).nonzero()[:, 0]
        tok = at // slots
        wt = wts.reshape(-1)[at].double()[:, None]
        if e < 0:
            mats = [w["sh_gate"], w["sh_up"]]
        else:
            mats = [w[k].view(E, -1)[e] for k in ("gate", "up")]
        xe = xq[tok]
        g = xe @ _dequant(c["gate"], mats[0], F, H).T.contiguous()
        u = xe @ _dequant(c["gate"], mats[1], F, H).T.contiguous()
        if c["biases"]:
            g, u = g + w["gate_b"][e].double(), u + w["up_b"][e].double()
        mid[at] = _glu(g, u, c["act"]) * wt
    return mid


def exact(c, seed):
    """The layers' `out` has no value here: the down stage takes the mids rounded
    to 8 bits, and the last bit of an f32 mid moves one of those codes now and
    then, by far more than any 32-bit sum is off."""
    s = _inputs(c, seed)
    if c["kind"] in ("matvec", "gemm"):
        x = _q8(s["x"])
        got = []
        for w in s["w"]:
            step, rb = 8192, row_bytes(FMT[c["quant"]], c["cols"])
            parts = [x @ _dequant(c["quant"], w[r * rb:min(r + step, c["rows"]) * rb], min(step, c["rows"] - r),
                                  c["cols"]).T.contiguous() for r in range(0, c["rows"], step)]
            got.append(torch.cat(parts, 1))
        return torch.stack(got)
    if c["kind"] == "prefill":
        return dict(mid=_experts(c, s["layers"][0], s["x"][0], s["ids"], s["wts"])[None], out=None)
    got = dict(logits=[], selected=[], mid=[])
    for w, x in zip(s["layers"], s["x"]):
        logits = x.double() @ w["router"].double().T.contiguous()
        if c["biases"]:
            logits = logits + w["router_b"].double()
        top = torch.topk(logits, c["top"], dim=1)
        ids, wts = top.indices, torch.softmax(top.values, 1)
        if c["shared"]:
            ids = torch.cat([ids, torch.full_like(ids[:, :1], -1)], 1)
            wts = torch.cat([wts, torch.ones_like(wts[:, :1])], 1)
        mid = _experts(c, w, x, ids, wts)
        for k, v in dict(logits=logits, selected=top.indices.int(), mid=mid).items():
            got[k].append(v)
    return dict({k: torch.stack(v) for k, v in got.items()}, out=None)
