"""Performance cases: the packed-matmul work a user of this library has it do.

Five kinds of call, each through the public ctypes binding of libprism_hip.so:

  project   prism_hip_project_device on f32 rows: the matvec of a decode step, the few
            tokens of a speculative or batched step, the many of a prompt (MUL_MAT).
  siblings  one quantization of the input shared by several matrices (q, k and v).
  ffn       the FFN step of one token on device pointers (gate, up, SwiGLU, down).
  prompt    the FFN chain over the tokens of a prompt, host arrays in and out, as the
            executor boundary is called by its host program.
  decode    whole greedy steps of the resident decoder, with their logits.

Weights are drawn in the native packed layouts: uniform codes, binary16 block scales
|N(0, 0.02)|, Q2_K minimum scales N(0, 0.01); inputs are N(0, 1).
"""

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "prism-inference_amd"))

import prism_hip as ph  # noqa: E402

KINDS = {"PTQ1": ph.KIND_PTQ1, "PQ2": ph.KIND_PQ2, "Q2_K": ph.KIND_Q2_K, "Q8_0": ph.KIND_Q8_0,
         "TQ1_0": ph.KIND_TQ1_0, "TQ2_0": ph.KIND_TQ2_0}
DEV = "cuda"


def listed():
    return [
        # One ternary projection of a small model's decode step: launches and latency.
        {"name": "matvec-small", "call": "project", "kind": "PTQ1", "rows": 2048, "cols": 2048, "tokens": 1,
         "pinned": False},
        # A down projection of a larger model, one token, in the contract a graph uses.
        {"name": "matvec-long-rows", "call": "project", "kind": "PQ2", "rows": 5120, "cols": 17408, "tokens": 1,
         "pinned": True},
        # The tied LM head of a 151936-token vocabulary: one pass over HBM.
        {"name": "lm-head", "call": "project", "kind": "Q8_0", "rows": 151936, "cols": 2048, "tokens": 1,
         "pinned": False},
        # One FFN step at batch 1 in 2-bit weights, with its residual.
        {"name": "ffn-step", "call": "ffn", "kind": "Q2_K", "rows": 6144, "cols": 2048, "tokens": 1, "pinned": False},
        # q, k and v of one attention layer for a seven-token draft.
        {"name": "qkv-draft", "call": "siblings", "kind": "PTQ1", "rows": 2048, "rows_b": 512, "rows_c": 512,
         "cols": 2048, "tokens": 7, "pinned": True},
        # Four and sixteen concurrent requests, one token each, on a larger layer.
        {"name": "batch-4", "call": "project", "kind": "PTQ1", "rows": 12288, "cols": 4096, "tokens": 4,
         "pinned": False},
        {"name": "batch-16", "call": "project", "kind": "Q2_K", "rows": 12288, "cols": 4096, "tokens": 16,
         "pinned": False},
        # Prompts: a short one, a long one, and a ragged one in the pinned contract on wide rows.
        {"name": "prompt-short", "call": "project", "kind": "PTQ1", "rows": 6144, "cols": 2048, "tokens": 128,
         "pinned": False},
        {"name": "prompt-long", "call": "project", "kind": "PTQ1", "rows": 6144, "cols": 2048, "tokens": 2048,
         "pinned": False},
        {"name": "prompt-ragged-pinned", "call": "project", "kind": "PTQ1", "rows": 4096, "cols": 14336,
         "tokens": 411, "pinned": True},
        # The FFN of one layer over a prompt, from and to host memory.
        {"name": "ffn-prompt-host", "call": "prompt", "kind": "PQ2", "rows": 6144, "cols": 2048, "tokens": 333,
         "pinned": True},
        # Greedy decode: 28 layers, 1024 cached positions, the tied head; four tokens and their logits.
        {"name": "decode", "call": "decode", "layers": 28, "pos": 1024, "vocab": 151936, "tokens": 4},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


MAX_FLOPS = 5.0e10  # rows * cols * tokens * 2 of the largest listed projections


def draw(rng):
    call = rng.choices(["project", "siblings", "ffn", "prompt", "decode"], [12, 2, 2, 2, 1])[0]
    if call == "decode":
        return {"call": "decode", "layers": rng.randint(2, 27), "pos": _log(rng, 16, 1023),
                "vocab": _log(rng, 16384, 151935), "tokens": 4}
    kind = rng.choices(list(KINDS), [8, 3, 3, 2, 1, 1])[0]
    pinned = rng.random() < 0.5
    unit = 128 if kind in ("PTQ1", "PQ2", "Q8_0") else 256
    while True:
        tokens = 1 if call == "ffn" or (call != "prompt" and rng.random() < 0.4) else _log(rng, 2, 2048)
        if call in ("ffn", "prompt"):  # hidden and FFN width, both whole blocks
            cols, rows = _log(rng, 1024, 5120) // 256 * 256, _log(rng, 2048, 17408) // 256 * 256
            if tokens == 1 and call == "prompt":
                continue
            macs = 3 * rows * cols
        else:
            cols, rows = _log(rng, 1024, 17408) // unit * unit, _log(rng, 512, 151936)
            macs = rows * cols * (3 if call == "siblings" else 1)
        # No more than the largest listed cases: operations, and bytes of weights.
        if 2.0 * macs * tokens <= MAX_FLOPS and macs <= 151936 * 4096:
            break
    case = {"call": call, "kind": kind, "rows": rows, "cols": cols, "tokens": tokens, "pinned": pinned}
    if call == "siblings":
        case["rows_b"], case["rows_c"] = max(1, rows // 4), max(1, rows // 4)
    return case


# ---- packed weights ------------------------------------------------------------------


def _gen(seed, salt):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + salt) & 0x7FFFFFFFFFFFFFFF)
    return g


def _half(g, n, sigma, signed=False):
    """n binary16 scales as bytes [n, 2]."""
    s = torch.randn(n, generator=g, device=DEV) * sigma
    s = s if signed else s.abs().clamp_(min=1e-5)
    return s.half().view(torch.uint8).view(n, 2)


def packed(kind, rows, cols, g):
    """Native bytes of a [rows][cols] tensor, on the GPU."""
    qk, size = ph.LAYOUT[KINDS[kind]]
    n = rows * cols // qk
    out = torch.empty((n, size), dtype=torch.uint8, device=DEV)
    if kind == "PTQ1":  # ceil(q * 256 / 243) of five base-3 digits; the last two bytes hold four
        q = torch.randint(0, 243, (n, 26), generator=g, device=DEV, dtype=torch.int32)
        q[:, 24:] -= q[:, 24:] % 3
        out[:, :26] = ((q * 256 + 242) // 243).to(torch.uint8)
        out[:, 26:] = _half(g, n, 0.02)
    elif kind == "PQ2":  # ternary codes 0..2, four to a byte
        c = torch.randint(0, 3, (n, 32, 4), generator=g, device=DEV, dtype=torch.uint8)
        out[:, :2] = _half(g, n, 0.02)
        out[:, 2:] = c[:, :, 0] | (c[:, :, 1] << 2) | (c[:, :, 2] << 4) | (c[:, :, 3] << 6)
    elif kind == "Q2_K":
        out[:, :80] = torch.randint(0, 256, (n, 80), generator=g, device=DEV, dtype=torch.uint8)
        out[:, 80:82] = _half(g, n, 0.02)
        out[:, 82:84] = _half(g, n, 0.01, signed=True)
    elif kind == "Q8_0":  # codes of N(0, 0.02) floats, their largest magnitude 127
        x = torch.randn((n, 32), generator=g, device=DEV) * 0.02
        d = x.abs().amax(1, keepdim=True) / 127.0
        out[:, :2] = d.half().view(torch.uint8).view(n, 2)
        out[:, 2:] = (x / d).round().clamp(-127, 127).to(torch.int8).view(torch.uint8)
    else:  # TQ1_0 / TQ2_0: any byte is a valid code
        out[:, : size - 2] = torch.randint(0, 256, (n, size - 2), generator=g, device=DEV, dtype=torch.uint8)
        out[:, size - 2:] = _half(g, n, 0.02)
    return out.view(-1)


# ---- one call's state ----------------------------------------------------------------

_ctx = None


def context():
    """One context per process, as one host thread of a serving program keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = ph.Context(0)
    return _ctx


class State(dict):
    """Inputs, outputs and the weights a program keeps resident; gives them back at its end."""

    def weight(self, case, rows, cols, salt, seed):
        w = packed(case["kind"], rows, cols, _gen(seed, salt))
        torch.cuda.synchronize()
        wid = context().weight_from_device(KINDS[case["kind"]], cols, rows, w)
        self.setdefault("weights", []).append(wid)
        return wid

    def __del__(self):
        try:
            if "decoder" in self:
                self["decoder"].close()
            for wid in self.get("weights", []):
                context().release(wid)
        except Exception:
            pass


def _sizes(case):
    return [(case["rows"], 1)] + [(case[k], s) for k, s in (("rows_b", 2), ("rows_c", 3)) if k in case]


def _floats(case, n, salt, seed):
    return torch.randn((case["tokens"], n), generator=_gen(seed, salt), device=DEV)


def _contract(case):
    """The Q8_0 contract of a prepared activation, or None for Q8_K blocks."""
    kind, cols = case["kind"], case["cols"]
    if kind in ("Q2_K", "TQ1_0", "TQ2_0") or (kind == "PQ2" and cols % 256 == 0):
        return None
    if not case["pinned"]:
        return ph.Q8_SOURCE
    return ph.Q8_PINNED_NATIVE if kind == "PTQ1" else ph.Q8_PINNED


def _decoder(case, seed):
    g = _gen(seed, 0)
    host = lambda t: t.cpu().numpy()  # noqa: E731
    hidden, ffn, heads, kv, dim, rows = 2048, 6144, 16, 4, 128, case["pos"]
    norm = lambda n: host(1.0 + 0.1 * torch.randn(n, generator=g, device=DEV))  # noqa: E731
    cache = lambda: host(torch.randn((rows, kv * dim), generator=g, device=DEV).half()).view(np.uint16)  # noqa: E731
    layers = []
    for _ in range(case["layers"]):
        m = {n: host(packed("PTQ1", r, c, g)) for n, r, c in (
            ("qkv", (heads + 2 * kv) * dim, hidden), ("o", hidden, heads * dim), ("gate", ffn, hidden),
            ("up", ffn, hidden), ("down", hidden, ffn))}
        m.update(norm=norm(hidden), post_norm=norm(hidden), q_norm=norm(dim), k_norm=norm(dim), kv_prefill=rows,
                 k_prefill=cache(), v_prefill=cache())
        layers.append(m)
    geometry = {"hidden": hidden, "ffn": ffn, "heads": heads, "kv_heads": kv, "head_dim": dim, "rope": 64,
                "rope_sections": (11, 11, 10, 0), "rope_base": 1e7, "eps": 1e-6, "vocab": case["vocab"],
                "layers": case["layers"], "max_tokens": rows + case["tokens"]}
    return ph.Decoder(context(), {"geometry": geometry, "layers": layers, "output_norm": norm(hidden),
                                  "lm_head": host(packed("Q8_0", case["vocab"], hidden, g))},
                      max_steps=case["tokens"])


def prepare(case, seed):
    s = State(case=case)
    call = case["call"]
    if call == "decode":
        s["decoder"] = _decoder(case, seed)
        s["token"] = int(seed) % case["vocab"]
        return s
    rows, cols, tokens = case["rows"], case["cols"], case["tokens"]
    x = _floats(case, cols, 9, seed)
    if call in ("project", "siblings"):
        s["ids"] = [s.weight(case, r, cols, salt, seed) for r, salt in _sizes(case)]
        s["out"] = [torch.empty((tokens, r), device=DEV) for r, _ in _sizes(case)]
        s["x"] = x
        if call == "siblings":  # Q8_K blocks of 292 bytes per 256 values, Q8_0 blocks of 40 per 32
            size = cols // 256 * 292 if _contract(case) is None else cols // 32 * 40
            s["blocks"] = torch.empty(tokens * size, dtype=torch.uint8, device=DEV)
        return s
    s["ids"] = [s.weight(case, rows, cols, 1, seed), s.weight(case, rows, cols, 2, seed),
                s.weight(case, cols, rows, 3, seed)]
    residual = _floats(case, cols, 8, seed)
    if call == "ffn":
        s.update(x=x, residual=residual, out=torch.empty((1, cols), device=DEV))
    else:
        s.update(x=x.cpu().numpy(), residual=residual.cpu().numpy())
    return s


def run(s):
    case, ctx = s["case"], context()
    call, tokens, pinned = case["call"], case["tokens"], case.get("pinned")
    if call == "project":
        ctx.project_device(s["ids"][0], ph.PATH_F32, s["x"], tokens, pinned, s["out"][0])
        return s["out"]
    if call == "siblings":
        contract = _contract(case)
        if contract is None:
            ctx.quantize_q8k_device(s["x"], case["cols"], tokens, pinned, s["blocks"])
        else:
            ctx.quantize_q8_device(s["x"], case["cols"], tokens, contract, s["blocks"])
        for wid, out in zip(s["ids"], s["out"]):
            ctx.project_device(wid, ph.PATH_Q8K if contract is None else ph.PATH_Q8, s["blocks"], tokens, pinned, out)
        return s["out"]
    if call == "ffn":
        ctx.ffn_chain_device(*s["ids"], s["x"], s["residual"], pinned, s["out"])
        return s["out"]
    if call == "prompt":
        return ctx.ffn_chain_tokens(*s["ids"], case["cols"], s["x"], residual=s["residual"], pinned=pinned)
    tokens_out, logits, _ = s["decoder"].generate(s["token"], case["pos"], tokens, logits=True)
    return {"tokens": tokens_out.astype(np.int64), "logits": logits}


# ---- what a pass cannot do without -----------------------------------------------------


def _weight_bytes(kind, rows, cols):
    qk, size = ph.LAYOUT[KINDS[kind]]
    return rows * cols // qk * size


def work(case):
    if case["call"] == "decode":
        per_layer = [(3072, 2048), (2048, 2048), (6144, 2048), (6144, 2048), (2048, 6144)]
        weights = case["layers"] * sum(_weight_bytes("PTQ1", r, c) for r, c in per_layer)
        weights += _weight_bytes("Q8_0", case["vocab"], 2048)
        macs = case["layers"] * (sum(r * c for r, c in per_layer) + 2 * 2048 * case["pos"]) + case["vocab"] * 2048
        cache = case["layers"] * 2 * case["pos"] * 512 * 2
        return {"bytes": case["tokens"] * (weights + cache + 4 * case["vocab"]), "flops": case["tokens"] * 2 * macs}
    rows, cols, tokens, kind = case["rows"], case["cols"], case["tokens"], case["kind"]
    if case["call"] in ("ffn", "prompt"):
        weights = 2 * _weight_bytes(kind, rows, cols) + _weight_bytes(kind, cols, rows)
        return {"bytes": weights + 3 * 4 * tokens * cols, "flops": 2.0 * 3 * rows * cols * tokens}
    total = sum(r for r, _ in _sizes(case))
    weights = sum(_weight_bytes(kind, r, cols) for r, _ in _sizes(case))
    return {"bytes": weights + 4 * tokens * (cols + total), "flops": 2.0 * total * cols * tokens}


def tolerance(case):
    # Projections are specified to the bit: exact integer block dots, and one binary32
    # order of the block sums.  So is the pinned SwiGLU with its polynomial exp.
    if case["call"] in ("project", "siblings") or (case["call"] == "prompt" and case["pinned"]):
        return "exact"
    # The source SwiGLU follows the platform's expf: another correctly rounded exp moves
    # an 8-bit code of the down projection's input now and then: one of 6144 codes is a
    # relative 3.5e-4 of the result (a step of 3.5 sigma / 127 against sigma * sqrt(6144)).
    if case["call"] in ("ffn", "prompt"):
        return {"rel": 1e-3, "max": 1e-2}
    # Whole decode steps carry a last-bit difference of exp, sin or cos through all layers.
    return {"rel": 1e-3, "max": 1e-2}


# ---- the same in 64 bits ----------------------------------------------------------------


def _values(kind, rows, cols, raw):
    """Weights as float64 [rows][cols] from native bytes."""
    qk, size = ph.LAYOUT[KINDS[kind]]
    b = raw.view(rows * cols // qk, size)
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731

    def digits(at, n, count):  # base-3 digits k of n bytes: [blocks][count][n] in element order
        q, got = b[:, at:at + n].to(torch.int32), []
        for _ in range(count):
            got.append(q * 3 >> 8)
            q = q * 3 & 255
        return torch.stack(got, 1).reshape(b.shape[0], -1).double()

    def pairs(at, n):  # 2-bit fields k of n bytes: [blocks][4][n]
        q = b[:, at:at + n].to(torch.int32)
        return torch.stack([q >> 2 * k & 3 for k in range(4)], 1).double()

    if kind == "PTQ1":
        v = (torch.cat([digits(0, 16, 5), digits(16, 8, 5), digits(24, 2, 4)], 1) - 1) * half(26)
    elif kind == "PQ2":
        v = (pairs(2, 32).transpose(1, 2).reshape(-1, 128) - 1) * half(0)
    elif kind == "Q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).double() * half(0)
    elif kind == "TQ1_0":
        v = (torch.cat([digits(0, 32, 5), digits(32, 16, 5), digits(48, 4, 4)], 1) - 1) * half(52)
    elif kind == "TQ2_0":
        v = (torch.cat([pairs(0, 32).reshape(-1, 128), pairs(32, 32).reshape(-1, 128)], 1) - 1) * half(64)
    else:
        s = b[:, :16].to(torch.int32)
        q = torch.cat([pairs(16, 32).reshape(-1, 128), pairs(48, 32).reshape(-1, 128)], 1).view(-1, 16, 16)
        v = half(80)[:, :, None] * (s & 15).double()[:, :, None] * q
        v = (v - half(82)[:, :, None] * (s >> 4).double()[:, :, None]).reshape(-1, 256)
    return v.reshape(rows, cols)


def _codes(case, x, cols):
    """The 8-bit activation blocks the contract rounds x to, as float64 values."""
    contract = _contract(dict(case, cols=cols))
    if contract is None:
        v = x.reshape(-1, 256)
        top = v.gather(1, v.abs().argmax(1, keepdim=True))
        inv = torch.where(top != 0, torch.full_like(top, -127.0) / top, torch.zeros_like(top))
        q = (v.double() * inv.double() if case["pinned"] else v * inv).round().clamp(max=127).double()
        scale = torch.where(inv != 0, torch.ones_like(inv) / inv, torch.zeros_like(inv))
    else:
        v = x.reshape(-1, 32)
        m = v.abs().amax(1, keepdim=True)
        if contract == ph.Q8_PINNED_NATIVE:
            d, inv = m * np.uint32(0x3C010204).view(np.float32).item(), torch.full_like(m, 127.0) / m
        else:
            d = m / torch.full_like(m, 127.0)
            inv = torch.ones_like(d) / d
        p = v * inv
        q = (p.sign() * (p.abs().double() + 0.5).floor() if contract == ph.Q8_SOURCE else p.round()).double()
        scale = d.half()
    return (q * scale.double()).reshape(-1, cols)


def _product(case, rows, cols, salt, seed, act):
    w = _values(case["kind"], rows, cols, packed(case["kind"], rows, cols, _gen(seed, salt)))
    return act @ w.T


def exact(case, seed):
    if case["call"] == "decode":
        return None  # a whole model: minutes in 64 bits
    rows, cols = case["rows"], case["cols"]
    act = _codes(case, _floats(case, cols, 9, seed), cols)
    if case["call"] in ("project", "siblings"):
        return [_product(case, r, cols, salt, seed, act) for r, salt in _sizes(case)]
    gate, up = (_product(case, rows, cols, salt, seed, act) for salt in (1, 2))
    h = (gate / (1.0 + torch.exp(-gate)) * up).float()
    out = _product(case, cols, rows, 3, seed, _codes(case, h, rows)) + _floats(case, cols, 8, seed).double()
    return out.cpu().numpy() if case["call"] == "prompt" else out
