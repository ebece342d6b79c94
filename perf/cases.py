"""The calls that a program built on this library spends its time in, as
measurable cases: one dict of plain sizes each, with the inputs, the call,
the work it cannot do without, and its result in 64 bits.

Five families, all through the C ABI on buffers that the caller owns:

  rotate    ouro_fwht_rows: the Walsh-Hadamard rotation of activation rows,
            with the int8 quantisation that feeds a ternary product
  linear    y = W x for one column (decode) or several (batched verify,
            prefill): ouro_weight_matmul of a resident ternary weight,
            ouro_matmul_q of a block-quantised or dense payload as it lies
            in a mapped shard
  head      ouro_weight_matvec_argmax: the lm_head of a greedy step
  delta     the gated delta-net: one decode step (the recurrence alone, or
            the whole layer block) and the prefill of packed prompts
  stack     the hybrid decoder: prefill of ragged prompts, then decode steps
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ouroboros_amd import _lib
from ouroboros_amd._lib import DT_BF16, DT_F32, FWHT_INVERSE, GDN_L2NORM_QK, GDN_SCALE_Q, GDN_V_GROUPED, call
from ouroboros_amd.ops import Weight
from ouroboros_amd.quant import QuantKind
from ouroboros_amd.stack import Card, Stack

D = 128  # head width of the delta-net and attention layers
EPS = 1e-6
TERNARY = ("I2_S", "TL1", "TQ1_0")
BLOCKED = ("Q8_0", "Q3K", "Q4K", "Q5K", "Q6K")
DENSE = ("F32", "F16", "BF16")
I2_WIDTHS = (512, 1024, 2048, 2560, 3072, 4096, 5120, 6144, 6912, 8192)  # rows that a resident I2 weight takes


def listed():
    return [
        # one token's residual row rotated and quantised ahead of a decode
        # step's projections: a call of a few microseconds, all latency
        {"name": "rotate_token", "family": "rotate", "rows": 1, "n": 2560, "block": 512, "bf16": False,
         "signs": True, "inverse": False, "quant": True, "store": False},
        # a prefill's FFN activations (an odd number of rows), rotated rows kept as well
        {"name": "rotate_prompt", "family": "rotate", "rows": 515, "n": 6912, "block": 256, "bf16": True,
         "signs": True, "inverse": False, "quant": True, "store": True},
        # one FFN projection of one decoded token, bitnet.cpp weights resident
        {"name": "ternary_token", "family": "linear", "kind": "I2_S", "out_len": 6912, "in_len": 2560, "k": 1},
        # the FFN's down projection over a prompt
        {"name": "ternary_prompt", "family": "linear", "kind": "I2_S", "out_len": 2560, "in_len": 6912, "k": 1500},
        # a square projection of one token, 4-bit blocks read in place
        {"name": "kquant_token", "family": "linear", "kind": "Q4K", "out_len": 8192, "in_len": 8192, "k": 1},
        # the same for the few columns of a batched verify, 6-bit blocks
        {"name": "kquant_verify", "family": "linear", "kind": "Q6K", "out_len": 4096, "in_len": 14336, "k": 6},
        # an unquantised projection for a small batch
        {"name": "dense_batch", "family": "linear", "kind": "BF16", "out_len": 8192, "in_len": 2560, "k": 4},
        # the lm_head of a greedy step: logits and the token
        {"name": "head_greedy", "family": "head", "kind": "TL1", "out_len": 248320, "in_len": 2560},
        # one decode step of a delta-net layer for a batch of sequences
        {"name": "delta_step", "family": "delta", "seqs": 32, "tokens": 0, "hk": 16, "hv": 32, "layer": True,
         "bf16": False, "ragged": 0},
        # the delta-net prefill of seven ragged prompts
        {"name": "delta_prompts", "family": "delta", "seqs": 7, "tokens": 9001, "hk": 16, "hv": 32, "layer": False,
         "bf16": True, "ragged": 3},
        # one user: a prompt, then tokens one at a time (a twelfth of the
        # 24-layer stack and its head: see _card)
        {"name": "stack_single", "family": "stack", "seqs": 1, "tokens": 300, "steps": 16, "ragged": 0},
        # a served batch: ragged prompts packed, then joint decode steps
        {"name": "stack_batch", "family": "stack", "seqs": 48, "tokens": 20000, "steps": 16, "ragged": 5},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(("rotate", "linear", "linear", "linear", "head", "delta", "delta", "stack"))
    if family == "rotate":
        block = 1 << rng.randint(6, 12)
        n = block * rng.randint(1, max(1, 8192 // block))
        quant = rng.random() < 0.7
        return {"family": "rotate", "rows": _log(rng, 1, 2048), "n": n, "block": block, "bf16": rng.random() < 0.5,
                "signs": rng.random() < 0.7, "inverse": rng.random() < 0.2, "quant": quant,
                "store": not quant or rng.random() < 0.5}
    if family == "linear":
        kind = rng.choice(("I2_S", "I2_S", "TL1", "TQ1_0") + BLOCKED + DENSE)
        unit = {"TL1": 128, "TQ1_0": 256, "Q8_0": 32, "F32": 1, "F16": 1, "BF16": 1}.get(kind, 256)
        in_len = rng.choice(I2_WIDTHS) if kind == "I2_S" else unit * max(1, _log(rng, 512, 14336) // unit)
        out_len = min(_log(rng, 64, 32768), (1 << 26) // in_len)
        most = 1024 if kind == "I2_S" else 16
        k = rng.choice((1, 1, _log(rng, 2, 16), _log(rng, 2, most)))
        return {"family": "linear", "kind": kind, "out_len": out_len, "in_len": in_len, "k": k}
    if family == "head":
        kind = rng.choice(("TL1", "TL1", "TQ1_0", "I2_S"))
        return {"family": "head", "kind": kind, "out_len": _log(rng, 8192, 248320),
                "in_len": rng.choice(I2_WIDTHS[:4]) if kind == "I2_S" else 256 * rng.randint(2, 10)}
    hk, hv = rng.choice(((16, 32), (16, 16), (4, 12), (8, 32)))
    if family == "delta":
        if rng.random() < 0.5:
            layer = rng.random() < 0.5
            return {"family": "delta", "seqs": _log(rng, 1, 64), "tokens": 0, "hk": hk, "hv": hv, "layer": layer,
                    "bf16": not layer and rng.random() < 0.5, "ragged": 0}
        seqs = _log(rng, 1, 16)
        return {"family": "delta", "seqs": seqs, "tokens": max(seqs, _log(rng, 33, 9000)), "hk": hk, "hv": hv,
                "layer": False, "bf16": True, "ragged": rng.randint(0, 1 << 20)}
    seqs = _log(rng, 1, 48)
    return {"family": "stack", "seqs": seqs, "tokens": max(seqs, _log(rng, 24, 12000)), "steps": rng.randint(1, 16),
            "ragged": rng.randint(0, 1 << 20)}


# ---- inputs ----

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _half_bytes(x):
    """fp16 of x as little-endian byte pairs."""
    return x.to(torch.float16).contiguous().view(torch.uint8).reshape(-1, 2)


def _lengths(case):
    """Lengths of the case's sequences, ragged by a seed that is part of the case."""
    n, total = case["seqs"], case["tokens"]
    share = np.random.default_rng(case["ragged"]).uniform(0.05, 1.0, n)
    lens = np.maximum(1, np.floor(share / share.sum() * (total - n)).astype(np.int64))
    lens[0] += total - lens.sum()
    assert lens.min() >= 1 and lens.sum() == total
    return lens


def _card():
    """One delta-net and one attention layer at the full widths, with a head
    of a twelfth of the vocabulary: a twelfth of the 24-layer stack.  Its
    activations are rounded to int8 ahead of every projection, so that one
    rounding changed in the last bit moves the logits of 24 layers by a fifth,
    of two by two to three percent."""
    return Card(n_layer=2, full_attention_interval=2, n_vocab=20693)


def _blocks(kind):
    return QuantKind[kind].block_bytes(), QuantKind[kind].block_elems()


def _payload(case, g):
    """Device bytes of a random weight tensor of the case's kind."""
    kind, out, n = case["kind"], case["out_len"], case["in_len"]
    if kind in DENSE:
        dt = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[kind]
        return (_randn(g, out, n) / math.sqrt(n)).to(dt).reshape(-1).view(torch.uint8)
    if kind == "I2_S":  # 2-bit codes 0..2, then the fp32 scale and 28 bytes of padding
        c = torch.randint(0, 3, (4, out * n // 4), generator=g, device="cuda", dtype=torch.uint8)
        scale = torch.zeros(8, dtype=torch.float32, device="cuda")
        scale[0] = 1.0 / math.sqrt(n * 2 / 3)
        return torch.cat([c[0] << 6 | c[1] << 4 | c[2] << 2 | c[3], scale.view(torch.uint8)])
    bb, be = _blocks(kind)
    nb = out * n // be
    if kind in ("TL1", "TQ1_0"):  # five trits a byte as ceil(v * 256 / 243), four in the tail bytes
        five, four = {"TL1": (24, 2), "TQ1_0": (48, 4)}[kind]
        v5 = torch.randint(0, 243, (nb, five), generator=g, device="cuda", dtype=torch.int32)
        v4 = torch.randint(0, 81, (nb, four), generator=g, device="cuda", dtype=torch.int32) * 3
        b = ((torch.cat([v5, v4], 1) * 256 + 242) // 243).to(torch.uint8)
        d = 0.02 + 0.02 * torch.rand(nb, generator=g, device="cuda")
        return torch.cat([b, _half_bytes(d)], 1).reshape(-1)
    b = _bytes(g, nb, bb)
    d = _half_bytes(1e-3 * (0.5 + torch.rand(nb, generator=g, device="cuda")))
    at = {"Q8_0": 0, "Q3K": 108, "Q4K": 0, "Q5K": 0, "Q6K": 208}[kind]
    b[:, at:at + 2] = d
    if kind in ("Q4K", "Q5K"):  # the minimum's scale, about half the range below zero
        b[:, 2:4] = _half_bytes(d.view(torch.float16).float().reshape(-1) * (8.0 if kind == "Q4K" else 16.0))
    return b.reshape(-1)


def _delta_inputs(case, seed):
    g = _gen(seed)
    n, hk, hv = case["seqs"], case["hk"], case["hv"]
    rows = case["tokens"] or n
    s = {"state": 0.02 * _randn(g, n, hv, D, D)}
    if case["layer"]:
        ch = 2 * hk * D + hv * D
        s.update(qkv=_randn(g, n, ch), z=_randn(g, n, hv * D), beta_raw=_randn(g, n, hv), alpha_raw=_randn(g, n, hv),
                 dt_bias=_randn(g, hv), a_log=-torch.exp(_randn(g, hv) - 1.0), conv_w=0.5 * _randn(g, ch, 4),
                 norm_w=1.0 + 0.1 * _randn(g, D), ring=_randn(g, n, ch, 3), out=torch.empty(n, hv * D, device="cuda"))
        return s
    dt = torch.bfloat16 if case["bf16"] else torch.float32
    s.update(q=_randn(g, rows, hk, D).to(dt), k=_randn(g, rows, hk, D).to(dt), v=_randn(g, rows, hv, D).to(dt),
             beta=torch.sigmoid(_randn(g, rows, hv)), gate=-torch.nn.functional.softplus(_randn(g, rows, hv) - 1.0),
             out=torch.empty(rows, hv, D, device="cuda"))
    return s


def prepare(case, seed):
    _lib.init()
    family = case["family"]
    s = {"case": case}
    if family == "rotate":
        g = _gen(seed)
        rows, n = case["rows"], case["n"]
        x = _randn(g, rows, n)
        x[torch.rand(rows, n, generator=g, device="cuda") < 0.01] *= 20.0  # the outliers that rotation is for
        dt = torch.bfloat16 if case["bf16"] else torch.float32
        s["x"] = x.to(dt)
        s["signs"] = (torch.randint(0, 2, (n,), generator=g, device="cuda") * 2.0 - 1.0) if case["signs"] else None
        s["y"] = torch.empty(rows, n, dtype=dt, device="cuda") if case["store"] else None
        s["xq"] = torch.empty(rows, n, dtype=torch.int8, device="cuda") if case["quant"] else None
        s["scale"] = torch.empty(rows, device="cuda") if case["quant"] else None
    elif family in ("linear", "head"):
        g = _gen(seed)
        out, n, k = case["out_len"], case["in_len"], case.get("k", 1)
        payload = _payload(case, g)
        if case["kind"] in TERNARY:
            s["weight"] = Weight(QuantKind[case["kind"]], payload.cpu().numpy(), out, n, max_cols=k)
        else:
            s["payload"] = payload
        s["x"] = _randn(g, k, n)
        s["y"] = torch.empty(k, out, device="cuda")
        s["idx"] = torch.zeros(1, dtype=torch.int32, device="cuda")
    elif family == "delta":
        s.update(_delta_inputs(case, seed))
        if case["tokens"]:
            s["cu"] = np.concatenate([[0], np.cumsum(_lengths(case))]).astype(np.int32)
            need = _lib.lib().ouro_gdn_chunk_workspace_bytes(case["tokens"], case["seqs"], case["hv"], D, 64)
            s["work"] = torch.empty(need, dtype=torch.uint8, device="cuda")
    else:
        g = _gen(seed)
        lens, steps = _lengths(case), case["steps"]
        card = _card()
        pages = int(sum((int(l) + steps + 63) // 64 for l in lens))
        n = case["seqs"]
        s["stack"] = Stack(card, seed & 0xffffffff, max_seqs=n, max_tokens=case["tokens"],
                           max_ctx=int(lens.max()) + steps + 1, kv_pages=pages)
        s["cu"] = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        s["tokens"] = torch.randint(0, card.n_vocab, (case["tokens"],), generator=g, device="cuda", dtype=torch.int32)
        # the text that the decode steps continue with is given, as when a
        # known continuation is scored, so that the logits stay comparable
        s["forced"] = torch.randint(0, card.n_vocab, (steps, n), generator=g, device="cuda", dtype=torch.int32)
        s["next"] = torch.zeros(n, dtype=torch.int32, device="cuda")
        s["logits"] = torch.empty(2, n, card.n_vocab, device="cuda")
    return s


# ---- one pass ----

def _p(t):
    return None if t is None else t.data_ptr()


def run(s):
    case = s["case"]
    family = case["family"]
    if family == "rotate":
        dt = DT_BF16 if case["bf16"] else DT_F32
        call("ouro_fwht_rows", _p(s["x"]), dt, _p(s["y"]), dt, case["rows"], case["n"], case["block"], _p(s["signs"]),
             FWHT_INVERSE if case["inverse"] else 0, _p(s["xq"]), _p(s["scale"]), None)
        return [s["y"], s["xq"], s["scale"]]
    if family == "head":
        call("ouro_weight_matvec_argmax", s["weight"].handle, _p(s["x"]), _p(s["y"]), _p(s["idx"]), None)
        return [s["y"], s["idx"]]
    if family == "linear":
        if "weight" in s:
            call("ouro_weight_matmul", s["weight"].handle, _p(s["x"]), case["k"], _p(s["y"]), None)
        else:
            call("ouro_matmul_q", _p(s["payload"]), int(QuantKind[case["kind"]]), case["out_len"], case["in_len"],
                 _p(s["x"]), case["k"], _p(s["y"]), None)
        return s["y"]
    if family == "delta":
        n, hk, hv = case["seqs"], case["hk"], case["hv"]
        if case["tokens"]:
            call("ouro_gdn_chunk_prefill", _p(s["state"]), _p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["gate"]),
                 _p(s["beta"]), _p(s["out"]), s["cu"].ctypes.data, n, case["tokens"], hk, hv, D, 64,
                 GDN_L2NORM_QK | GDN_SCALE_Q, EPS, _p(s["work"]), None)
            return [s["out"], s["state"]]
        if case["layer"]:
            call("ouro_gdn_layer_decode", _p(s["qkv"]), _p(s["z"]), _p(s["beta_raw"]), _p(s["alpha_raw"]),
                 _p(s["dt_bias"]), _p(s["a_log"]), _p(s["conv_w"]), _p(s["norm_w"]), _p(s["ring"]), _p(s["state"]),
                 _p(s["out"]), n, hk, hv, D, GDN_V_GROUPED, EPS, None, None)
            return [s["out"], s["state"], s["ring"]]
        dt = DT_BF16 if case["bf16"] else DT_F32
        call("ouro_gdn_decode", _p(s["state"]), _p(s["q"]), _p(s["k"]), dt, _p(s["v"]), dt, _p(s["gate"]),
             _p(s["beta"]), _p(s["out"]), n, hk, hv, D, GDN_L2NORM_QK | GDN_SCALE_Q, EPS, None)
        return [s["out"], s["state"]]
    handle = s["stack"].handle
    call("ouro_stack_prefill", handle, _p(s["tokens"]), s["cu"].ctypes.data, case["seqs"], _p(s["next"]),
         _p(s["logits"][0]), None)
    for i in range(case["steps"]):
        last = i + 1 == case["steps"]
        call("ouro_stack_decode", handle, _p(s["forced"][i]), _p(s["next"]), _p(s["logits"][1]) if last else None, None)
    return s["logits"]


# ---- the work of one pass ----

def _stack_work(case):
    c = _card()
    e, f, d = c.n_embd, c.n_ff, c.head_dim
    di, dv, qd, kvd = c.ssm_n_k_heads * d, c.ssm_n_v_heads * d, c.n_head * d, c.n_head_kv * d
    attn = c.n_layer // c.full_attention_interval
    delta = c.n_layer - attn
    weights = delta * ((2 * di + 2 * dv + 2 * c.ssm_n_v_heads) * e + e * dv) + \
        attn * ((2 * qd + 2 * kvd) * e + e * qd) + c.n_layer * 3 * e * f
    head = c.n_vocab * e
    n, t, steps = case["seqs"], case["tokens"], case["steps"]
    lens = _lengths(case)
    state = delta * n * c.ssm_n_v_heads * d * d * 4
    keys = sum(int(l) * steps + steps * (steps + 1) // 2 for l in lens)  # read by all decode steps
    kv = attn * kvd * 4 * 2
    moved = (1 + steps) * ((weights + head) // 4) + state * (1 + 2 * steps) + kv * (t + keys) + \
        (t + n * steps) * e * 4 + 2 * n * c.n_vocab * 4
    products = 2 * (t + n * steps) * weights + 2 * n * (1 + steps) * head
    pairs = sum(int(l) * (int(l) + 1) // 2 for l in lens) + keys
    recur = (t + n * steps) * delta * c.ssm_n_v_heads * 6 * d * d
    return {"bytes": moved, "flops": products + 4 * attn * qd * pairs + recur}


def work(case):
    family = case["family"]
    if family == "rotate":
        n = case["rows"] * case["n"]
        size = 2 if case["bf16"] else 4
        moved = n * size * (2 if case["store"] else 1) + (n + 4 * case["rows"] if case["quant"] else 0) + \
            (4 * case["n"] if case["signs"] else 0)
        return {"bytes": moved, "flops": n * math.log2(case["block"])}
    if family in ("linear", "head"):
        out, n, k = case["out_len"], case["in_len"], case.get("k", 1)
        return {"bytes": QuantKind[case["kind"]].row_bytes(n) * out + 4 * k * (n + out), "flops": 2 * out * n * k}
    if family == "delta":
        n, hk, hv = case["seqs"], case["hk"], case["hv"]
        rows = case["tokens"] or n
        state = 2 * n * hv * D * D * 4
        if case["layer"]:
            ch = 2 * hk * D + hv * D
            rest = n * ch * 4 * 7 + n * hv * (2 * D + 2) * 4 + ch * 16
        else:
            rest = rows * (D * (2 * hk + hv) * (2 if case["bf16"] else 4) + hv * (8 + 4 * D))
        if not case["tokens"]:
            return {"bytes": state + rest, "flops": rows * hv * 6 * D * D}
        # per 64-token chunk and v-head: four 64x64x128 and three 64x128x128 products
        return {"bytes": state + rest, "flops": rows / 64 * hv * 2 * (4 * 64 * 64 * D + 3 * 64 * D * D)}
    return _stack_work(case)


def tolerance(case):
    """About four times the largest error against 64 bits over a few hundred
    drawn cases (rel / max): I2_S 3.6e-8 / 1.1e-7, the other linear kinds
    5.5e-7 / 2.1e-6, a delta-net step 1.5e-7 / 4.4e-6, its prefill (16-bit
    products of split operands) 5.1e-6 / 1.1e-4.  The stack's is the largest
    change of its logits when every norm moves in its last bit (_card):
    0.031 / 0.18, of which rel is held to 0.03."""
    family = case["family"]
    if family == "rotate":
        return "exact"
    if family in ("linear", "head"):
        return {"rel": 1.5e-7, "max": 5e-7} if case["kind"] == "I2_S" else {"rel": 2.2e-6, "max": 1e-5}
    if family == "delta":
        return {"rel": 2e-5, "max": 5e-4} if case["tokens"] else {"rel": 6e-7, "max": 2e-5}
    return {"rel": 0.03, "max": 0.6}


# ---- results in 64 bits ----

def _quant_rows(x):
    """int8 rows and the fp32 scale of quantize_row_i8_s."""
    amax = x.abs().amax(1).double().clamp_min(float(np.float32(1e-5)))
    s = (127.0 / amax).float()
    p = (x * s[:, None]).double()
    return torch.sign(p) * torch.floor(p.abs() + 0.5).clamp_max(128.0), s


def _trits(b, five, four, groups):
    """Trits of blocks b [nb, bytes]: bytes in `groups` (of five digits), then the four-digit tail."""
    b = b.to(torch.int32)
    out, at = [], 0
    for size, digits in [(gsize, 5) for gsize in groups] + [(four, 4)]:
        part = b[:, at:at + size]
        out += [((((part * 3 ** i) & 255) * 3) >> 8) - 1 for i in range(digits)]
        at += size
    return torch.cat(out, 1).double()


def _dequant(kind, payload, rows, n):
    """fp64 [rows, n] of payload bytes of whole rows."""
    if kind in DENSE:
        dt = {"F32": torch.float32, "F16": torch.float16, "BF16": torch.bfloat16}[kind]
        return payload.view(dt).reshape(rows, n).double()
    if kind == "I2_S":
        p = payload.reshape(-1, 32)
        return torch.stack([(p >> (6 - 2 * i)) & 3 for i in range(4)], 1).double().reshape(rows, n) - 1.0
    bb, _ = _blocks(kind)
    b = payload.reshape(-1, bb)

    def half(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).double()

    if kind in ("TL1", "TQ1_0"):
        five, four, groups = {"TL1": (24, 2, (16, 8)), "TQ1_0": (48, 4, (32, 16))}[kind]
        return (_trits(b, five, four, groups) * half(five + four)).reshape(rows, n)
    if kind == "Q8_0":
        return (b[:, 2:].contiguous().view(torch.int8).double() * half(0)).reshape(rows, n)
    if kind == "Q6K":
        lo, hi = b[:, :128].reshape(-1, 2, 2, 32).int(), b[:, 128:192].reshape(-1, 2, 1, 32).int()
        q = torch.stack([(lo[:, :, i % 2] >> (4 * (i // 2)) & 15) | ((hi[:, :, 0] >> (2 * i) & 3) << 4) for i in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        return ((q - 32).double().reshape(-1, 16, 16) * sc[:, :, None] * half(208)[:, :, None]).reshape(rows, n)
    if kind == "Q3K":
        hm, qs, sb = b[:, :32].int(), b[:, 32:96].reshape(-1, 2, 32).int(), b[:, 96:108].int()
        q = torch.stack([((qs[:, i // 4] >> (2 * (i % 4))) & 3) - 4 + 4 * ((hm >> i) & 1) for i in range(8)], 1)
        low = torch.cat([sb[:, :8] & 15, sb[:, :8] >> 4], 1)
        sc = low | torch.cat([(sb[:, 8:12] >> (2 * i) & 3) << 4 for i in range(4)], 1)
        return (q.double().reshape(-1, 16, 16) * (sc - 32).double()[:, :, None] * half(108)[:, :, None]).reshape(rows, n)
    # Q4K, Q5K: eight 32-element sub-blocks with a 6-bit scale and minimum each
    s = b[:, 4:16].int()
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | (s[:, :4] >> 6 << 4)], 1).double()
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | (s[:, 4:8] >> 6 << 4)], 1).double()
    qs = b[:, -128:].reshape(-1, 4, 1, 32).int()
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if kind == "Q5K":
        qh = b[:, 16:48].int()
        q = q + torch.stack([((qh >> i) & 1) << 4 for i in range(8)], 1)
    return (q.double() * (half(0) * sc)[:, :, None] - (half(2) * mn)[:, :, None]).reshape(rows, n)


def _exact_linear(case, seed):
    g = _gen(seed)
    kind, out, n, k = case["kind"], case["out_len"], case["in_len"], case.get("k", 1)
    payload = _payload(case, g)
    x = _randn(g, k, n)
    xs = x.double()
    scale = None
    if kind == "I2_S":
        xs, scale = _quant_rows(x)
    row = QuantKind[kind].row_bytes(n)
    step = max(1, (1 << 25) // n)
    y = torch.empty(k, out, dtype=torch.float64, device="cuda")
    for r in range(0, out, step):
        m = min(step, out - r)
        y[:, r:r + m] = xs @ _dequant(kind, payload[r * row:(r + m) * row], m, n).T
    if scale is not None:
        y = y / scale.double()[:, None] * payload[out * n // 4:out * n // 4 + 4].clone().view(torch.float32).double()
    return y


def _recur(state, q, k, v, gate, beta):
    """One step of the recurrence: state [n, hv, j, i] (i = the k index), vectors [n, hv, D]."""
    state *= torch.exp(gate)[:, :, None, None]
    dv = beta[:, :, None] * (v - torch.matmul(state, k[:, :, :, None])[..., 0])
    state += dv[:, :, :, None] * k[:, :, None, :]
    return torch.matmul(state, q[:, :, :, None])[..., 0]


def _heads(x, hv):
    """l2-normed head vectors [n, hk, D] for every v-head (v-head h uses k-head h % hk)."""
    x = x / (x.square().sum(-1, keepdim=True).sqrt() + EPS)
    return x.repeat(1, hv // x.shape[1], 1)


def _exact_delta(case, seed):
    s = {name: t.double() for name, t in _delta_inputs(case, seed).items()}
    n, hk, hv = case["seqs"], case["hk"], case["hv"]
    state = s["state"]
    if case["layer"]:
        di = hk * D
        taps = torch.cat([s["ring"], s["qkv"][:, :, None]], 2)
        c = torch.nn.functional.silu((taps * s["conv_w"]).sum(2))
        q, k = (_heads(c[:, i * di:(i + 1) * di].reshape(n, hk, D), hv) for i in (0, 1))
        beta = torch.sigmoid(s["beta_raw"])
        gate = s["a_log"] * torch.nn.functional.softplus(s["alpha_raw"] + s["dt_bias"])
        o = _recur(state, q / math.sqrt(D), k, c[:, 2 * di:].reshape(n, hv, D), gate, beta)
        z = s["z"].reshape(n, hv, D)
        y = o / (o.square().mean(-1, keepdim=True) + EPS).sqrt() * s["norm_w"] * torch.nn.functional.silu(z)
        y = y.reshape(n, hv // hk, hk, D).transpose(1, 2).reshape(n, hv * D)
        return [y, state, taps[:, :, 1:]]
    if not case["tokens"]:
        o = _recur(state, _heads(s["q"], hv) / math.sqrt(D), _heads(s["k"], hv), s["v"], s["gate"], s["beta"])
        return [o, state]
    lens = _lengths(case)
    if int(lens.max()) > 6000:
        return None
    start = torch.tensor(np.cumsum(lens) - lens, device="cuda")
    length = torch.tensor(lens, device="cuda")
    out = torch.empty(case["tokens"], hv, D, dtype=torch.float64, device="cuda")
    order = torch.argsort(length, descending=True)  # the sequences still running are a prefix
    st = state[order].contiguous()
    start, left = start[order], sorted(lens.tolist(), reverse=True)
    running = len(left)
    for t in range(left[0]):
        while left[running - 1] <= t:
            running -= 1
        at = start[:running] + t
        out[at] = _recur(st[:running], _heads(s["q"][at], hv) / math.sqrt(D), _heads(s["k"][at], hv), s["v"][at],
                         s["gate"][at], s["beta"][at])
    state[order] = st
    return [out, state]


def exact(case, seed):
    family = case["family"]
    if family == "linear":
        return _exact_linear(case, seed)
    if family == "head":
        y = _exact_linear(case, seed)
        return [y, None]
    if family == "delta":
        return _exact_delta(case, seed)
    if family == "stack":
        return None
    s = prepare(case, seed)
    n, block = case["n"], case["block"]
    x = s["x"].double()
    signs = s["signs"].double() if case["signs"] else torch.ones(n, dtype=torch.float64, device="cuda")
    if not case["inverse"]:
        x = x * signs
    h = 1
    while h < block:
        p = x.reshape(-1, 2, h)
        x = torch.stack([p[:, 0] + p[:, 1], p[:, 0] - p[:, 1]], 1).reshape(case["rows"], n)
        h *= 2
    x = x / math.sqrt(block)
    if case["inverse"]:
        x = x * signs
    scale = 127.0 / x.abs().amax(1).clamp_min(1e-5) if case["quant"] else None
    return [x if case["store"] else None, None, scale]
