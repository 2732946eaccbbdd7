"""The calls this backend is timed on.

Each case is a call, or a short chain of calls, that a program serving a
quantized model makes through the public entry points (rsllm_amd.backend):
weights prepared once and resident, activations on the device (or on the host
where the case is the host-pointer form), outputs in buffers the program keeps.

Kinds
  matmul   matmul_quant_f32_dev: one projection, f32 activations; decode (1..32
           tokens) and prefill (33..2048)
  ffn      matmul_quant_f32_dev twice: the up and down projections of a dense FFN
  bf16     matmul_q4k_bf16_dev: prefill with bf16 activations
  host     matmul_quant_f32: the host-pointer drop-in on resident weights
  int8     quantize_q8_0_batch_dev + matmul_q8_0_batch_dev: the int8-activation path
  lora     matmul_grouped_lora_down_dev: the grouped attention output projection
  shared   apply_shared_expert_dev: the SwiGLU expert every token takes
  moe      moe_routed_dev: the routed experts
  block    one DS-V4 decoder block's matmuls in order: q and kv projections,
           grouped output projection, output projection, router, shared expert,
           routed experts

Values: weights are random codes with block scales that make a product of unit
activations about 1 (so chained calls stay in the range a model's activations
have); activations are N(0, 1); routing draws experts uniformly without
replacement, with softmax weights.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rsllm_amd import backend as B
from rsllm_amd.ggml import GgmlType as G

MAX_FLOPS = 150e9  # no drawn case does more than the largest listed one


# ---------------------------------------------------------------------------
# Cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # A small attention projection (DS-V4 q_a) for four sequences decoded
        # together: the smallest call, mostly latency.
        {"name": "mla_q8_0_t4", "kind": "matmul", "dtype": "Q8_0", "out": 1024, "in": 4096, "tok": 4},
        # A dense FFN's two large projections, one decoded token: the weight
        # stream.
        {"name": "ffn_q6k_t1", "kind": "ffn", "dtype": "Q6_K", "embd": 4096, "ff": 14336, "tok": 1},
        # The same with eight sequences decoded together.
        {"name": "ffn_q6k_t8", "kind": "ffn", "dtype": "Q6_K", "embd": 4096, "ff": 14336, "tok": 8},
        # A square attention projection for a full decode batch.
        {"name": "attn_q8_0_t32", "kind": "matmul", "dtype": "Q8_0", "out": 4096, "in": 4096, "tok": 32},
        # The int8-activation path, activations quantised on the way in.
        {"name": "int8_q8_0_t16", "kind": "int8", "out": 4096, "in": 4096, "tok": 16},
        # The drop-in for a program whose activations live in host memory.
        {"name": "host_q4k_t1", "kind": "host", "dtype": "Q4_K", "out": 4096, "in": 4096, "tok": 1},
        # The grouped output projection over a prompt of ragged length.
        {"name": "lora_q8_0_t300", "kind": "lora", "dtype": "Q8_0", "groups": 8, "in": 4096,
         "rank": 1024, "tok": 300},
        # A dense FFN projection over a prompt, bf16 activations.
        {"name": "prefill_q4k_bf16_t512", "kind": "bf16", "out": 14336, "in": 4096, "tok": 512},
        # The attention output projection over a long prompt, f32 activations.
        {"name": "prefill_q8_0_t2000", "kind": "matmul", "dtype": "Q8_0", "out": 4096, "in": 8192,
         "tok": 2000},
        # Routed experts for a decode batch (64 wide experts, top-8).
        {"name": "moe_q4k_t32", "kind": "moe", "gate_up": "Q4_K", "down": "Q4_K", "experts": 64,
         "top": 8, "embd": 7168, "ff": 2048, "tok": 32},
        # DS-V4 routed experts over a prompt (256 experts, top-6, 2-bit formats).
        {"name": "moe_dsv4_t512", "kind": "moe", "gate_up": "IQ2_XXS", "down": "Q2_K",
         "experts": 256, "top": 6, "embd": 4096, "ff": 2048, "tok": 512},
        # All matmuls of one DS-V4 block for one decoded token.
        {"name": "block_dsv4_t1", "kind": "block", "gate_up": "Q4_K", "down": "Q2_K", "tok": 1},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _tokens(rng, most=2048):
    """Decode batches and prompts equally often, each over its whole range."""
    return _log_int(rng, 1, 32) if rng.random() < 0.5 else _log_int(rng, 33, most)


def _capped(tok, flops_per_token):
    return max(1, min(tok, int(MAX_FLOPS // flops_per_token)))


def _in_dim(rng, dtype, lo=1024, hi=14336):
    """Whole 256-element blocks; Q8_0 rows now and then only whole 32-element
    blocks."""
    if dtype == "Q8_0" and rng.random() < 0.15:
        return 32 * _log_int(rng, lo // 32, hi // 32)
    return 256 * _log_int(rng, lo // 256, hi // 256)


def draw(rng):
    kind = rng.choices(["matmul", "ffn", "bf16", "host", "int8", "lora", "shared", "moe", "block"],
                       [10, 2, 2, 2, 3, 3, 3, 5, 1])[0]
    if kind == "matmul":
        dt = rng.choice(["Q4_K", "Q6_K", "Q8_0"])
        out, ind = _log_int(rng, 256, 16384), _in_dim(rng, dt)
        return {"kind": kind, "dtype": dt, "out": out, "in": ind,
                "tok": _capped(_tokens(rng), 2 * out * ind)}
    if kind == "ffn":
        dt = rng.choice(["Q4_K", "Q6_K", "Q8_0"])
        e, f = 256 * _log_int(rng, 8, 32), 256 * _log_int(rng, 16, 56)
        return {"kind": kind, "dtype": dt, "embd": e, "ff": f, "tok": _log_int(rng, 1, 32)}
    if kind == "bf16":
        out, ind = _log_int(rng, 512, 16384), 256 * _log_int(rng, 4, 56)
        return {"kind": kind, "out": out, "in": ind,
                "tok": _capped(_log_int(rng, 33, 2048), 2 * out * ind)}
    if kind == "host":
        dt = rng.choice(["Q4_K", "Q6_K", "Q8_0"])
        return {"kind": kind, "dtype": dt, "out": _log_int(rng, 256, 14336), "in": _in_dim(rng, dt),
                "tok": _log_int(rng, 1, 64)}
    if kind == "int8":
        return {"kind": kind, "out": _log_int(rng, 256, 14336), "in": _in_dim(rng, "Q8_0"),
                "tok": _log_int(rng, 1, 64)}
    if kind == "lora":
        return {"kind": kind, "dtype": "Q8_0", "groups": rng.choice([4, 8, 16]),
                "in": 256 * _log_int(rng, 4, 16), "rank": 64 * _log_int(rng, 2, 16),
                "tok": _tokens(rng, 512)}
    if kind == "shared":
        dt = rng.choice(["Q8_0", "Q4_K", "Q6_K"])
        e, f = 256 * _log_int(rng, 8, 28), 256 * _log_int(rng, 4, 16)
        return {"kind": kind, "dtype": dt, "embd": e, "ff": f, "tok": _tokens(rng, 512)}
    if kind == "moe":
        if rng.random() < 0.35:
            return {"kind": kind, "gate_up": "Q4_K", "down": "Q4_K", "experts": 64, "top": 8,
                    "embd": 7168, "ff": 2048, "tok": _log_int(rng, 1, 128)}
        return {"kind": kind, "gate_up": rng.choice(["IQ2_XXS", "Q4_K"]), "down": "Q2_K",
                "experts": 256, "top": 6, "embd": 4096, "ff": 2048, "tok": _log_int(rng, 1, 500)}
    return {"kind": kind, "gate_up": rng.choice(["IQ2_XXS", "Q4_K"]), "down": "Q2_K",
            "tok": _log_int(rng, 2, 24)}


# ---------------------------------------------------------------------------
# Inputs, on the GPU, from the seed alone
# ---------------------------------------------------------------------------

def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + stream * 7919) % (1 << 62))
    return g


# Standard deviation of a weight of each format at block scale d = 1 (codes
# and sub-block scales uniform), and dmin / d that centres it.
_STD = {"Q4_K": 255.0, "Q6_K": 683.0, "Q8_0": 73.6, "Q2_K": 13.9, "IQ2_XXS": 42.0}
_DMIN = {"Q4_K": 7.5, "Q2_K": 1.5}


def _halves(n, scale, g):
    d = (torch.rand(n, 1, device="cuda", generator=g) + 0.5) * scale
    return d.to(torch.float16).view(torch.uint8).reshape(n, 2)


def _gguf(dtype, rows, in_dim, g):
    """Random GGUF rows, [blocks x block bytes] uint8."""
    t = G[dtype]
    n = rows * (in_dim // t.block_elements())
    b = torch.randint(0, 256, (n, t.block_bytes()), dtype=torch.uint8, device="cuda", generator=g)
    d = _halves(n, 1.0 / (_STD[dtype] * math.sqrt(in_dim)), g)
    if dtype == "Q8_0":
        b[:, 2:][b[:, 2:] == 128] = 129  # quantisers write -127..127
        b[:, 0:2] = d
    elif dtype == "Q6_K":
        s = b[:, 192:208].view(torch.int8)
        s.copy_(s >> 1)  # -64..63
        b[:, 208:210] = d
    elif dtype == "IQ2_XXS":
        b[:, 0:2] = d
    else:
        dmin = _halves(n, _DMIN[dtype] / (_STD[dtype] * math.sqrt(in_dim)), g)
        at = 0 if dtype == "Q4_K" else 80
        b[:, at:at + 2], b[:, at + 2:at + 4] = d, dmin
    return b


def _resident(dtype, rows, in_dim, seed, stream):
    """A weight as a program keeps it: the device layout."""
    raw = _gguf(dtype, rows, in_dim, _gen(seed, stream)).reshape(-1)
    if dtype == "Q4_K":
        return raw
    w = torch.empty_like(raw)
    B.prepare_weights_dev(w.data_ptr(), raw.data_ptr(), raw.numel(), G[dtype], in_dim,
                          torch.cuda.current_stream().cuda_stream)
    return w


def _acts(tok, dim, seed, stream):
    return torch.randn(tok, dim, device="cuda", generator=_gen(seed, stream))


def _routing(tok, experts, top, seed, stream):
    g = _gen(seed, stream)
    ids = torch.rand(tok, experts, device="cuda", generator=g).topk(top, dim=1).indices
    w = torch.softmax(torch.randn(tok, top, device="cuda", generator=g), dim=1)
    return ids.to(torch.int32).contiguous(), w.contiguous()


class _HostModel:
    """Weights resident under their host address for as long as this lives."""

    def __init__(self, host, dtype, in_dim, seed):
        self.host = host
        self.model = B.model_upload(int(seed % (1 << 64)).to_bytes(32, "little"),
                                    [("w", host, G[dtype], in_dim)])

    def __del__(self):
        B.model_release(self.model)


BLOCK = {"embd": 4096, "q_rank": 1024, "heads": 32768, "kv": 512, "groups": 8, "group_in": 4096,
         "rank": 1024, "experts": 256, "top": 6, "ff": 2048}


def _block_weights(case):
    """(name, dtype, rows, in_dim) of a block's quantized weights, in order."""
    b = BLOCK
    e, f, n = b["embd"], b["ff"], b["experts"]
    return [("q_a", "Q8_0", b["q_rank"], e), ("q_b", "Q8_0", b["heads"], b["q_rank"]),
            ("kv", "Q8_0", b["kv"], e),
            ("o_a", "Q8_0", b["groups"] * b["rank"], b["group_in"]),
            ("o_b", "Q8_0", e, b["groups"] * b["rank"]),
            ("s_gate", "Q8_0", f, e), ("s_up", "Q8_0", f, e), ("s_down", "Q8_0", e, f),
            ("gate", case["gate_up"], n * f, e), ("up", case["gate_up"], n * f, e),
            ("down", case["down"], n * e, f)]


def _empty(*shape, dtype=torch.float32):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def prepare(case, seed):
    kind, t = case["kind"], case["tok"]
    B.init(0)
    s = {"case": case, "stream": torch.cuda.current_stream().cuda_stream}
    if kind == "matmul":
        s["w"] = _resident(case["dtype"], case["out"], case["in"], seed, 1)
        s["x"] = _acts(t, case["in"], seed, 2)
        s["y"] = _empty(t, case["out"])
    elif kind == "ffn":
        s["w_up"] = _resident(case["dtype"], case["ff"], case["embd"], seed, 1)
        s["w_down"] = _resident(case["dtype"], case["embd"], case["ff"], seed, 3)
        s["x"] = _acts(t, case["embd"], seed, 2)
        s["h"], s["y"] = _empty(t, case["ff"]), _empty(t, case["embd"])
    elif kind == "bf16":
        s["w"] = _resident("Q4_K", case["out"], case["in"], seed, 1)
        s["x"] = _acts(t, case["in"], seed, 2).to(torch.bfloat16)
        s["y"] = _empty(t, case["out"])
    elif kind == "host":
        host = _gguf(case["dtype"], case["out"], case["in"], _gen(seed, 1)).reshape(-1).cpu().numpy()
        s["model"] = _HostModel(host, case["dtype"], case["in"], seed)
        s["x"] = _acts(t, case["in"], seed, 2).cpu().numpy().reshape(-1)
        s["y"] = np.empty(t * case["out"], np.float32)
    elif kind == "int8":
        blocks = case["in"] // 32
        s["w"] = _resident("Q8_0", case["out"], case["in"], seed, 1)
        s["x"] = _acts(t, case["in"], seed, 2)
        s["xq"], s["scale"] = _empty(t, blocks * 32, dtype=torch.int8), _empty(t, blocks)
        s["status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
        s["y"] = _empty(t, case["out"])
    elif kind == "lora":
        s["w"] = _resident(case["dtype"], case["groups"] * case["rank"], case["in"], seed, 1)
        s["x"] = _acts(t, case["groups"] * case["in"], seed, 2)
        s["y"] = _empty(t, case["groups"] * case["rank"])
    elif kind == "shared":
        e, f = case["embd"], case["ff"]
        for k, (n, rows, ind) in enumerate((("gate", f, e), ("up", f, e), ("down", e, f))):
            s[n] = _resident(case["dtype"], rows, ind, seed, 3 + k)
        s["x"], s["y"] = _acts(t, e, seed, 2), _empty(t, e)
    elif kind == "moe":
        e, f, n = case["embd"], case["ff"], case["experts"]
        for k, (name, dt, rows, ind) in enumerate((("gate", case["gate_up"], n * f, e),
                                                   ("up", case["gate_up"], n * f, e),
                                                   ("down", case["down"], n * e, f))):
            s[name] = _resident(dt, rows, ind, seed, 3 + k)
        s["x"], s["y"] = _acts(t, e, seed, 2), _empty(t, e)
        s["ids"], s["wts"] = _routing(t, n, case["top"], seed, 6)
    else:
        b = BLOCK
        for k, (name, dt, rows, ind) in enumerate(_block_weights(case)):
            s[name] = _resident(dt, rows, ind, seed, 10 + k)
        s["router"] = torch.randn(b["experts"], b["embd"], device="cuda",
                                  generator=_gen(seed, 30)) / math.sqrt(b["embd"])
        s["x"] = _acts(t, b["embd"], seed, 2)
        s["ids"], s["wts"] = _routing(t, b["experts"], b["top"], seed, 6)
        s["q1"], s["q2"], s["kv_y"] = _empty(t, b["q_rank"]), _empty(t, b["heads"]), _empty(t, b["kv"])
        s["a"], s["h"] = _empty(t, b["groups"] * b["rank"]), _empty(t, b["embd"])
        s["logits"], s["y"] = _empty(t, b["experts"]), _empty(t, b["embd"])
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------

def _matmul(y, w, x, tok, in_dim, out_dim, dtype, stream):
    B.matmul_quant_f32_dev(y.data_ptr(), tok * out_dim, w.data_ptr(), w.numel(), x.data_ptr(),
                           tok * in_dim, tok, in_dim, out_dim, G[dtype], stream)


def _shared(y, x, gate, up, down, dtype, tok, e, f, stream):
    dt = G[dtype]
    B.apply_shared_expert_dev(y.data_ptr(), tok * e, x.data_ptr(), tok * e, gate.data_ptr(),
                              gate.numel(), dt, up.data_ptr(), up.numel(), dt, down.data_ptr(),
                              down.numel(), dt, tok, e, f, 10.0, stream)


def _moe(y, x, s, c, tok, e, f, n, top):
    B.moe_routed_dev(y.data_ptr(), tok * e, x.data_ptr(), tok * e, s["gate"].data_ptr(),
                     s["up"].data_ptr(), s["gate"].numel(), s["down"].data_ptr(),
                     s["down"].numel(), s["ids"].data_ptr(), s["wts"].data_ptr(), tok * top, tok,
                     e, f, n, top, G[c["gate_up"]], G[c["down"]], 10.0, s["stream"])


def _lora(y, w, x, tok, groups, in_dim, rank, dtype, stream):
    B.matmul_grouped_lora_down_dev(y.data_ptr(), tok * groups * rank, w.data_ptr(), w.numel(),
                                   x.data_ptr(), tok * groups * in_dim, tok, groups, in_dim, rank,
                                   G[dtype], stream)


def run(s):
    c, st = s["case"], s["stream"]
    kind, t = c["kind"], c["tok"]
    if kind == "matmul":
        _matmul(s["y"], s["w"], s["x"], t, c["in"], c["out"], c["dtype"], st)
        return s["y"]
    if kind == "ffn":
        _matmul(s["h"], s["w_up"], s["x"], t, c["embd"], c["ff"], c["dtype"], st)
        _matmul(s["y"], s["w_down"], s["h"], t, c["ff"], c["embd"], c["dtype"], st)
        return [s["h"], s["y"]]
    if kind == "bf16":
        B.matmul_q4k_bf16_dev(s["y"].data_ptr(), t * c["out"], s["w"].data_ptr(), s["w"].numel(),
                              s["x"].data_ptr(), t * c["in"], t, c["in"], c["out"], G.Q4_K, st)
        return s["y"]
    if kind == "host":
        B.matmul_quant_f32(s["y"], s["model"].host, s["x"], t, c["in"], c["out"], G[c["dtype"]])
        return s["y"]
    if kind == "int8":
        B.quantize_q8_0_batch_dev(s["x"].data_ptr(), s["x"].numel(), s["xq"].data_ptr(),
                                  s["xq"].numel(), s["scale"].data_ptr(), s["scale"].numel(), t,
                                  c["in"], s["status"].data_ptr(), st)
        B.matmul_q8_0_batch_dev(s["y"].data_ptr(), t * c["out"], s["w"].data_ptr(), s["w"].numel(),
                                s["xq"].data_ptr(), s["xq"].numel(), s["scale"].data_ptr(),
                                s["scale"].numel(), t, c["in"], c["out"], st)
        return [s["xq"], s["scale"], s["status"], s["y"]]
    if kind == "lora":
        _lora(s["y"], s["w"], s["x"], t, c["groups"], c["in"], c["rank"], c["dtype"], st)
        return s["y"]
    if kind == "shared":
        _shared(s["y"], s["x"], s["gate"], s["up"], s["down"], c["dtype"], t, c["embd"], c["ff"], st)
        return s["y"]
    if kind == "moe":
        s["y"].zero_()  # the call accumulates
        _moe(s["y"], s["x"], s, c, t, c["embd"], c["ff"], c["experts"], c["top"])
        return s["y"]
    b = BLOCK
    e = b["embd"]
    _matmul(s["q1"], s["q_a"], s["x"], t, e, b["q_rank"], "Q8_0", st)
    _matmul(s["q2"], s["q_b"], s["q1"], t, b["q_rank"], b["heads"], "Q8_0", st)
    _matmul(s["kv_y"], s["kv"], s["x"], t, e, b["kv"], "Q8_0", st)
    _lora(s["a"], s["o_a"], s["q2"], t, b["groups"], b["group_in"], b["rank"], "Q8_0", st)
    _matmul(s["h"], s["o_b"], s["a"], t, b["groups"] * b["rank"], e, "Q8_0", st)
    B.matmul_weight_f32_dev(s["logits"].data_ptr(), t * b["experts"], s["router"].data_ptr(),
                            s["router"].numel() * 4, s["h"].data_ptr(), t * e, t, e, b["experts"],
                            G.F32, st)
    _shared(s["y"], s["h"], s["s_gate"], s["s_up"], s["s_down"], "Q8_0", t, e, b["ff"], st)
    _moe(s["y"], s["h"], s, c, t, e, b["ff"], b["experts"], b["top"])
    return [s["kv_y"], s["h"], s["logits"], s["y"]]


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------

def _weight_bytes(dtype, rows, in_dim):
    return rows * G[dtype].row_bytes(in_dim)


def _moe_work(gate_up, down, experts, top, e, f, t):
    """Each expert some token takes is read once: of `experts`, this many on
    average."""
    active = experts * (1.0 - (1.0 - top / experts) ** t)
    per = 2 * _weight_bytes(gate_up, f, e) + _weight_bytes(down, e, f)
    return active * per + 2 * t * e * 4 + t * top * 8, t * top * 6.0 * e * f


def work(case):
    kind, t = case["kind"], case["tok"]
    if kind in ("matmul", "host", "bf16"):
        dt = case.get("dtype", "Q4_K")
        nbytes = (_weight_bytes(dt, case["out"], case["in"]) +
                  t * case["in"] * (2 if kind == "bf16" else 4) + t * case["out"] * 4)
        flops = 2.0 * t * case["in"] * case["out"]
    elif kind == "ffn":
        e, f, dt = case["embd"], case["ff"], case["dtype"]
        nbytes = _weight_bytes(dt, f, e) + _weight_bytes(dt, e, f) + t * (2 * e + 2 * f) * 4
        flops = 4.0 * t * e * f
    elif kind == "int8":
        blocks = case["in"] // 32
        nbytes = (_weight_bytes("Q8_0", case["out"], case["in"]) + t * case["in"] * 4 +
                  2 * t * blocks * 36 + t * case["out"] * 4)
        flops = 2.0 * t * case["in"] * case["out"]
    elif kind == "lora":
        g, d, r = case["groups"], case["in"], case["rank"]
        nbytes = _weight_bytes(case["dtype"], g * r, d) + t * g * (d + r) * 4
        flops = 2.0 * t * g * d * r
    elif kind == "shared":
        e, f, dt = case["embd"], case["ff"], case["dtype"]
        nbytes = 2 * _weight_bytes(dt, f, e) + _weight_bytes(dt, e, f) + 2 * t * e * 4
        flops = 6.0 * t * e * f
    elif kind == "moe":
        nbytes, flops = _moe_work(case["gate_up"], case["down"], case["experts"], case["top"],
                                  case["embd"], case["ff"], t)
    else:
        b = BLOCK
        nbytes, flops = _moe_work(case["gate_up"], case["down"], b["experts"], b["top"], b["embd"],
                                  b["ff"], t)
        for _, dt, rows, ind in _block_weights(case)[:8]:
            nbytes += _weight_bytes(dt, rows, ind)
            flops += 2.0 * t * rows * ind
        nbytes += b["experts"] * b["embd"] * 4
        nbytes += 4 * t * (2 * b["embd"] + 2 * b["q_rank"] + 2 * b["heads"] + b["kv"] + 2 * b["groups"] *
                           b["rank"] + 5 * b["embd"] + b["experts"])
        flops += 2.0 * t * b["experts"] * b["embd"]
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """The int8 path computes in a fixed order on whole numbers: exact. Decode
    holds activations to about 16 bits of each group's largest value; prompts of
    more than 32 tokens may hold them in f16 (11 bits) for the matrix cores."""
    kind, t = case["kind"], case["tok"]
    if kind == "int8":
        return "exact"
    if kind == "moe":
        return {"rel": 2e-4}
    if kind == "block":
        return {"rel": 4e-4}
    if t > 32:
        return {"rel": 2e-3}
    return {"rel": 2e-4}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------

# The IQ2_XXS format's 256 magnitude groups: digit j of a base-3 number is
# element j's magnitude (0: 8, 1: 25, 2: 43).
_IQ2_CODES = """
0 2 4 6 8 10 12 18 20 24 26 28 30 36 42 46 48 54 56 62 74 82 84 90 94 108 138 150 162 164 182 218
244 246 252 262 264 270 272 276 288 298 300 306 318 324 326 330 342 356 376 378 388 412 414 432 462
480 486 490 492 498 510 514 516 522 524 546 570 594 650 660 730 732 738 748 756 774 786 792 796 810
816 828 846 854 864 912 922 972 978 990 994 1006 1026 1068 1100 1134 1148 1216 1218 1224 1242 1270
1296 1300 1368 1414 1458 1460 1466 1488 1504 1512 1514 1564 1572 1620 1622 1702 1704 1710 1728 1742
1782 1810 1830 1926 1950 1962 2010 2136 2188 2190 2196 2202 2206 2208 2214 2220 2228 2232 2242 2244
2250 2268 2286 2314 2322 2326 2350 2358 2382 2390 2400 2430 2436 2448 2484 2500 2522 2532 2592 2674
2676 2682 2700 2704 2754 2796 2800 2810 2866 2898 2916 2922 2926 2932 2934 2970 2976 3000 3026 3072
3142 3222 3224 3248 3322 3360 3402 3412 3418 3450 3510 3570 3648 3654 3672 3696 3726 3766 3822 3852
3888 3892 3978 3980 4026 4160 4374 4376 4382 4402 4430 4458 4470 4482 4546 4618 4620 4626 4630 4644
4662 4698 4730 4764 4786 4806 4824 4862 4944 5032 5106 5112 5124 5130 5176 5198 5238 5296 5346 5366
5376 5464 5644 5688 5834 5868 5890 5920 5994 6090 6354 6402
"""


def _iq2_grid():
    codes = torch.tensor([int(v) for v in _IQ2_CODES.split()], device="cuda")
    mags = torch.tensor([8.0, 25.0, 43.0], dtype=torch.float64, device="cuda")
    return torch.stack([mags[(codes // 3 ** j) % 3] for j in range(8)], dim=1)


def _f16_col(b, at):
    return b[:, at:at + 2].contiguous().view(torch.float16).to(torch.float64)


def _values(dtype, b):
    """GGUF blocks [n x bytes] -> [n x elements] float64."""
    f64 = torch.float64
    n = b.shape[0]
    if dtype == "Q8_0":
        return b[:, 2:].contiguous().view(torch.int8).to(f64) * _f16_col(b, 0)
    if dtype == "Q4_K":
        s = b[:, 4:16].to(torch.int64)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | (s[:, 0:4] >> 6 << 4)], dim=1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | (s[:, 4:8] >> 6 << 4)], dim=1)
        q = b[:, 16:].reshape(n, 4, 1, 32)
        q = torch.cat([q & 15, q >> 4], dim=2).reshape(n, 8, 32).to(f64)
        w = (_f16_col(b, 0) * sc.to(f64))[:, :, None] * q
        return (w - (_f16_col(b, 2) * mn.to(f64))[:, :, None]).reshape(n, 256)
    if dtype == "Q6_K":
        ql, qh = b[:, 0:128].reshape(n, 2, 2, 32), b[:, 128:192].reshape(n, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], dim=2)  # [n, half, quarter, 32]
        hi = torch.cat([(qh >> (2 * k)) & 3 for k in range(4)], dim=2)
        q = (lo | (hi << 4)).to(f64) - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).to(f64) * _f16_col(b, 208)
        return (q.reshape(n, 16, 16) * sc[:, :, None]).reshape(n, 256)
    if dtype == "Q2_K":
        qs = b[:, 16:80].reshape(n, 2, 1, 32)
        q = torch.cat([(qs >> (2 * k)) & 3 for k in range(4)], dim=2).reshape(n, 16, 16).to(f64)
        sc = b[:, 0:16].to(torch.int64)
        w = (_f16_col(b, 80) * (sc & 15).to(f64))[:, :, None] * q
        return (w - (_f16_col(b, 82) * (sc >> 4).to(f64))[:, :, None]).reshape(n, 256)
    assert dtype == "IQ2_XXS"
    qs = b[:, 2:66].reshape(n, 8, 8)
    mag = _iq2_grid()[qs[:, :, 0:4].to(torch.int64)]  # [n, 8, 4, 8]
    aux = qs[:, :, 4:8].to(torch.int64)
    aux = aux[..., 0] | aux[..., 1] << 8 | aux[..., 2] << 16 | aux[..., 3] << 24
    sign7 = torch.stack([(aux >> (7 * k)) & 127 for k in range(4)], dim=2)
    bits = torch.stack([(sign7 >> k) & 1 for k in range(7)], dim=3)
    bits = torch.cat([bits, bits.sum(dim=3, keepdim=True) & 1], dim=3)
    db = _f16_col(b, 0) * ((aux >> 28).to(f64) + 0.5) * 0.25
    return (mag * (1.0 - 2.0 * bits.to(f64)) * db[:, :, None, None]).reshape(n, 256)


def _mul(x, dtype, b, rows, in_dim):
    """x [t x in] @ W^T in float64, a few rows of W at a time."""
    t = G[dtype]
    per = in_dim // t.block_elements()
    step = max(1, (1 << 25) // in_dim)
    y = torch.empty(x.shape[0], rows, dtype=torch.float64, device="cuda")
    for r in range(0, rows, step):
        k = min(step, rows - r)
        w = _values(dtype, b[r * per:(r + k) * per]).reshape(k, in_dim)
        y[:, r:r + k] = x @ w.T
    return y


def _swiglu(g, u, c=10.0):
    g, u = g.clamp(max=c), u.clamp(min=-c, max=c)
    return g * torch.sigmoid(g) * u


def _exact_moe(x, gate, up, down, gate_up_t, down_t, ids, wts, e, f, out):
    pg = f * (e // G[gate_up_t].block_elements())
    pd = e * (f // G[down_t].block_elements())
    for ex in torch.unique(ids).tolist():
        tok, slot = torch.nonzero(ids == ex, as_tuple=True)
        xe = x[tok]
        a = _swiglu(_mul(xe, gate_up_t, gate[ex * pg:(ex + 1) * pg], f, e),
                    _mul(xe, gate_up_t, up[ex * pg:(ex + 1) * pg], f, e))
        y = _mul(a, down_t, down[ex * pd:(ex + 1) * pd], e, f)
        out.index_add_(0, tok, y * wts[tok, slot].to(torch.float64)[:, None])
    return out


def exact(case, seed):
    kind, t, f64 = case["kind"], case["tok"], torch.float64

    def blocks(dtype, rows, ind, stream):
        return _gguf(dtype, rows, ind, _gen(seed, stream))

    if kind in ("matmul", "host", "bf16"):
        dt = case.get("dtype", "Q4_K")
        x = _acts(t, case["in"], seed, 2)
        x = x.to(torch.bfloat16).to(f64) if kind == "bf16" else x.to(f64)
        y = _mul(x, dt, blocks(dt, case["out"], case["in"], 1), case["out"], case["in"])
        return y.cpu().numpy().reshape(-1) if kind == "host" else y
    if kind == "ffn":
        e, f, dt = case["embd"], case["ff"], case["dtype"]
        h = _mul(_acts(t, e, seed, 2).to(f64), dt, blocks(dt, f, e, 1), f, e)
        return [h, _mul(h, dt, blocks(dt, e, f, 3), e, f)]
    if kind == "int8":
        # the quantised activations are whole numbers of a 32-bit recipe, not
        # sums: only the product has a 64-bit value
        x = _acts(t, case["in"], seed, 2).reshape(t, -1, 32)
        d = x.abs().amax(dim=2, keepdim=True) / 127.0
        q = torch.round(x * (1.0 / d)).clamp(-128, 127).to(f64) * d.to(f64)
        w = blocks("Q8_0", case["out"], case["in"], 1)
        return [None, None, None, _mul(q.reshape(t, -1), "Q8_0", w, case["out"], case["in"])]
    if kind == "lora":
        g, d, r = case["groups"], case["in"], case["rank"]
        x = _acts(t, g * d, seed, 2).to(f64).reshape(t, g, d)
        w = blocks(case["dtype"], g * r, d, 1)
        per = w.shape[0] // g
        return torch.cat([_mul(x[:, k].contiguous(), case["dtype"], w[k * per:(k + 1) * per], r, d)
                          for k in range(g)], dim=1)
    if kind == "shared":
        e, f, dt = case["embd"], case["ff"], case["dtype"]
        x = _acts(t, e, seed, 2).to(f64)
        a = _swiglu(_mul(x, dt, blocks(dt, f, e, 3), f, e), _mul(x, dt, blocks(dt, f, e, 4), f, e))
        return _mul(a, dt, blocks(dt, e, f, 5), e, f)
    if kind == "moe":
        e, f, n, gu, dn = case["embd"], case["ff"], case["experts"], case["gate_up"], case["down"]
        ids, wts = _routing(t, n, case["top"], seed, 6)
        return _exact_moe(_acts(t, e, seed, 2).to(f64), blocks(gu, n * f, e, 3),
                          blocks(gu, n * f, e, 4), blocks(dn, n * e, f, 5), gu, dn, ids, wts, e, f,
                          torch.zeros(t, e, dtype=f64, device="cuda"))
    b = BLOCK
    e, f = b["embd"], b["ff"]
    w = {name: (dt, blocks(dt, rows, ind, 10 + k), rows, ind)
         for k, (name, dt, rows, ind) in enumerate(_block_weights(case))}

    def mul(x, name):
        dt, blk, rows, ind = w[name]
        return _mul(x, dt, blk, rows, ind)

    x = _acts(t, e, seed, 2).to(f64)
    q = mul(mul(x, "q_a"), "q_b").reshape(t, b["groups"], b["group_in"])
    per = w["o_a"][1].shape[0] // b["groups"]
    a = torch.cat([_mul(q[:, k].contiguous(), "Q8_0", w["o_a"][1][k * per:(k + 1) * per], b["rank"],
                        b["group_in"]) for k in range(b["groups"])], dim=1)
    h = mul(a, "o_b")
    router = torch.randn(b["experts"], e, device="cuda", generator=_gen(seed, 30)) / math.sqrt(e)
    ids, wts = _routing(t, b["experts"], b["top"], seed, 6)
    y = mul(_swiglu(mul(h, "s_gate"), mul(h, "s_up")), "s_down")
    y = _exact_moe(h, w["gate"][1], w["up"][1], w["down"][1], case["gate_up"], case["down"], ids,
                   wts, e, f, y)
    return [mul(x, "kv"), h, h @ router.to(f64).T, y]
