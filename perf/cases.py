"""Workloads the library is timed on: its public operators over the sizes,
layouts, types and options that programs call them with.

Every case names an operator and its extents. `listed` holds one case of each
kind of use; `draw` gives further ones of the same ranges. The reference
results come from plain torch in 64 bits.
"""
from __future__ import annotations

import math

import torch

import __graft_entry__

_pkg = __graft_entry__.load_package()

_MAX_MACS = 2048 * 11008 * 4096      # the largest listed matmul
_MAX_SCORES = 32 * 2048 * 2048       # the largest listed attention


def listed():
    return [
        # The smallest dispatch of the benchmark configurations: 128x512x256,
        # where the call itself is what costs.
        {"name": "matmul_small", "op": "matmul", "dtype": "f16", "m": 128,
         "n": 512, "k": 256, "b_transposed": False, "a_transposed": False,
         "out_f32": False},
        # A projection of a whole prompt, weights as linalg.matmul has them.
        {"name": "matmul_prompt", "op": "matmul", "dtype": "f16", "m": 2048,
         "n": 11008, "k": 4096, "b_transposed": False, "a_transposed": False,
         "out_f32": False},
        # Sizes that no tile divides, in rows that are not 16-byte aligned: a
        # dynamic shape, f32 result.
        {"name": "matmul_odd", "op": "matmul", "dtype": "f16", "m": 777,
         "n": 3001, "k": 4099, "b_transposed": False, "a_transposed": False,
         "out_f32": True},
        # The headline quantized product: exact i32 sums, column-major B.
        {"name": "matmul_int8", "op": "matmul", "dtype": "i8", "m": 4096,
         "n": 4096, "k": 4096, "b_transposed": True, "a_transposed": False,
         "out_f32": False},
        # The batched micro model of the integration tests.
        {"name": "batch_matmul", "op": "linear", "batch": 4, "m": 1024,
         "n": 1024, "k": 128, "b_transposed": False, "bias": False,
         "activation": "none", "multiplier": False},
        # A linear layer over a prompt of 300 tokens with its bias, GELU and
        # gate fused, weights stored as [out, in].
        {"name": "linear_gated", "op": "linear", "batch": 1, "m": 300,
         "n": 11008, "k": 4096, "b_transposed": True, "bias": True,
         "activation": "gelu_tanh", "multiplier": True},
        # A gated feed-forward block for one token, recorded once in a command
        # buffer and submitted for each token: gate, up and down projections
        # with a barrier between them.
        {"name": "ffn_token", "op": "ffn", "m": 1, "hidden": 4096,
         "inner": 11008},
        # Weight-only quantization, one token.
        {"name": "w8a16_token", "op": "w8a16", "m": 1, "n": 11008, "k": 4096,
         "w_transposed": False},
        # The same over a prompt, weights stored as [out, in].
        {"name": "w8a16_prompt", "op": "w8a16", "m": 512, "n": 11008,
         "k": 4096, "w_transposed": True},
        # Causal self-attention over a whole prompt.
        {"name": "attention_prompt", "op": "attention", "batch": 1,
         "heads": 32, "kv_heads": 32, "seq_q": 2048, "seq_kv": 2048,
         "cache": 2048, "d": 128, "dv": 128, "causal": True, "mask": False,
         "out_f32": False},
        # One new token of each of four sequences against the filled part of
        # a longer KV cache, grouped-query heads.
        {"name": "attention_token", "op": "attention", "batch": 4,
         "heads": 32, "kv_heads": 8, "seq_q": 1, "seq_kv": 3001,
         "cache": 4096, "d": 128, "dv": 128, "causal": False, "mask": False,
         "out_f32": False},
        # Grouped heads with an additive mask over a length that nothing
        # divides.
        {"name": "attention_masked", "op": "attention", "batch": 2,
         "heads": 9, "kv_heads": 3, "seq_q": 777, "seq_kv": 777, "cache": 777,
         "d": 64, "dv": 64, "causal": False, "mask": True, "out_f32": False},
    ]


# ------------------------------------------------------------------- draws --

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _extent(rng, lo, hi):
    """Log-uniform, a multiple of 128, of 8, or whatever comes."""
    v, unit = _log(rng, lo, hi), rng.choice((128, 128, 8, 8, 1))
    return min(hi, max(lo, unit, v // unit * unit))


def _matmul_extents(rng, batch=1):
    while True:
        # a token or a few, a prompt, or anything between
        m = rng.choice((rng.randint(1, 16), _log(rng, 1, 2048),
                        _log(rng, 64, 2048)))
        n, k = _extent(rng, 64, 11008), _extent(rng, 64, 11008)
        if batch * m * n * k <= _MAX_MACS // 2:
            return m, n, k


def draw(rng):
    op = rng.choice(("matmul", "matmul_i8", "linear", "ffn", "w8a16",
                     "attention", "attention"))
    if op == "matmul":
        m, n, k = _matmul_extents(rng)
        return {"op": "matmul", "dtype": "f16", "m": m, "n": n, "k": k,
                "b_transposed": rng.random() < 0.5,
                "a_transposed": rng.random() < 0.2,
                "out_f32": rng.random() < 0.3}
    if op == "matmul_i8":
        m, n, k = _matmul_extents(rng)
        return {"op": "matmul", "dtype": "i8", "m": m, "n": n, "k": k,
                "b_transposed": rng.random() < 0.5, "a_transposed": False,
                "out_f32": False}
    if op == "linear":
        batch = rng.choice((1, 1, 2, 4, 9))
        m, n, k = _matmul_extents(rng, batch)
        return {"op": "linear", "batch": batch, "m": m, "n": n, "k": k,
                "b_transposed": rng.random() < 0.5,
                "bias": rng.random() < 0.5,
                "activation": rng.choice(("none", "relu", "gelu_tanh",
                                          "silu")),
                "multiplier": rng.random() < 0.5}
    if op == "ffn":
        return {"op": "ffn", "m": _log(rng, 1, 64),
                "hidden": 64 * rng.randint(8, 64),
                "inner": 64 * rng.randint(16, 172)}
    if op == "w8a16":
        m, n, k = _matmul_extents(rng)
        return {"op": "w8a16", "m": m, "n": n, "k": k,
                "w_transposed": rng.random() < 0.5}
    while True:
        batch = rng.choice((1, 1, 2, 4, 8))
        kv_heads = rng.choice((1, 2, 3, 4, 8))
        heads = kv_heads * rng.choice((1, 3, 4, 8))
        d = rng.choice((64, 64, 128, 128, 128, 80, 96, 40, 192))
        dv = 128 if d == 192 else d
        token = rng.random() < 0.4
        if token:  # one token or a few against a cache
            seq_q, seq_kv = rng.choice((1, 1, 1, 2, 5)), _log(rng, 64, 8192)
        else:
            seq_q = seq_kv = _extent(rng, 64, 2048)
        if batch * heads * seq_q * seq_kv <= _MAX_SCORES // 2:
            break
    mask = rng.random() < 0.3
    return {"op": "attention", "batch": batch, "heads": heads,
            "kv_heads": kv_heads, "seq_q": seq_q, "seq_kv": seq_kv,
            "cache": seq_kv + rng.choice((0, 1000)), "d": d, "dv": dv,
            "causal": not token and not mask and rng.random() < 0.7,
            "mask": mask, "out_f32": rng.random() < 0.2}


# ------------------------------------------------------------------ inputs --

class _Values:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, *shape, std=1.0):
        t = torch.randn(shape, generator=self.g, device="cuda",
                        dtype=torch.float32)
        return t.mul_(std).to(torch.float16)

    def uniform(self, *shape, low, high):
        t = torch.rand(shape, generator=self.g, device="cuda",
                       dtype=torch.float32)
        return t.mul_(high - low).add_(low).to(torch.float16)

    def int8(self, *shape):
        return torch.randint(-128, 128, shape, generator=self.g,
                             device="cuda", dtype=torch.int8)


def _inputs(case, seed):
    v, op = _Values(seed), case["op"]
    if op == "matmul":
        m, n, k = case["m"], case["n"], case["k"]
        a_shape = (k, m) if case["a_transposed"] else (m, k)
        b_shape = (n, k) if case["b_transposed"] else (k, n)
        if case["dtype"] == "i8":
            return {"a": v.int8(*a_shape), "b": v.int8(*b_shape)}
        return {"a": v.uniform(*a_shape, low=-1.0, high=1.0),
                "b": v.normal(*b_shape, std=0.02)}
    if op == "linear":
        z, m, n, k = case["batch"], case["m"], case["n"], case["k"]
        lead = (z,) if z > 1 else ()
        b_shape = (n, k) if case["b_transposed"] else (k, n)
        return {"x": v.normal(*lead, m, k),
                "w": v.normal(*lead, *b_shape, std=1.0 / math.sqrt(k)),
                "bias": v.normal(n, std=0.5) if case["bias"] else None,
                "mul": (v.normal(*lead, m, n) if case["multiplier"]
                        else None)}
    if op == "ffn":
        m, h, i = case["m"], case["hidden"], case["inner"]
        return {"x": v.normal(m, h), "gate": v.normal(h, i, std=0.02),
                "up": v.normal(h, i, std=0.02),
                "down": v.normal(i, h, std=0.02)}
    if op == "w8a16":
        m, n, k = case["m"], case["n"], case["k"]
        return {"x": v.normal(m, k),
                "w": v.int8(*((n, k) if case["w_transposed"] else (k, n))),
                "scale": v.uniform(n, low=0.001, high=0.02)}
    b, d, dv = case["batch"], case["d"], case["dv"]
    sq, skv, cache = case["seq_q"], case["seq_kv"], case["cache"]
    mask = None
    if case["mask"]:
        # a bias by distance with a tenth of the keys hidden from each query
        mask = v.normal(sq, skv)
        mask.masked_fill_(torch.rand(sq, skv, generator=v.g, device="cuda")
                          < 0.1, -math.inf)
    return {"q": v.normal(b, case["heads"], sq, d),
            "k": v.normal(b, case["kv_heads"], cache, d)[:, :, :skv],
            "v": v.normal(b, case["kv_heads"], cache, dv)[:, :, :skv],
            "mask": mask}


def _record_ffn(case):
    """gate = silu(x . Wg); hidden = gate * (x . Wu); y = hidden . Wd, over
    the binding table x, Wg, Wu, Wd, gate, hidden, y."""
    m, h, i = case["m"], case["hidden"], case["inner"]
    slot = _pkg.slot

    def consts(n, k, **epilogue):
        return _pkg.batch_matmul_constants(m, n, k, k, n, n, 0, 1, m * k,
                                           k * n, m * n, **epilogue)

    cb = _pkg.CommandBuffer()
    cb.dispatch("batch_matmul_f16", consts(i, h, activation=_pkg.ACT_SILU),
                [slot(0), slot(1), slot(4)])
    cb.barrier()
    cb.dispatch("batch_matmul_f16",
                consts(i, h, has_multiplier=True, ld_multiplier=i,
                       batch_stride_multiplier=m * i),
                [slot(0), slot(2), slot(5), slot(4)])
    cb.barrier()
    cb.dispatch("batch_matmul_f16", consts(h, i),
                [slot(5), slot(3), slot(6)])
    return cb.end()


def prepare(case, seed):
    state = {"case": case, "in": _inputs(case, seed)}
    if case["op"] == "ffn":
        t, m = state["in"], case["m"]

        def out(n):
            return torch.empty(m, n, dtype=torch.float16, device="cuda")

        state["cb"] = _record_ffn(case)
        state["out"] = {"gate": out(case["inner"]),
                        "hidden": out(case["inner"]), "y": out(case["hidden"])}
        o = state["out"]
        state["table"] = [t["x"], t["gate"], t["up"], t["down"], o["gate"],
                          o["hidden"], o["y"]]
    return state


def run(state):
    case, t = state["case"], state["in"]
    op = case["op"]
    if op == "matmul":
        return _pkg.matmul(t["a"], t["b"],
                           b_transposed=case["b_transposed"],
                           a_transposed=case["a_transposed"],
                           out_dtype=(torch.float32 if case["out_f32"]
                                      else None))
    if op == "linear":
        if case["batch"] == 1:
            return _pkg.linear(t["x"], t["w"], t["bias"],
                               activation=case["activation"],
                               multiplier=t["mul"],
                               w_transposed=case["b_transposed"])
        return _pkg.batch_matmul(t["x"], t["w"], bias=t["bias"],
                                 activation=case["activation"],
                                 multiplier=t["mul"],
                                 b_transposed=case["b_transposed"])
    if op == "ffn":
        state["cb"].submit(state["table"])
        return state["out"]
    if op == "w8a16":
        return _pkg.quantized_matmul(t["x"], t["w"], t["scale"],
                                     w_transposed=case["w_transposed"])
    return _pkg.attention(t["q"], t["k"], t["v"], causal=case["causal"],
                          mask=t["mask"],
                          out_dtype=(torch.float32 if case["out_f32"]
                                     else None))


def work(case):
    op = case["op"]
    if op in ("matmul", "linear", "w8a16"):
        z = case.get("batch", 1)
        m, n, k = case["m"], case["n"], case["k"]
        i8 = case.get("dtype") == "i8"
        a, b, c = (1, 1, 4) if i8 else (2, 2, 2)
        if op == "w8a16":
            b = 1
        if case.get("out_f32"):
            c = 4
        nbytes = z * (a * m * k + b * n * k + c * m * n)
        if case.get("multiplier"):
            nbytes += z * 2 * m * n
        if case.get("bias") or op == "w8a16":
            nbytes += 2 * n
        return {"bytes": nbytes, "flops": 2 * z * m * n * k}
    if op == "ffn":
        m, h, i = case["m"], case["hidden"], case["inner"]
        return {"bytes": 2 * (3 * h * i + 2 * m * h + 2 * m * i),
                "flops": 6 * m * h * i}
    b, h, hk = case["batch"], case["heads"], case["kv_heads"]
    sq, skv, d, dv = case["seq_q"], case["seq_kv"], case["d"], case["dv"]
    pairs = sq * skv
    if case["causal"]:  # query i sees keys 0..i
        seen = min(sq, skv)
        pairs = seen * (seen + 1) // 2 + (sq - seen) * skv
    nbytes = 2 * b * (h * sq * d + hk * skv * (d + dv))
    nbytes += (4 if case["out_f32"] else 2) * b * h * sq * dv
    if case["mask"]:
        nbytes += 2 * sq * skv
    return {"bytes": nbytes, "flops": 2 * b * h * pairs * (d + dv)}


def tolerance(case):
    """About four times what results in another order of summation differ by."""
    if case.get("dtype") == "i8":
        return "exact"
    if case["op"] == "attention":
        # probabilities rounded to f16 against another running maximum, and
        # the result's rounding: 2.9e-4 from 64 bits over 3001 keys
        return {"rel": 1.2e-3, "max": 1.2e-2}
    if case.get("out_f32"):
        # f32 sums: 4e-7 from 64 bits at 4099 terms, more at 11008
        return {"rel": 5e-6, "max": 1e-4}
    # results rounded once to f16, 2.1e-4 from 64 bits; the feed-forward
    # block rounds three times, 3.6e-4
    return {"rel": 1e-3, "max": 4e-3}


# --------------------------------------------------------------- reference --

_ACTIVATIONS = {
    "none": lambda v: v, "relu": torch.relu, "silu": torch.nn.functional.silu,
    "gelu_tanh": lambda v: torch.nn.functional.gelu(v, approximate="tanh"),
}


def exact(case, seed):
    t = {n: v if v is None else v.double()
         for n, v in _inputs(case, seed).items()}
    op = case["op"]
    if op == "matmul":
        a = t["a"].t() if case["a_transposed"] else t["a"]
        b = t["b"].t() if case["b_transposed"] else t["b"]
        c = torch.mm(a, b)
        return c.to(torch.int32) if case["dtype"] == "i8" else c
    if op == "linear":
        w = t["w"].transpose(-1, -2) if case["b_transposed"] else t["w"]
        y = torch.matmul(t["x"], w.contiguous())
        if t["bias"] is not None:
            y = y + t["bias"]
        y = _ACTIVATIONS[case["activation"]](y)
        return y if t["mul"] is None else y * t["mul"]
    if op == "ffn":
        gate = torch.nn.functional.silu(t["x"] @ t["gate"])
        hidden = gate * (t["x"] @ t["up"])
        return {"gate": gate, "hidden": hidden, "y": hidden @ t["down"]}
    if op == "w8a16":
        w = t["w"].t() if case["w_transposed"] else t["w"]
        return torch.mm(t["x"], w) * t["scale"]
    b, h, hk = case["batch"], case["heads"], case["kv_heads"]
    sq, skv = case["seq_q"], case["seq_kv"]
    hidden_keys = torch.zeros(sq, skv, dtype=torch.float64, device="cuda")
    if case["causal"]:
        later = torch.ones(sq, skv, dtype=torch.bool, device="cuda").triu(1)
        hidden_keys.masked_fill_(later, -math.inf)
    if t["mask"] is not None:
        hidden_keys = hidden_keys + t["mask"]
    out = torch.empty(b, h, sq, case["dv"], dtype=torch.float64,
                      device="cuda")
    for z in range(b):
        for head in range(h):
            kv = head // (h // hk)
            s = torch.mm(t["q"][z, head], t["k"][z, kv].t())
            s = s * case["d"] ** -0.5 + hidden_keys
            # a query that sees no key gets zeros
            p = torch.softmax(s, -1).nan_to_num_(0.0)
            out[z, head] = torch.mm(p, t["v"][z, kv])
    return out
