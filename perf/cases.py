"""Timed cases of the framework: one pass each through its public entry points.

The cases are the calls a speculative-decoding server makes with this
framework, over the range it makes them: a decoder layer's quantized linears
while a block is verified (M = 4 .. 64 rows), while a prompt is prefilled
(tens to thousands of rows, ragged) and for a single decoded token; the fused
lm_head + greedy + accept; the routed experts of a MoE layer for a verify
block and for a prompt; and the rollback pair of a gated-delta layer.  Layer
widths are those of bench.py's 27B-, 9B-class and top-8-of-256 workloads.
"""

from __future__ import annotations

import math

import torch

import __graft_entry__

__graft_entry__.load_package()

from dflash_mlx_amd import gdn, lm_head, moe  # noqa: E402
from dflash_mlx_amd.verify_linear import (  # noqa: E402
    QuantizedLinear, install_verify_linears, prewarm_verify_kernels)
from dflash_mlx_amd.verify_qmm import quantized_matmul  # noqa: E402

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}
_DEV = "cuda:0"


# ---------------------------------------------------------------- the cases

def listed():
    return [
        # one decoded token through the smallest projection of a 9B-class
        # layer (k or v): latency and the launch are all of it
        {"name": "decode_kv_9b", "kind": "linear", "m": 1, "k": 4096, "n": 1024, "gs": 64,
         "bits": 4, "dtype": "bf16"},
        # the flagship: one 27B-class layer's seven verify linears on a
        # 16-token block (q/k/v and gate/up as siblings)
        {"name": "verify_layer_27b", "kind": "layer", "m": 16, "hidden": 5120, "kv": 1024,
         "inter": 17408, "gs": 64, "bits": 4, "dtype": "bf16"},
        # the same block through an 8-bit 9B-class layer
        {"name": "verify_layer_9b_8bit", "kind": "layer", "m": 16, "hidden": 4096, "kv": 1024,
         "inter": 12288, "gs": 64, "bits": 8, "dtype": "bf16"},
        # two requests' blocks (or a draft tree) verified together, f16, gs 128
        {"name": "verify_wide_9b_f16", "kind": "layer", "m": 32, "hidden": 4096, "kv": 1024,
         "inter": 12288, "gs": 128, "bits": 4, "dtype": "f16"},
        # a short prompt (or the ragged tail of a long one)
        {"name": "prompt_77_27b", "kind": "layer", "m": 77, "hidden": 5120, "kv": 1024,
         "inter": 17408, "gs": 64, "bits": 4, "dtype": "bf16"},
        # a prefill chunk of 512
        {"name": "prefill_512_27b", "kind": "layer", "m": 512, "hidden": 5120, "kv": 1024,
         "inter": 17408, "gs": 64, "bits": 4, "dtype": "bf16"},
        # a long prompt in one chunk, not a round number of rows: the largest
        {"name": "prefill_2000_9b", "kind": "layer", "m": 2000, "hidden": 4096, "kv": 1024,
         "inter": 12288, "gs": 64, "bits": 4, "dtype": "bf16"},
        # prefill of an 8-bit down projection, f16
        {"name": "prefill_down_8bit", "kind": "linear", "m": 333, "k": 12288, "n": 4096,
         "gs": 64, "bits": 8, "dtype": "f16"},
        # the end of every verify cycle, with the logits (sampling wants them)
        {"name": "lm_head_accept", "kind": "lm_head", "m": 16, "k": 5120, "v": 151936,
         "gs": 64, "dtype": "bf16"},
        # routed experts of one MoE layer: a verify block ...
        {"name": "moe_verify", "kind": "moe", "t": 16, "topk": 8, "experts": 256, "d": 2048,
         "inter": 512, "gs": 64, "dtype": "bf16"},
        # ... and a prompt
        {"name": "moe_prefill", "kind": "moe", "t": 500, "topk": 8, "experts": 256, "d": 2048,
         "inter": 512, "gs": 64, "dtype": "bf16"},
        # a gated-delta layer's verify step and its rollback to 9 of 16 tokens
        {"name": "gdn_rollback", "kind": "gdn", "b": 1, "t": 16, "keep": 9, "hk": 16, "hv": 32,
         "d": 128},
    ]


def _log_int(rng, lo, hi, multiple=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, int(round(v / multiple)) * multiple)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "layer", "layer", "layer", "lm_head", "moe",
                       "moe", "gdn"])
    if kind == "gdn":
        t = rng.randint(2, 32)
        hk = rng.choice([4, 8, 16])
        return {"kind": kind, "b": rng.choice([1, 1, 2]), "t": t, "keep": rng.randint(1, t),
                "hk": hk, "hv": hk * rng.choice([1, 2, 4]), "d": 128}
    gs = rng.choice([64, 64, 64, 128, 32])
    dtype = rng.choice(["bf16", "bf16", "f16"])
    if kind == "lm_head":
        return {"kind": kind, "m": rng.randint(1, 32), "k": _log_int(rng, 1024, 5120, 256),
                "v": _log_int(rng, 8000, 151936, 8), "gs": gs, "dtype": dtype}
    if kind == "moe":
        return {"kind": kind, "t": _log_int(rng, 1, 500), "topk": rng.choice([2, 4, 8]),
                "experts": rng.choice([32, 64, 128, 256]), "d": _log_int(rng, 1024, 2048, 256),
                "inter": _log_int(rng, 256, 768, 128), "gs": rng.choice([64, 64, 128]),
                "dtype": dtype}
    bits = rng.choice([4, 4, 4, 8])
    if kind == "linear":  # K whole groups, N ragged at times
        return {"kind": kind, "m": _log_int(rng, 1, 2000), "k": _log_int(rng, 512, 12288, gs),
                "n": _log_int(rng, 256, 16384, rng.choice([4, 32, 64, 128])), "gs": gs,
                "bits": bits, "dtype": dtype}
    hidden = _log_int(rng, 1024, 5120, 256)
    return {"kind": kind, "m": _log_int(rng, 1, 800), "hidden": hidden,
            "kv": rng.choice([256, 512, 1024]),
            "inter": _log_int(rng, 2 * hidden, 3.4 * hidden, 256), "gs": gs, "bits": bits,
            "dtype": dtype}


# ---------------------------------------------------------------- inputs

class _Source:
    """Seeded random tensors on the GPU."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=_DEV)
        self.gen.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, generator=self.gen, device=_DEV)

    def uniform(self, *shape):
        return torch.rand(shape, generator=self.gen, device=_DEV)

    def integers(self, high, *shape):
        return torch.randint(0, high, shape, generator=self.gen, device=_DEV, dtype=torch.int32)

    def quantized(self, n, k, gs, bits, dtype):
        """Packed words, scales and biases [n, ...] of N(0, 0.02) weights: per
        group the end of the range with the larger magnitude is the bias and
        the scale points to the other one, as MLX checkpoints hold them."""
        per, top = 32 // bits, float(2 ** bits - 1)
        words = torch.empty((n, k // per), dtype=torch.int32, device=_DEV)
        scales = torch.empty((n, k // gs), dtype=_DTYPES[dtype], device=_DEV)
        biases = torch.empty_like(scales)
        shifts = torch.arange(per, device=_DEV, dtype=torch.int32) * bits
        rows = max(1, (1 << 27) // k)  # row blocks: bounded temporaries
        for r0 in range(0, n, rows):
            r1 = min(n, r0 + rows)
            w = (self.normal(r1 - r0, k) * 0.02).reshape(r1 - r0, k // gs, gs)
            hi, lo = w.amax(-1), w.amin(-1)
            down = hi.abs() >= lo.abs()
            s = torch.where(down, lo - hi, hi - lo) / top
            b = torch.where(down, hi, lo)
            q = ((w - b[..., None]) / s[..., None]).round_().clamp_(0, top).to(torch.int32)
            words[r0:r1] = (q.reshape(r1 - r0, k // per, per) << shifts).sum(-1, dtype=torch.int32)
            scales[r0:r1], biases[r0:r1] = s.to(scales.dtype), b.to(scales.dtype)
        return words, scales, biases


_LAYER = (("self_attn", "q_proj"), ("self_attn", "k_proj"), ("self_attn", "v_proj"),
          ("self_attn", "o_proj"), ("mlp", "gate_proj"), ("mlp", "up_proj"), ("mlp", "down_proj"))


def _layer_shapes(c):
    h, kv, i = c["hidden"], c["kv"], c["inter"]
    return ((h, h), (kv, h), (kv, h), (h, h), (i, h), (i, h), (h, i))


def _inputs(case, seed):
    """The plain tensors of a case, from the seed alone."""
    src = _Source(seed)
    kind = case["kind"]
    if kind == "gdn":
        b, t, hk, hv, d = (case[n] for n in ("b", "t", "hk", "hv", "d"))
        unit = torch.nn.functional.normalize
        return {"q": (unit(src.normal(b, t, hk, d), dim=-1) / d ** 0.5).to(torch.bfloat16),
                "k": unit(src.normal(b, t, hk, d), dim=-1).to(torch.bfloat16),
                "v": src.normal(b, t, hv, d).to(torch.bfloat16),
                "g": src.uniform(b, t, hv) * 0.15 + 0.85,
                "beta": src.uniform(b, t, hv).to(torch.bfloat16),
                "state": src.normal(b, hv, d, d) * 0.1}
    dtype, gs, bits = case["dtype"], case["gs"], case.get("bits", 4)
    dt = _DTYPES[dtype]
    if kind == "linear":
        return {"x": src.normal(case["m"], case["k"]).to(dt),
                "w": src.quantized(case["n"], case["k"], gs, bits, dtype)}
    if kind == "layer":
        m, h = case["m"], case["hidden"]
        # normed hidden states; the down projection reads the product of two
        return {"x": [src.normal(m, h).to(dt), src.normal(m, h).to(dt), src.normal(m, h).to(dt),
                      (src.normal(m, case["inter"]) * src.normal(m, case["inter"])).to(dt)],
                "w": [src.quantized(n, k, gs, bits, dtype) for n, k in _layer_shapes(case)]}
    if kind == "lm_head":
        return {"h": src.normal(case["m"], case["k"]).to(dt),
                "ids": src.integers(case["v"], case["m"]),
                "w": src.quantized(case["v"], case["k"], gs, 4, dtype)}
    e, d, i = case["experts"], case["d"], case["inter"]
    x = src.normal(case["t"], d).to(dt)
    probs, inds = torch.softmax(src.normal(case["t"], e), -1).topk(case["topk"], -1)
    sets = []
    for n, k in ((i, d), (i, d), (d, i)):
        sets.append(tuple(a.reshape(e, n, -1) for a in src.quantized(e * n, k, gs, 4, dtype)))
    return {"x": x, "inds": inds, "scores": probs / probs.sum(-1, keepdim=True), "w": sets}


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = case
    if case["kind"] == "layer":
        root = torch.nn.Module()
        root.self_attn, root.mlp = torch.nn.Module(), torch.nn.Module()
        for (parent, name), w in zip(_LAYER, s.pop("w")):
            setattr(getattr(root, parent), name,
                    QuantizedLinear(*w, group_size=case["gs"], bits=case["bits"]))
        install_verify_linears(root, enable_qmm=True)
        prewarm_verify_kernels(root, input_dtype=_DTYPES[case["dtype"]])
        s["layer"] = root
    return s


# ---------------------------------------------------------------- one pass

def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear":
        return quantized_matmul(state["x"], *state["w"], group_size=c["gs"], bits=c["bits"])
    if kind == "layer":
        attn, mlp = state["layer"].self_attn, state["layer"].mlp
        xa, xo, xm, xd = state["x"]
        return [attn.q_proj(xa), attn.k_proj(xa), attn.v_proj(xa), attn.o_proj(xo),
                mlp.gate_proj(xm), mlp.up_proj(xm), mlp.down_proj(xd)]
    if kind == "lm_head":
        r = lm_head.lm_head_greedy_accept(state["h"], *state["w"], verify_ids=state["ids"],
                                          group_size=c["gs"], return_logits=True)
        return {"logits": r.logits, "posterior": r.posterior, "accept_len": r.accept_len,
                "bonus": r.bonus}
    if kind == "moe":
        h, y = moe.switch_glu(state["x"], state["inds"], *state["w"], group_size=c["gs"])
        return {"h": h, "y": y, "out": moe.moe_combine(y, state["scores"])}
    y, after, tape = gdn.gated_delta_kernel_with_tape(
        *(state[n] for n in ("q", "k", "v", "g", "beta", "state")))
    n = c["keep"]
    back = gdn.tape_replay_kernel(tape[:, :n], state["k"][:, :n], state["g"][:, :n],
                                  state["state"])
    return {"y": y, "state": after, "tape": tape, "rolled_back": back}


# ---------------------------------------------------------------- its work

def _weight_bytes(n, k, gs, bits):
    return n * k * bits // 8 + 4 * n * (k // gs)


def work(case):
    kind = case["kind"]
    if kind == "gdn":
        b, t, keep, hk, hv, d = (case[n] for n in ("b", "t", "keep", "hk", "hv", "d"))
        state = 4 * b * hv * d * d
        step_in = 2 * b * hk * d * 2 + 2 * b * hv * d + 4 * b * hv + 2 * b * hv
        step_out = 2 * b * hv * d + 4 * b * hv * d
        # the state in, the advanced and the rolled-back state out
        return {"bytes": 3 * state + t * (step_in + step_out),
                "flops": (7 * t + 3 * keep) * b * hv * d * d}
    gs, bits = case["gs"], case.get("bits", 4)
    if kind == "moe":
        t, p = case["t"], case["t"] * case["topk"]
        e, d, i = case["experts"], case["d"], case["inter"]
        touched = e * (1 - (1 - case["topk"] / e) ** t)  # experts some token is routed to
        return {"bytes": int(touched * 3 * _weight_bytes(d, i, gs, 4) + 2 * t * d + 12 * p +
                             2 * p * (i + d) + 2 * t * d),
                "flops": 2 * p * 3 * d * i + 2 * p * d}
    if kind == "lm_head":
        m, k, v = case["m"], case["k"], case["v"]
        return {"bytes": _weight_bytes(v, k, gs, 4) + 2 * m * k + 2 * m * v + 8 * m,
                "flops": 2 * m * k * v}
    m = case["m"]
    if kind == "linear":
        shapes, read = ((case["n"], case["k"]),), case["k"]
    else:
        shapes, read = _layer_shapes(case), 3 * case["hidden"] + case["inter"]
    return {"bytes": sum(_weight_bytes(n, k, gs, bits) + 2 * m * n for n, k in shapes) +
            2 * m * read,
            "flops": sum(2 * m * n * k for n, k in shapes)}


def tolerance(case):
    # Outputs are rounded once to 16 bits from 32-bit sums (measured against
    # 64 bits: 1.7e-3 in bf16, 2.1e-4 in f16); the experts' chain rounds the
    # projections, the SwiGLU steps and the pair outputs in turn.  The largest
    # difference is one unit in the last place, more down a chain.
    bf16 = case.get("dtype", "bf16") == "bf16"
    if case["kind"] == "moe":
        return {"rel": 1.2e-2, "max": 6e-2} if bf16 else {"rel": 1.6e-3, "max": 8e-3}
    tol = {"rel": 7e-3, "max": 1.6e-2} if bf16 else {"rel": 9e-4, "max": 2e-3}
    if case["kind"] == "lm_head":
        tol["differ"] = 0.07  # one token of a block, where two logits tie in 16 bits
    return tol


# ---------------------------------------------------------------- in 64 bits

def _dequantized(w, gs, bits):
    words, scales, biases = w
    per = 32 // bits
    shifts = torch.arange(per, device=words.device, dtype=torch.int32) * bits
    q = ((words[..., None] >> shifts) & (2 ** bits - 1)).reshape(*words.shape[:-1], -1)
    return (q.double() * scales.double().repeat_interleave(gs, -1) +
            biases.double().repeat_interleave(gs, -1))


def _product(x, w, gs, bits):
    """x . dequant(w)^T in 64 bits, by blocks of weight rows."""
    n, k = w[0].shape[0], x.shape[-1]
    rows = max(1, (1 << 27) // k)
    return torch.cat([x.double() @ _dequantized([a[r:r + rows] for a in w], gs, bits).T
                      for r in range(0, n, rows)], dim=-1)


def _recurrence(t, s, n_steps, tape=None):
    """(outputs, state, innovations) of n_steps gated-delta steps from the
    state; with a tape, its innovations are replayed instead."""
    rep = t["v"].shape[2] // t["k"].shape[2]
    k = t["k"].double().repeat_interleave(rep, 2)
    q = t["q"].double().repeat_interleave(rep, 2)
    v, g, beta = t["v"].double(), t["g"].double(), t["beta"].double()
    ys, ds = [], []
    for i in range(n_steps):
        s = s * g[:, i, :, None, None]
        if tape is None:
            kv = (s * k[:, i, :, None, :]).sum(-1)
            d = (v[:, i] - kv) * beta[:, i, :, None]
        else:
            d = tape[:, i]
        s = s + d[..., None] * k[:, i, :, None, :]
        ys.append((s * q[:, i, :, None, :]).sum(-1))
        ds.append(d)
    return torch.stack(ys, 1), s, torch.stack(ds, 1)


def exact(case, seed):
    t = _inputs(case, seed)
    kind = case["kind"]
    if kind == "gdn":
        y, after, tape = _recurrence(t, t["state"].double(), case["t"])
        back = _recurrence(t, t["state"].double(), case["keep"], tape)[1]
        return {"y": y, "state": after, "tape": tape, "rolled_back": back}
    gs, bits = case["gs"], case.get("bits", 4)
    if kind == "linear":
        return _product(t["x"], t["w"], gs, bits)
    if kind == "layer":
        return [_product(t["x"][i], w, gs, bits) for i, w in zip((0, 0, 0, 1, 2, 2, 3), t["w"])]
    if kind == "lm_head":
        return {"logits": _product(t["h"], t["w"], gs, bits), "posterior": None,
                "accept_len": None, "bonus": None}
    flat = t["inds"].reshape(-1)
    token = torch.arange(flat.numel(), device=flat.device) // case["topk"]
    x, p = t["x"].double(), flat.numel()
    h = torch.empty((p, case["inter"]), dtype=torch.float64, device=flat.device)
    y = torch.empty((p, case["d"]), dtype=torch.float64, device=flat.device)
    for e in flat.unique().tolist():
        at = (flat == e).nonzero().reshape(-1)
        gate, up, down = (_dequantized([a[e] for a in w], gs, 4) for w in t["w"])
        h[at] = torch.nn.functional.silu(x[token[at]] @ gate.T) * (x[token[at]] @ up.T)
        y[at] = h[at] @ down.T
    out = (y.reshape(case["t"], case["topk"], -1) * t["scores"].double()[..., None]).sum(1)
    return {"h": h, "y": y, "out": out}
