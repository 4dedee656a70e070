"""What this framework is timed on: the calls that a program on it makes.

A case is one of five kinds of work, each through the public entry points of
rkhip:

* products: one token's matrix products of a decoder layer (QKV, Wo, W1 with
  W3, W2), from host buffers (matvecs) or device pointers (matvecs_device);
* block_scaled: one token's products of a DeepSeek-V4.1-shaped layer: E4M3
  attention projections, then the routed experts' E2M1 rows in a Batch;
* forward: token activations through a run of resident layers
  (Stage.forward), one token (decode) or a prompt (prefill);
* generate: a whole generation, prompt and decode steps, of one sequence or
  of several side by side, dense or mixture-of-experts;
* tensor: the rakkan_tensor_v1 matrix products, on host or device buffers.

Every result is held to the bits of the reference's CPU path, so every
case's tolerance is "exact".
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "rakkan-mesh_amd"))
import rkhip  # noqa: E402

_KINDS = {"q8": rkhip.Q8, "q4": rkhip.Q4, "f32": rkhip.F32, "bf16": rkhip.BF16}
_device = None


def _dev():
    """The program's one opened device."""
    global _device
    if _device is None:
        _device = rkhip.Device(0)
    return _device


# ---- the cases ----

_LLAMA_8B = {"dim": 4096, "heads": 32, "kv_heads": 8, "head_dim": 128, "hidden": 14336}
_QWEN_7B = {"dim": 3584, "heads": 28, "kv_heads": 4, "head_dim": 128, "hidden": 18944, "bias": True}
_QWEN_MOE = {"dim": 2048, "heads": 32, "kv_heads": 4, "head_dim": 128, "hidden": 768, "qk_norm": True, "experts": 128,
             "topk": 8}
_LLAMA2C = {"dim": 288, "heads": 6, "kv_heads": 6, "head_dim": 48, "hidden": 768}


def listed():
    return [
        # a host program's smallest products: a llama2.c layer, four round trips
        {"name": "products_host_288", "kind": "products", "format": "q8", "dim": 288, "q_dim": 288, "kv_dim": 288,
         "hidden": 768, "host": True},
        # an 8B-shape layer's Q8 products for one token, activations resident
        {"name": "products_q8_8b", "kind": "products", "format": "q8", "dim": 4096, "q_dim": 4096, "kv_dim": 1024,
         "hidden": 14336, "host": False},
        # a bfloat16 layer (a checkpoint run without quantizing)
        {"name": "products_bf16_2048", "kind": "products", "format": "bf16", "dim": 2048, "q_dim": 2048, "kv_dim": 512,
         "hidden": 8192, "host": False},
        # DeepSeek-V4.1's decode products: wq_b, wo_b, six of the routed experts
        {"name": "block_scaled_layer", "kind": "block_scaled", "q_rows": 32768, "q_cols": 1280, "dim": 5120,
         "o_cols": 8192, "expert_rows": 2304, "experts": 24, "slots": 6},
        # one decode token through a node's layers of an 8B-shape Q8 model
        {"name": "decode_q8_8b", "kind": "forward", "format": "q8", **_LLAMA_8B, "layers": 4, "pos": 640, "tokens": 1,
         "ctx": 1024},
        # the same late in a long conversation, Q4
        {"name": "decode_q4_long", "kind": "forward", "format": "q4", **_QWEN_7B, "layers": 3, "pos": 6000,
         "tokens": 1, "ctx": 8192},
        # a long prompt through a Q4 model's layers
        {"name": "prefill_q4_512", "kind": "forward", "format": "q4", **_QWEN_7B, "layers": 2, "pos": 0, "tokens": 512,
         "ctx": 1024},
        # the smallest whole model: the llama2.c decoder, 8 + 64 tokens, latency alone
        {"name": "generate_288", "kind": "generate", "format": "q8", **_LLAMA2C, "layers": 6, "vocab": 32000,
         "seqs": 1, "prompt": 8, "steps": 64, "ctx": 256, "temperature": 0.0},
        # a mixture-of-experts decoder: one sequence
        {"name": "generate_moe_1", "kind": "generate", "format": "q8", **_QWEN_MOE, "layers": 8, "vocab": 151936,
         "seqs": 1, "prompt": 64, "steps": 32, "ctx": 128, "temperature": 0.0},
        # and sixteen sequences served together
        {"name": "generate_moe_16", "kind": "generate", "format": "q8", **_QWEN_MOE, "layers": 8, "vocab": 151936,
         "seqs": 16, "prompt": 64, "steps": 32, "ctx": 128, "temperature": 0.0},
        # a sandboxed program's float32 product (a batch through an MLP layer)
        {"name": "tensor_f32_1024", "kind": "tensor", "dtype": "f32", "m": 1024, "k": 784, "n": 1024,
         "transposed": True, "host": False},
        # and its quantized one
        {"name": "tensor_i8_2048", "kind": "tensor", "dtype": "i8", "m": 2048, "k": 2048, "n": 2048,
         "transposed": False, "host": False},
    ]


def _log(rng, lo, hi, step=1):
    """A size spread over the logarithm of [lo, hi], a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(step, int(v / step + 0.5) * step)


def draw(rng):
    kind = rng.choice(["products", "block_scaled", "forward", "forward", "generate", "tensor"])
    if kind == "products":
        fmt = rng.choice(["q8", "q4", "bf16", "f32"])
        step = 32 if fmt in ("q8", "q4") else 2
        dim = _log(rng, 64, 4096, step)
        return {"kind": kind, "format": fmt, "dim": dim, "q_dim": _log(rng, max(64, dim / 2), dim * 1.5, step),
                "kv_dim": _log(rng, max(32, dim / 8), dim, step), "hidden": _log(rng, dim, dim * 3.5, step),
                "host": rng.random() < 0.3}
    if kind == "block_scaled":
        return {"kind": kind, "q_rows": _log(rng, 256, 32768), "q_cols": _log(rng, 128, 2048, 32),
                "dim": _log(rng, 256, 5120, 32), "o_cols": _log(rng, 512, 8192, 32),
                "expert_rows": _log(rng, 128, 2304, 32), "experts": rng.randint(6, 24), "slots": rng.randint(1, 6)}
    if kind == "tensor":
        dtype = rng.choice(["f32", "i8"])
        top = 1100 if dtype == "f32" else 2048
        return {"kind": kind, "dtype": dtype, "m": _log(rng, 1, top), "k": _log(rng, 8, top), "n": _log(rng, 8, top),
                "transposed": rng.random() < 0.5, "host": rng.random() < 0.4}
    hd = rng.choice([48, 64, 64, 128, 128, 128])
    kv = rng.choice([1, 2, 4, 8])
    heads = kv * rng.choice([1, 2, 4, 7])
    while heads * hd > 4096:
        heads -= kv
    heads += heads % 2 if heads * hd % 32 else 0
    kv = max(k for k in (1, 2, 4, 8) if heads % k == 0 and k <= kv)
    norm = rng.random() < 0.3
    model = {"dim": _log(rng, 256, 4096, 32), "heads": heads, "kv_heads": kv, "head_dim": hd,
             "hidden": _log(rng, 512, 14336, 32), "qk_norm": norm, "bias": not norm and rng.random() < 0.4}
    fmt = rng.choice(["q8", "q4"])
    if kind == "forward":
        tokens = 1 if rng.random() < 0.5 else _log(rng, 2, 512)
        pos = _log(rng, 1, 6000) if tokens == 1 else rng.choice([0, _log(rng, 1, 512)])
        return {"kind": kind, "format": fmt, **model, "layers": rng.randint(1, 2), "pos": pos, "tokens": tokens,
                "ctx": min(8192, pos + tokens + _log(rng, 1, 512))}
    seqs = rng.choice([1, 1, _log(rng, 2, 16)])
    prompt, steps = _log(rng, 2, 128), _log(rng, 4, 32)
    case = {"kind": kind, "format": fmt, **model, "layers": rng.randint(1, 4), "vocab": _log(rng, 512, 65536),
            "seqs": seqs, "prompt": prompt, "steps": steps, "ctx": prompt + steps + _log(rng, 1, 256),
            "temperature": rng.choice([0.0, 0.0, 0.8])}
    if rng.random() < 0.4:
        case.update(format="q8", experts=rng.choice([16, 60, 128]), topk=rng.choice([2, 4, 8]),
                    hidden=_log(rng, 128, 1024, 32))
    return case


# ---- inputs ----

class _Source:
    """Random weights: codes and scales cut from pools at drawn offsets, so
    that models of gigabytes take a moment to make."""

    def __init__(self, seed, largest):
        self.rng = np.random.Generator(np.random.SFC64(seed))
        self.raw = self.rng.bit_generator.random_raw((largest + (1 << 20)) // 8 + 1).view(np.uint8)
        self.codes = np.maximum(self.raw.view(np.int8), -127)
        self.scales = self.rng.uniform(2e-5, 2e-4, largest // 32 + (1 << 15)).astype(np.float32)

    def _cut(self, pool, n):
        o = int(self.rng.integers(0, pool.size - n + 1))
        return pool[o:o + n]

    def matrix(self, fmt, rows, cols, gain=1.0):
        """(format, rows, cols, codes or values, scales)."""
        n = rows * cols
        if fmt == "q8":
            return fmt, rows, cols, self._cut(self.codes, n), self._cut(self.scales, n // 32) * np.float32(gain)
        if fmt == "q4":  # 4-bit codes: 16 times the scale for the same weights
            return fmt, rows, cols, self._cut(self.raw, n // 2), self._cut(self.scales, n // 32) * np.float32(16 * gain)
        w = self._cut(self.codes, n).astype(np.float32) * np.float32(1e-4)
        if fmt == "bf16":
            return fmt, rows, cols, (w.view(np.uint32) + 0x8000 >> 16).astype(np.uint16), None
        return fmt, rows, cols, w, None

    def mx(self, fmt, rows, cols):
        n = rows * cols
        if fmt == "fp8":
            w = self._cut(self.raw, n) & np.uint8(0xEF)  # exponents below 8: finite, no NaN code
            return fmt, rows, cols, w, self.rng.integers(114, 122, (rows + 31) // 32 * (cols // 32)).astype(np.uint8)
        return fmt, rows, cols, self._cut(self.raw, n // 2), self.rng.integers(114, 122, n // 32).astype(np.uint8)

    def normal(self, *shape, mean=0.0, dev=1.0):
        return self.rng.normal(mean, dev, shape).astype(np.float32)


def _upload(m):
    fmt, rows, cols, w, s = m
    if fmt == "fp8" or fmt == "fp4":
        return _dev().upload_mx(rkhip.FP8 if fmt == "fp8" else rkhip.FP4, rows, cols, w, s)
    return _dev().upload(_KINDS[fmt], rows, cols, w, s)


def _layer(c, src):
    """A decoder layer's matrices and vectors, on the host."""
    dim, q, kv = c["dim"], c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    f, h = c["format"], c["hidden"]
    d = {"wq": src.matrix(f, q, dim), "wk": src.matrix(f, kv, dim), "wv": src.matrix(f, kv, dim),
         "wo": src.matrix(f, dim, q)}
    if c.get("experts"):
        d["router"] = src.matrix(f, c["experts"], dim, 10.0)
        for n, r, k in (("e1", h, dim), ("e2", dim, h), ("e3", h, dim)):
            d[n] = [src.matrix(f, r, k) for _ in range(c["experts"])]
    else:
        d.update(w1=src.matrix(f, h, dim), w2=src.matrix(f, dim, h), w3=src.matrix(f, h, dim))
    d["rms_att"], d["rms_ffn"] = src.normal(dim, mean=1, dev=0.1), src.normal(dim, mean=1, dev=0.1)
    if c.get("bias"):
        d.update(bq=src.normal(q, dev=0.5), bk=src.normal(kv, dev=0.5), bv=src.normal(kv, dev=0.5))
    if c.get("qk_norm"):
        d.update(q_norm=src.normal(c["head_dim"], mean=1, dev=0.1), k_norm=src.normal(c["head_dim"], mean=1, dev=0.1))
    return d


def _model(c, seed):
    """(layers, head or None, source) of a forward or generate case."""
    q = c["heads"] * c["head_dim"]
    src = _Source(seed, max(c["dim"] * max(c["hidden"], q, c.get("vocab", 0)), 1 << 16))
    layers = [_layer(c, src) for _ in range(c["layers"])]
    head = None
    if "vocab" in c:
        head = {"embed": src.matrix("q8", c["vocab"], c["dim"], 100.0), "rms_final": src.normal(c["dim"], mean=1, dev=0.1)}
        head["prompts"] = src.rng.integers(0, c["vocab"], (c["seqs"], c["prompt"])).astype(np.int32)
    return layers, head, src


def _rope(c):
    half = c["head_dim"] // 2
    freq = np.exp(-np.log(1e6) * (2 * np.arange(half, dtype=np.float64)) / c["head_dim"])
    ang = np.arange(c["ctx"], dtype=np.float64)[:, None] * freq[None, :]
    return np.cos(ang).astype(np.float32), np.sin(ang).astype(np.float32)


class _State:
    """What the program holds; what it opened on the device is freed with it."""

    def __init__(self):
        self.opened = []

    def own(self, x):
        self.opened.append(x)
        return x

    def __del__(self):
        torch.cuda.synchronize()
        for x in reversed(self.opened):
            x.free()


def _stage(c, seed, st):
    layers, head, src = _model(c, seed)
    held = []
    for d in layers:
        up = {k: st.own(_upload(v)) if isinstance(v, tuple) else v for k, v in d.items() if not isinstance(v, list)}
        if "router" in d:
            e = {n: [st.own(_upload(m)) for m in d[n]] for n in ("e1", "e2", "e3")}
            up["moe"] = st.own(rkhip.Moe(_dev(), up.pop("router"), e["e1"], e["e2"], e["e3"], c["topk"]))
        held.append(up)
    cos, sin = _rope(c)
    s = st.own(rkhip.Stage(_dev(), c["dim"], c["hidden"], c["heads"], c["kv_heads"], c["ctx"], held, cos.ravel(),
                           sin.ravel(), head_dim=c["head_dim"], norm_eps=1e-6, qkv_bias=bool(c.get("bias")),
                           qk_norm=bool(c.get("qk_norm")), seqs=c.get("seqs", 1)))
    if head:
        m = st.own(_upload(head["embed"]))
        s.set_head(m, m, head["rms_final"])
        for z in range(c["seqs"]):
            s.sampler(c["temperature"], seed + z + 1, z)
    return s, head, src


def _products_of(c):
    """The layer's four calls: (input width, [rows])."""
    return [(c["dim"], [c["q_dim"], c["kv_dim"], c["kv_dim"]]), (c["q_dim"], [c["dim"]]),
            (c["dim"], [c["hidden"], c["hidden"]]), (c["hidden"], [c["dim"]])]


def _products_inputs(c, seed):
    src = _Source(seed, 2 * c["dim"] * max(c["hidden"], c["q_dim"]))
    return [(src.normal(cols), [src.matrix(c["format"], r, cols, 20.0) for r in rows]) for cols, rows in _products_of(c)]


def _block_scaled_inputs(c, seed):
    d, h, e = c["dim"], c["expert_rows"], c["experts"]
    src = _Source(seed, max(c["q_rows"] * c["q_cols"], d * c["o_cols"], e * h * d // 2))
    return {"wq": src.mx("fp8", c["q_rows"], c["q_cols"]), "wo": src.mx("fp8", d, c["o_cols"]),
            "w1": src.mx("fp4", e * h, d), "w3": src.mx("fp4", e * h, d), "w2": src.mx("fp4", e * d, h),
            "xq": src.normal(c["q_cols"]), "xo": src.normal(c["o_cols"]), "x": src.normal(d),
            "ids": src.rng.permutation(e)[:c["slots"]].astype(np.uint32)}


def _tensor_inputs(c, seed):
    rng = np.random.Generator(np.random.SFC64(seed))
    a, b = (c["m"], c["k"]), (c["n"], c["k"]) if c["transposed"] else (c["k"], c["n"])
    if c["dtype"] == "f32":
        return rng.normal(0, 1, a).astype(np.float32), rng.normal(0, 1, b).astype(np.float32)
    return rng.integers(-127, 128, a, dtype=np.int8), rng.integers(-127, 128, b, dtype=np.int8)


def prepare(case, seed):
    st = _State()
    st.case = c = case
    dev = _dev()
    if c["kind"] == "products":
        st.calls = []
        for x, ms in _products_inputs(c, seed):
            held = [st.own(_upload(m)) for m in ms]
            if c["host"]:
                st.calls.append((held, x))
            else:
                xd = torch.from_numpy(x).cuda()
                outs = [torch.empty(m.rows, dtype=torch.float32, device="cuda") for m in held]
                st.calls.append((held, xd, outs, [o.data_ptr() for o in outs]))
    elif c["kind"] == "block_scaled":
        v = _block_scaled_inputs(c, seed)
        d, h, n = c["dim"], c["expert_rows"], c["slots"]
        for k in ("wq", "wo", "w1", "w3", "w2"):
            setattr(st, k, st.own(_upload(v[k])))
        st.xq, st.xo = torch.from_numpy(v["xq"]).cuda(), torch.from_numpy(v["xo"]).cuda()
        st.q = torch.empty(c["q_rows"], dtype=torch.float32, device="cuda")
        st.o = torch.empty(d, dtype=torch.float32, device="cuda")
        st.x, st.ids = v["x"], v["ids"].view(np.float32)
        # the arena: input, expert ids, gate, up, outputs, the quantize scratch
        sizes = [d, 64, n * h, n * h, n * d, max(d, n * h), max(d, n * h) // 32 + 4]
        at = np.concatenate(([0], np.cumsum([(s + 63) // 64 * 64 for s in sizes]))).tolist()
        st.at = at
        st.arena = st.own(dev.arena(at[-1], d + 64 + n * d))
        st.arena.set_quant_scratch(at[5], at[6])
    elif c["kind"] == "forward":
        st.stage, _, src = _stage(c, seed, st)
        if c["pos"]:
            st.stage.forward(src.normal(c["pos"], c["dim"]), 0)
        st.x = src.normal(c["tokens"], c["dim"])
    elif c["kind"] == "generate":
        st.stage, head, _ = _stage(c, seed, st)
        st.prompts = head["prompts"]
    else:
        a, b = _tensor_inputs(c, seed)
        if c["host"]:
            st.a, st.b = a, b
        else:
            st.a, st.b = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
            st.c = torch.empty(c["m"], c["n"], dtype=torch.float32 if c["dtype"] == "f32" else torch.int32,
                               device="cuda")
    return st


def run(st):
    c, dev = st.case, _dev()
    if c["kind"] == "products":
        if c["host"]:
            return [dev.matvecs(ms, x) for ms, x in st.calls]
        for ms, x, outs, ptrs in st.calls:
            dev.matvecs_device(ms, ptrs, x.data_ptr(), x.numel())
        return [outs for _, _, outs, _ in st.calls]
    if c["kind"] == "block_scaled":
        d, h, n, at = c["dim"], c["expert_rows"], c["slots"], st.at
        dev.matvecs_device([st.wq], [st.q.data_ptr()], st.xq.data_ptr(), st.xq.numel())
        dev.matvecs_device([st.wo], [st.o.data_ptr()], st.xo.data_ptr(), st.xo.numel())
        b = st.arena.begin()
        b.write(at[0], st.x)
        b.write(at[1], st.ids)
        b.expert_matvecs(st.w1, h, at[1], n, at[0], 0, 0, at[2], h)
        b.expert_matvecs(st.w3, h, at[1], n, at[0], 0, 0, at[3], h)
        b.silumul(at[2], at[3], n * h)
        b.expert_matvecs(st.w2, d, at[1], n, at[2], h, 1, at[4], d)
        y = b.read(at[4], n * d)
        b.submit()
        return [st.q, st.o, y]
    if c["kind"] == "forward":
        return st.stage.forward(st.x, c["pos"])
    if c["kind"] == "generate":
        s, steps = st.stage, c["steps"]
        if c["temperature"]:
            for z in range(c["seqs"]):
                s.sampler(c["temperature"], 1234 + z, z)
        if c["seqs"] == 1:
            s.generate_start(st.prompts[0])
            s.generate_run(c["prompt"] + steps - 2)
            logits = s.generate_run(1, want_logits=True)[0]
            return {"logits": logits, "tokens": s.tokens(c["prompt"], steps)}
        s.seqs_start(st.prompts)
        s.seqs_run(steps - 1)
        logits = s.seqs_run(1, want_logits=True)[0]
        return {"logits": logits, "tokens": np.stack([s.seqs_tokens(z, c["prompt"], steps) for z in range(c["seqs"])])}
    if c["host"]:
        return dev.tensor_matmul(st.a, st.b, c["transposed"])
    dt = rkhip.TENSOR_F32 if c["dtype"] == "f32" else rkhip.TENSOR_I8
    dev._check(rkhip.lib().rk_tensor_matmul_device(dev.h, dt, int(c["transposed"]), c["m"], c["k"], c["n"],
                                                   st.a.data_ptr(), st.b.data_ptr(), st.c.data_ptr(), None))
    return st.c


# ---- what a pass cannot do without ----

def _bytes(fmt, rows, cols):
    return {"q8": rows * cols * 1.125, "q4": rows * cols * 0.625, "bf16": rows * cols * 2.0, "f32": rows * cols * 4.0,
            "fp8": rows * cols + rows * cols / 1024, "fp4": rows * cols * (0.5 + 1 / 32)}[fmt]


def _chosen(experts, topk, tokens):
    """Distinct experts that a step of `tokens` tokens is expected to take."""
    return experts * (1 - (1 - topk / experts) ** tokens)


def _step(c, tokens, positions):
    """(bytes, multiply-adds) of `tokens` tokens through the layers together,
    attending to `positions` cached positions in all."""
    q, kv = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    f, dim, h = c["format"], c["dim"], c["hidden"]
    att = dim * (2 * q + 2 * kv)
    b = _bytes(f, 1, att) + 8.0 * kv * positions
    macs = tokens * att + 2.0 * q * positions
    if c.get("experts"):
        b += _bytes(f, c["experts"], dim) + 3 * _bytes(f, h, dim) * _chosen(c["experts"], c["topk"], tokens)
        macs += tokens * (c["experts"] + 3.0 * h * c["topk"]) * dim
    else:
        b += 3 * _bytes(f, h, dim)
        macs += tokens * 3.0 * h * dim
    return c["layers"] * b, c["layers"] * macs


def work(case):
    c = case
    if c["kind"] == "products":
        b = sum(_bytes(c["format"], r, k) + 4 * r for k, rows in _products_of(c) for r in rows)
        b += sum(4 * k for k, _ in _products_of(c))
        return {"bytes": b, "flops": sum(2.0 * r * k for k, rows in _products_of(c) for r in rows)}
    if c["kind"] == "block_scaled":
        d, h, n = c["dim"], c["expert_rows"], c["slots"]
        sizes = [("fp8", c["q_rows"], c["q_cols"]), ("fp8", d, c["o_cols"])] + [("fp4", n * h, d)] * 3
        return {"bytes": sum(_bytes(*s) for s in sizes) + 4.0 * (c["q_rows"] + c["q_cols"] + 2 * d + c["o_cols"] + n * d),
                "flops": sum(2.0 * r * k for _, r, k in sizes)}
    if c["kind"] == "tensor":
        m, k, n, e = c["m"], c["k"], c["n"], 4 if c["dtype"] == "f32" else 1
        return {"bytes": e * (m * k + k * n) + 4.0 * m * n, "flops": 2.0 * m * k * n}
    if c["kind"] == "forward":
        t, p = c["tokens"], c["pos"]
        # a prompt's cached positions are read once for the tokens together
        b, macs = _step(c, t, p + t)
        if t > 1:
            macs += c["layers"] * 2.0 * c["heads"] * c["head_dim"] * (t * p + t * (t + 1) / 2 - (p + t))
        return {"bytes": b + 8.0 * t * c["dim"], "flops": 2.0 * macs}
    s, n, steps = c["seqs"], c["prompt"], c["steps"]
    b = macs = 0.0
    if n > 1:  # the sequences' prompts together
        pb, pm = _step(c, s * (n - 1), s * (n - 1))
        b, macs = b + pb, macs + pm
    for i in range(steps):
        sb, sm = _step(c, s, s * (n + i))
        b += sb + _bytes("q8", c["vocab"], c["dim"]) + 4.0 * s * c["vocab"]
        macs += sm + 1.0 * s * c["vocab"] * c["dim"]
    return {"bytes": b, "flops": 2.0 * macs}


def tolerance(case):
    return "exact"


# ---- 64-bit results ----

def _f64(m):
    """A matrix's values in 64 bits, on the GPU."""
    fmt, rows, cols, w, s = m
    t = torch.from_numpy(np.ascontiguousarray(w)).cuda()
    if fmt == "f32":
        return t.double().view(rows, cols)
    if fmt == "bf16":
        return (t.to(torch.int32) << 16).view(torch.float32).double().view(rows, cols)
    sc = torch.from_numpy(np.ascontiguousarray(s)).cuda().view(-1, 1)
    if fmt == "q8":
        return (t.view(-1, 32).double() * sc.double()).view(rows, cols)
    if fmt == "q4":  # byte j of a block: codes j (low) and j + 16 (high), 8 above the weight
        t = t.view(-1, 16)
        return ((torch.cat([t & 15, t >> 4], 1).double() - 8) * sc.double()).view(rows, cols)
    p = torch.exp2(sc.double() - 127)
    if fmt == "fp8":
        v = t.view(torch.float8_e4m3fn).double().view(rows, cols // 32, 32)
        return (v * p.view(-1, cols // 32).repeat_interleave(32, 0)[:rows, :, None]).view(rows, cols)
    grid = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, 0, -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device="cuda")
    t = t.view(-1, 16)
    return (grid[torch.stack([t & 15, t >> 4], 2).view(-1, 32).long()] * p).view(rows, cols)


def _q8(x):
    """Rows of x as their Q8_0 codes times the scale, a block of 32 each."""
    b = x.reshape(-1, 32)
    d = b.abs().amax(1, keepdim=True) / 127
    return torch.where(d > 0, torch.round(b / torch.where(d > 0, d, 1.0)) * d, 0.0).view(x.shape)


def _e4m3(x):
    """Rows of x as E4M3 codes times a power-of-two scale, a block of 32 each."""
    b = x.reshape(-1, 32)
    s = torch.exp2(torch.ceil(torch.log2(b.abs().amax(1, keepdim=True).clamp_min(1e-4) / 448)))
    return ((b / s).float().to(torch.float8_e4m3fn).double() * s).view(x.shape)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * torch.from_numpy(w).cuda().double()


def _rotate(x, cos, sin):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cos - b * sin, a * sin + b * cos], -1).reshape(x.shape)


def _forward64(c, layers, x, pos, caches):
    """Rows x of one sequence at positions pos.. through the layers, in 64
    bits; caches: a list of [keys, values] a layer, extended."""
    hd, nh, nk, n = c["head_dim"], c["heads"], c["kv_heads"], x.shape[0]
    cos, sin = (torch.from_numpy(t[pos:pos + n]).cuda().double()[:, None] for t in _rope(c))
    seen = torch.arange(pos + n, device="cuda")[None, :] <= torch.arange(pos, pos + n, device="cuda")[:, None]
    for li, d in enumerate(layers):
        a = _q8(_norm(x, d["rms_att"]))
        q, k, v = (a @ _f64(d[w]).T for w in ("wq", "wk", "wv"))
        if c.get("bias"):
            q, k, v = (t + torch.from_numpy(d[w]).cuda().double() for t, w in ((q, "bq"), (k, "bk"), (v, "bv")))
        q, k, v = q.view(n, nh, hd), k.view(n, nk, hd), v.view(n, nk, hd)
        if c.get("qk_norm"):
            q, k = _norm(q, d["q_norm"]), _norm(k, d["k_norm"])
        q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
        if caches[li]:
            k, v = torch.cat([caches[li][0], k]), torch.cat([caches[li][1], v])
        caches[li] = [k, v]
        out = torch.empty(n, nh, hd, dtype=torch.float64, device="cuda")
        for h in range(nh):
            g = h // (nh // nk)
            sc = (q[:, h] @ k[:, g].T / math.sqrt(hd)).masked_fill(~seen, -math.inf)
            out[:, h] = torch.softmax(sc, -1) @ v[:, g]
        x = x + _q8(out.view(n, -1)) @ _f64(d["wo"]).T
        a = _q8(_norm(x, d["rms_ffn"]))
        if c.get("experts"):
            p, sel = torch.topk(torch.softmax(a @ _f64(d["router"]).T, -1), c["topk"])
            p, y = p / p.sum(-1, keepdim=True), torch.zeros_like(x)
            for e in sorted(set(sel.flatten().tolist())):
                t, slot = torch.nonzero(sel == e, as_tuple=True)
                h1, h3 = a[t] @ _f64(d["e1"][e]).T, a[t] @ _f64(d["e3"][e]).T
                y[t] += _q8(p[t, slot, None] * torch.nn.functional.silu(h1) * h3) @ _f64(d["e2"][e]).T
            x = x + y
        else:
            h = torch.nn.functional.silu(a @ _f64(d["w1"]).T) * (a @ _f64(d["w3"]).T)
            x = x + _q8(h) @ _f64(d["w2"]).T
    return x


def exact(case, seed):
    c = case
    if c["kind"] == "tensor":
        a, b = (torch.from_numpy(t).double().cuda() for t in _tensor_inputs(c, seed))
        r = a @ (b.T if c["transposed"] else b)
        return r if c["dtype"] == "f32" else None
    if c["kind"] == "products":
        q = _q8 if c["format"] in ("q8", "q4") else (lambda t: t)
        return [[_f64(m) @ q(torch.from_numpy(x).cuda().double()) for m in ms] for x, ms in _products_inputs(c, seed)]
    if c["kind"] == "block_scaled":
        v = _block_scaled_inputs(c, seed)
        xq, xo, x = (_e4m3(torch.from_numpy(v[k]).cuda().double()) for k in ("xq", "xo", "x"))
        d, h, y = c["dim"], c["expert_rows"], []
        for e in v["ids"].tolist():
            w1, w3, w2 = ((f, r, k, w[e * r * k // 2:(e + 1) * r * k // 2], s[e * r * k // 32:(e + 1) * r * k // 32])
                          for (f, _, k, w, s), r in ((v["w1"], h), (v["w3"], h), (v["w2"], d)))
            y.append(_f64(w2) @ _e4m3(torch.nn.functional.silu(_f64(w1) @ x) * (_f64(w3) @ x)))
        return [_f64(v["wq"]) @ xq, _f64(v["wo"]) @ xo, torch.cat(y)]
    layers, head, src = _model(c, seed)
    if c["kind"] == "forward":
        caches = [None] * c["layers"]
        if c["pos"]:
            past = torch.from_numpy(src.normal(c["pos"], c["dim"])).cuda().double()
            _forward64(c, layers, past, 0, caches)
        x = torch.from_numpy(src.normal(c["tokens"], c["dim"])).cuda().double()
        return _forward64(c, layers, x, c["pos"], caches)
    if c["temperature"] or c["seqs"] * c["layers"] > 32 or c.get("experts") and c["seqs"] > 1:
        return None  # drawn tokens, or too long in 64 bits
    embed, outs = _f64(head["embed"]), []
    for z in range(c["seqs"]):
        caches, toks, logits = [None] * c["layers"], head["prompts"][z].tolist(), None
        for i in range(c["steps"]):
            new = toks[0 if i == 0 else -1:]
            x = _forward64(c, layers, embed[new], len(toks) - len(new), caches)
            logits = embed @ _q8(_norm(x[-1], head["rms_final"]))
            toks.append(int(logits.argmax()))
        outs.append(logits)
    return {"logits": outs[0] if c["seqs"] == 1 else torch.stack(outs), "tokens": None}
