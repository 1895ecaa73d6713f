"""The work that programs built on tensor-ash have it do, as measurable cases.

A case is a dict of plain values; ``path`` says which part of the library it
takes and the other values are its sizes and options:

* ``gemm``        one fused-epilogue matrix product (``Executor.run_ops``):
                  f32, f32 activations on f16 weights, or f16 activations;
* ``decode_mlp``  the SwiGLU MLPs of several layers for 1-8 new tokens on
                  packed f16 weights, one dependent op graph;
* ``decode_layer``   one new token through a whole decoder layer, recorded
                  once (``prepare_exec_ops``) and replayed, as a decode loop
                  does;
* ``prefill_mlp``    a prompt's SwiGLU MLP on f16 weights, one op graph;
* ``prefill_layer``  a prompt through a whole decoder layer, one mixed-op
                  graph (``run_exec_ops``);
* ``attention``   causal prefill attention of a prompt (or of its next chunk
                  against a warm cache).

Sizes are those of the repository's own benchmark and tests (the five
BASELINE workloads, TinyLlama- and Llama-3-8B-shaped layers) or generic.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "tensor-ash_amd"))

import tensor_ash as ta  # noqa: E402

ACT = {"none": ta.ACTIVATION_NONE, "relu": ta.ACTIVATION_RELU, "silu": ta.ACTIVATION_SILU,
       "gelu": ta.ACTIVATION_GELU}
EPS = 1e-5


def listed():
    return [
        # The smallest call: one 512^3 product with bias + ReLU, where the
        # submission and the launch count as much as the arithmetic.
        dict(name="gemm_512", path="gemm", kind="f32", batch=1, m=512, n=512, k=512, bias=True, act="relu",
             binary="none"),
        # The repository's headline workload.
        dict(name="gemm_4096", path="gemm", kind="f32", batch=1, m=4096, n=4096, k=4096, bias=True, act="relu",
             binary="none"),
        # A batch of independent products with per-batch bias + GELU.
        dict(name="gemm_batched_gelu", path="gemm", kind="f32", batch=8, m=2048, n=2048, k=2048, bias=True,
             act="gelu", binary="none"),
        # Sizes that fit no tile: odd rows, columns and depth, gated by D.
        dict(name="gemm_ragged", path="gemm", kind="f32", batch=1, m=1000, n=1531, k=777, bias=True, act="silu",
             binary="mul"),
        # A small output over a very deep K.
        dict(name="gemm_deep_k", path="gemm", kind="f32", batch=1, m=64, n=256, k=65536, bias=False, act="none",
             binary="none"),
        # Greedy decoding of one sequence: eight TinyLlama MLPs per pass
        # (554 MB of weights, more than the last-level cache holds).
        dict(name="decode_mlp_m1", path="decode_mlp", rows=1, hidden=2048, ffn=5632, layers=8),
        # The same for eight sequences together.
        dict(name="decode_mlp_m8", path="decode_mlp", rows=8, hidden=2048, ffn=5632, layers=8),
        # One new token of one sequence through a whole TinyLlama layer.
        dict(name="decode_layer", path="decode_layer", hidden=2048, heads=32, kv_heads=4, dh=64, ffn=5632,
             t_max=2048, pos=1023, cache="f32"),
        # A 512-token prompt through a whole TinyLlama layer.
        dict(name="prefill_layer_512", path="prefill_layer", tokens=512, hidden=2048, heads=32, kv_heads=4, dh=64,
             ffn=5632, acts="f16"),
        # A 2048-token prompt's MLP at Llama-3-8B widths.
        dict(name="prefill_mlp_2048", path="prefill_mlp", tokens=2048, hidden=4096, ffn=14336),
        # Attention of a 2048-token prompt, f16 caches and activations.
        dict(name="attention_2048", path="attention", tokens=2048, heads=32, kv_heads=8, dh=128, pos=0, dtype="f16"),
        # Attention of a prompt's next 512 tokens against a warm f32 cache.
        dict(name="attention_chunk_f32", path="attention", tokens=512, heads=32, kv_heads=4, dh=64, pos=512,
             dtype="f32"),
    ]


# ------------------------------------------------------------------ drawing


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi):
    """Log-uniform; one in three as it comes (odd ones among them), else a
    multiple of 8 or of 64."""
    v = _log(rng, lo, hi)
    step = rng.choice([1, 8, 64])
    return max(1, (v + step // 2) // step * step)


def draw(rng):
    path = rng.choice(["gemm", "gemm", "gemm", "decode_mlp", "decode_layer", "prefill_mlp", "prefill_layer",
                       "attention", "attention"])
    if path == "gemm":
        kind = rng.choice(["f32", "f32", "f32", "f16w", "f16w", "a16"])
        deep = kind == "f32" and rng.random() < 0.2
        while True:
            batch = rng.choice([1, 1, 1, 2, 3, 8])
            if deep:
                batch, m, n, k = 1, _size(rng, 16, 256), _size(rng, 64, 512), _size(rng, 8192, 131072)
            else:
                m, n, k = _size(rng, 1, 4096), _size(rng, 64, 6144), _size(rng, 64, 6144)
            if kind == "a16":  # its kernels take whole multiples of these only
                m, n, k = max(1, round(m / 64)) * 64, max(1, round(n / 64)) * 64, max(1, round(k / 32)) * 32
            if batch * m * n * k <= 4096 ** 3:
                break
        plain = kind == "a16"  # f16 activations take no epilogue
        return dict(path=path, kind=kind, batch=batch, m=m, n=n, k=k, bias=not plain and rng.random() < 0.5,
                    act="none" if plain else rng.choice(["none", "relu", "silu", "gelu"]),
                    binary="none" if plain else rng.choice(["none", "none", "add", "mul"]))
    if path == "decode_mlp":
        hidden = 64 * _log(rng, 8, 48)
        return dict(path=path, rows=rng.randint(1, 8), hidden=hidden, ffn=64 * _log(rng, 16, 128),
                    layers=rng.randint(2, 8))
    if path == "decode_layer":
        dh = rng.choice([64, 128])
        kv_heads = rng.choice([2, 4, 8])
        heads = kv_heads * rng.choice([1, 4, 8] if dh * kv_heads <= 512 else [1, 4])
        t_max = 2048
        return dict(path=path, hidden=heads * dh, heads=heads, kv_heads=kv_heads, dh=dh, ffn=64 * _log(rng, 16, 128),
                    t_max=t_max, pos=rng.randint(0, t_max - 1), cache=rng.choice(["f32", "f16"]))
    if path == "prefill_mlp":
        return dict(path=path, tokens=_size(rng, 16, 2048), hidden=64 * _log(rng, 8, 64),
                    ffn=64 * _log(rng, 16, 224))
    if path == "prefill_layer":
        dh = rng.choice([64, 128])
        kv_heads = rng.choice([2, 4, 8])
        heads = kv_heads * rng.choice([1, 4])
        return dict(path=path, tokens=_size(rng, 32, 1024), hidden=heads * dh, heads=heads, kv_heads=kv_heads, dh=dh,
                    ffn=64 * _log(rng, 16, 128), acts=rng.choice(["f32", "f16"]))
    kv_heads = rng.choice([1, 4, 8])
    return dict(path="attention", tokens=_size(rng, 16, 2048), heads=kv_heads * rng.choice([1, 4]), kv_heads=kv_heads,
                dh=rng.choice([64, 128]), pos=rng.choice([0, 0, _log(rng, 1, 2048)]),
                dtype=rng.choice(["f32", "kv16", "f16"]))


# ---------------------------------------------------------- device tensors

_ENGINE = None


def _engine():
    """One context and executor for the program, routing on the heuristics."""
    global _ENGINE
    if _ENGINE is None:
        torch.cuda.init()
        ctx = ta.Context("index:0")
        _ENGINE = ta.Executor(ctx, n_slots=2, max_calls_per_submit=64, tune=False)
    return _ENGINE


class _Memory:
    """The device memory of a library tensor, for torch (keeps it alive)."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tensor.shape, "typestr": "<f2" if tensor.f16 else "<f4",
            "data": (tensor.device_address, False), "strides": None, "version": 3}


def _view(tensor):
    return torch.as_tensor(_Memory(tensor), device="cuda")


def _put(ex, value, shape=None, f16=False):
    t = ex.tensor(list(shape or value.shape), f16)
    _view(t).copy_(value.reshape(t.shape))
    return t


class _Inputs:
    """Seeded inputs: activations are standard normal, f16 weights normal
    with 0.02, norm weights around 1.  The same draws feed exact()."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda") * std

    def weight(self, k, n, batch=None):
        return (self.normal(*((k, n) if batch is None else (batch, k, n))) * 0.02).half()

    def gain(self, n):
        return 1.0 + 0.1 * self.normal(n)


def _packed(w):
    """pack_f16w_row_tiles on the GPU: [K, N] -> [N / tile][K][tile]."""
    k, n = w.shape
    tile = ta.f16w_row_tile_n(k, n)
    return w.view(k, n // tile, tile).permute(1, 0, 2).contiguous().view(k, n)


def _rope_table(t_max, dh):
    inv = 10000.0 ** (-2.0 * torch.arange(dh // 2, device="cuda", dtype=torch.float64) / dh)
    theta = torch.arange(t_max, device="cuda", dtype=torch.float64)[:, None] * inv[None, :]
    return torch.stack([theta.cos(), theta.sin()], dim=-1).float()


# ------------------------------------------------------------------ inputs


def _gemm_inputs(c, seed):
    r = _Inputs(seed)
    plane = (lambda *s: s) if c["batch"] == 1 else (lambda *s: (c["batch"], *s))
    v = {"a": r.normal(*plane(c["m"], c["k"]))}
    if c["kind"] == "f32":
        v["b"] = r.normal(*plane(c["k"], c["n"]))
    else:
        v["b"] = r.weight(c["k"], c["n"], None if c["batch"] == 1 else c["batch"])
    if c["kind"] == "a16":
        v["a"] = v["a"].half()
    if c["bias"]:
        v["bias"] = r.normal(*plane(c["n"]))
    if c["binary"] != "none":
        v["d"] = r.normal(*plane(c["m"], c["n"]))
    return v


def _mlp_weights(r, hidden, ffn):
    return {"up": r.weight(hidden, ffn), "gate": r.weight(hidden, ffn), "down": r.weight(ffn, hidden)}


def _decode_mlp_inputs(c, seed):
    r = _Inputs(seed)
    return {"x": r.normal(c["rows"], c["hidden"]),
            "layers": [_mlp_weights(r, c["hidden"], c["ffn"]) for _ in range(c["layers"])]}


def _decode_layer_inputs(c, seed):
    r = _Inputs(seed)
    hid, kv = c["hidden"], c["kv_heads"] * c["dh"]
    cache = torch.float16 if c["cache"] == "f16" else torch.float32
    v = {"x": r.normal(1, hid), "g1": r.gain(hid), "g2": r.gain(hid), "table": _rope_table(c["t_max"], c["dh"]),
         "q": r.weight(hid, hid), "k": r.weight(hid, kv), "v": r.weight(hid, kv), "o": r.weight(hid, hid),
         **_mlp_weights(r, hid, c["ffn"])}
    v["kt"] = r.normal(c["kv_heads"], c["dh"], c["t_max"]).to(cache)
    v["vc"] = r.normal(c["kv_heads"], c["t_max"], c["dh"]).to(cache)
    return v


def _prefill_layer_inputs(c, seed):
    r = _Inputs(seed)
    hid = c["hidden"]
    return {"x": r.normal(c["tokens"], hid), "g1": r.gain(hid), "g2": r.gain(hid),
            "table": _rope_table(c["tokens"], c["dh"]),
            "qkv": r.weight(hid, (c["heads"] + 2 * c["kv_heads"]) * c["dh"]), "o": r.weight(hid, hid),
            **_mlp_weights(r, hid, c["ffn"])}


def _attention_inputs(c, seed):
    r = _Inputs(seed)
    t = c["pos"] + c["tokens"]
    q = r.normal(c["heads"], c["tokens"], c["dh"])
    kt, v = r.normal(c["kv_heads"], c["dh"], t), r.normal(c["kv_heads"], t, c["dh"])
    return {"q": q.half() if c["dtype"] == "f16" else q,
            "kt": kt if c["dtype"] == "f32" else kt.half(), "v": v if c["dtype"] == "f32" else v.half()}


# ----------------------------------------------------------------- prepare


def _prepare_gemm(ex, c, v):
    t = {key: _put(ex, x, f16=x.dtype == torch.float16) for key, x in v.items()}
    plane = [c["m"], c["n"]] if c["batch"] == 1 else [c["batch"], c["m"], c["n"]]
    out = ex.tensor(plane, f16=c["kind"] == "a16")
    binary = {"none": ta.BINARY_NONE, "add": ta.BINARY_ADD_SCALED, "mul": ta.BINARY_MUL}[c["binary"]]
    op = ta.MatmulOp(t["a"], t["b"], out, epilogue=ta.Epilogue(
        bias=t.get("bias"), activation=ACT[c["act"]], binary=binary, d=t.get("d"), beta=0.5))
    return {"call": lambda: ex.run_ops([op]), "out": _view(out)}


def _mlp_ops(x, residual, up, gate, out, w, **kw):
    """up; gate * SiLU * up; down + residual."""
    pack = {key: val for key, val in kw.items() if key == "packed_b"}
    E = ta.Epilogue
    return [ta.MatmulOp(x, w["up"], up, **kw),
            ta.MatmulOp(x, w["gate"], gate, epilogue=E(activation=ta.ACTIVATION_SILU, binary=ta.BINARY_MUL, d=up),
                        **kw),
            ta.MatmulOp(gate, w["down"], out, epilogue=E(binary=ta.BINARY_ADD_SCALED, d=residual, beta=1.0), **pack)]


def _prepare_decode_mlp(ex, c, v):
    x, ops = _put(ex, v["x"]), []
    for layer in v["layers"]:
        w = {key: _put(ex, _packed(val), f16=True) for key, val in layer.items()}
        up, gate, y = ex.tensor([c["rows"], c["ffn"]]), ex.tensor([c["rows"], c["ffn"]]), \
            ex.tensor([c["rows"], c["hidden"]])
        ops += _mlp_ops(x, x, up, gate, y, w, packed_b=True)
        x = y
    return {"call": lambda: ex.run_op_graph(ops), "out": _view(x)}


def _prepare_decode_layer(ex, c, v):
    hid, h, hkv, dh, t_max = c["hidden"], c["heads"], c["kv_heads"], c["dh"], c["t_max"]
    group = h // hkv
    pos = ex.create_pos_buffer()
    pos.set(c["pos"])
    w = {key: _put(ex, _packed(v[key]), f16=True) for key in ("q", "k", "v", "o", "up", "gate", "down")}
    x, g1, g2, table = (_put(ex, v[key]) for key in ("x", "g1", "g2", "table"))
    kt, vc = (_put(ex, v[key], f16=c["cache"] == "f16") for key in ("kt", "vc"))
    q, k, vv, o = ex.tensor([1, hid]), ex.tensor([1, hkv * dh]), ex.tensor([1, hkv * dh]), ex.tensor([1, hid])
    qh, attn, flat = ex.tensor([hkv, group, dh]), ex.tensor([hkv, group, dh]), ex.tensor([1, hid])
    up, gate, y = ex.tensor([1, c["ffn"]]), ex.tensor([1, c["ffn"]]), ex.tensor([1, hid])
    scratch = ex.tensor([hkv * ta.ATTN_DECODE_MAX_CHUNKS * group * (dh + 2)])
    E, at = ta.ExecOp, dict(head_dim=dh, pos_addr=pos.device_address)
    normed, row = dict(packed_b=True, normed_a=(g1, EPS)), ta.CopyDesc((hid, 1, 1), (1, 0, 0), (1, 0, 0))
    ops = [
        E.matmul(ta.MatmulOp(x, w["q"], q, store=ta.MatmulStore(ta.STORE_ROPE, ta.MatmulStoreDesc(**at), table=table),
                             **normed)),
        E.matmul(ta.MatmulOp(x, w["k"], k, store=ta.MatmulStore(
            ta.STORE_ROPE_SCATTER, ta.MatmulStoreDesc(pos_scale=1, stride_head=dh * t_max, stride_dim=t_max, **at),
            table=table, dst=kt), **normed)),
        E.matmul(ta.MatmulOp(x, w["v"], vv, store=ta.MatmulStore(
            ta.STORE_SCATTER, ta.MatmulStoreDesc(pos_scale=dh, stride_head=t_max * dh, stride_dim=1, **at), dst=vc),
            **normed)),
        E.copy_strided(q, qh, row),
        E.attn_decode(qh, kt, vc, scratch, attn, ta.AttnDecodeDesc(1, 1.0 / math.sqrt(dh), pos.device_address)),
        E.copy_strided(attn, flat, row),
        E.matmul(ta.MatmulOp(flat, w["o"], o, epilogue=ta.Epilogue(binary=ta.BINARY_ADD_SCALED, d=x, beta=1.0),
                             packed_b=True)),
    ] + [E.matmul(op) for op in _mlp_ops(o, o, up, gate, y, w, packed_b=True, normed_a=(g2, EPS))]
    step = ex.prepare_exec_ops(ops)
    return {"call": step.run, "out": {"y": _view(y), "kt": _view(kt), "v": _view(vc)}, "keep": (pos, step)}


def _prepare_prefill_mlp(ex, c, v):
    w = {key: _put(ex, val, f16=True) for key, val in v["layers"][0].items()}
    x = _put(ex, v["x"])
    up, gate, y = ex.tensor([c["tokens"], c["ffn"]]), ex.tensor([c["tokens"], c["ffn"]]), \
        ex.tensor([c["tokens"], c["hidden"]])
    ops = _mlp_ops(x, x, up, gate, y, w)
    return {"call": lambda: ex.run_op_graph(ops), "out": _view(y)}


def _prepare_prefill_layer(ex, c, v):
    t, hid, h, hkv, dh = c["tokens"], c["hidden"], c["heads"], c["kv_heads"], c["dh"]
    qkv_n, f16 = (h + 2 * hkv) * dh, c["acts"] == "f16"
    w = {key: _put(ex, v[key], f16=True) for key in ("qkv", "o", "up", "gate", "down")}
    x, g1, g2, table = (_put(ex, v[key]) for key in ("x", "g1", "g2", "table"))
    xn, qkv, attn, o, on = (ex.tensor([t, n]) for n in (hid, qkv_n, hid, hid, hid))
    up, gate, y = ex.tensor([t, c["ffn"]]), ex.tensor([t, c["ffn"]]), ex.tensor([t, hid])
    kt, vc = ex.tensor([hkv, dh, t], f16), ex.tensor([hkv, t, dh], f16)
    E, scale = ta.ExecOp, 1.0 / math.sqrt(dh)
    ops = [E.rms_norm(x, g1, xn, EPS), E.matmul(ta.MatmulOp(xn, w["qkv"], qkv))]
    if f16:
        qkv16, q16, attn16 = ex.tensor([t, qkv_n], True), ex.tensor([h, t, dh], True), ex.tensor([t, hid], True)
        ops += [E.copy_strided(qkv, qkv16, ta.CopyDesc((qkv_n, t, 1), (1, qkv_n, 0), (1, qkv_n, 0))),
                E.prefill_qkv_pack(qkv16, table, q16, kt, vc, ta.PrefillQkvPackDesc(h, hkv, dh, dh, 0)),
                E.flash_attn(q16, kt, vc, attn16, ta.FlashAttentionDesc(t, 0, scale, out_token_major_heads=h)),
                E.copy_strided(attn16, attn, ta.CopyDesc((hid, t, 1), (1, hid, 0), (1, hid, 0)))]
    else:
        q, k = ex.tensor([t, hid]), ex.tensor([t, hkv * dh])
        ops += [E.copy_strided(qkv, q, ta.CopyDesc((hid, t, 1), (1, qkv_n, 0), (1, hid, 0))),
                E.copy_strided(qkv, k, ta.CopyDesc((hkv * dh, t, 1), (1, qkv_n, 0), (1, hkv * dh, 0), src_offset=hid)),
                E.rope(q, table, q, ta.RopeDesc(h, dh, dh, 0)),
                E.rope_scatter(k, table, kt, ta.RopeDesc(hkv, dh, dh, 0), ta.RopeScatterDesc(0, (1, dh * t, t))),
                E.copy_strided(qkv, vc, ta.CopyDesc((dh, hkv, t), (1, dh, qkv_n), (1, t * dh, dh),
                                                    src_offset=hid + hkv * dh)),
                E.flash_attn(q, kt, vc, attn, ta.FlashAttentionDesc(t, 0, scale, token_major_heads=h,
                                                                    out_token_major_heads=h))]
    ops += [E.matmul(ta.MatmulOp(attn, w["o"], o, epilogue=ta.Epilogue(binary=ta.BINARY_ADD_SCALED, d=x, beta=1.0))),
            E.rms_norm(o, g2, on, EPS)] + [E.matmul(op) for op in _mlp_ops(on, o, up, gate, y, w)]
    return {"call": lambda: ex.run_exec_ops(ops), "out": {"y": _view(y), "kt": _view(kt), "v": _view(vc)}}


def _prepare_attention(ex, c, v):
    q, kt, vc = (_put(ex, v[key], f16=v[key].dtype == torch.float16) for key in ("q", "kt", "v"))
    out = ex.tensor([c["heads"], c["tokens"], c["dh"]], f16=c["dtype"] == "f16")
    desc = ta.FlashAttentionDesc(c["pos"] + c["tokens"], c["pos"], 1.0 / math.sqrt(c["dh"]))
    return {"call": lambda: ex.flash_attention(q, kt, vc, out, desc), "out": _view(out)}


def prepare(case, seed):
    ex, path = _engine(), case["path"]
    values = _values(case, seed)
    state = {"gemm": _prepare_gemm, "decode_mlp": _prepare_decode_mlp, "decode_layer": _prepare_decode_layer,
             "prefill_mlp": _prepare_prefill_mlp, "prefill_layer": _prepare_prefill_layer,
             "attention": _prepare_attention}[path](ex, case, values)
    torch.cuda.synchronize()  # the library runs on streams of its own
    return state


def _values(case, seed):
    path = case["path"]
    if path == "prefill_mlp":
        return _decode_mlp_inputs(dict(rows=case["tokens"], hidden=case["hidden"], ffn=case["ffn"], layers=1), seed)
    return {"gemm": _gemm_inputs, "decode_mlp": _decode_mlp_inputs, "decode_layer": _decode_layer_inputs,
            "prefill_layer": _prefill_layer_inputs, "attention": _attention_inputs}[path](case, seed)


def run(state):
    """One pass: a submission, and the wait for it that the library's calls
    include."""
    state["call"]()
    return state["out"]


# -------------------------------------------------------- work, tolerances


def work(case):
    c, path = case, case["path"]
    if path == "gemm":
        mn, mk, kn = c["m"] * c["n"], c["m"] * c["k"], c["k"] * c["n"]
        a, b, o = {"f32": (4, 4, 4), "f16w": (4, 2, 4), "a16": (2, 2, 2)}[c["kind"]]
        extra = 4 * c["n"] * c["bias"] + 4 * mn * (c["binary"] != "none")
        return {"bytes": c["batch"] * (a * mk + b * kn + o * mn + extra), "flops": 2 * c["batch"] * mn * c["k"]}
    if path in ("decode_mlp", "prefill_mlp"):
        rows, layers = c.get("rows", c.get("tokens")), c.get("layers", 1)
        weights = 3 * c["hidden"] * c["ffn"]
        return {"bytes": layers * 2 * weights + 8 * rows * c["hidden"], "flops": 2 * layers * rows * weights}
    if path == "attention":
        t, pos, h, dh = c["tokens"], c["pos"], c["heads"], c["dh"]
        io, kv = {"f32": (4, 4), "kv16": (4, 2), "f16": (2, 2)}[c["dtype"]]
        pairs = t * pos + t * (t + 1) // 2
        return {"bytes": 2 * io * h * t * dh + 2 * kv * c["kv_heads"] * (t + pos) * dh, "flops": 4 * dh * h * pairs}
    hid, kv = c["hidden"], c["kv_heads"] * c["dh"]
    weights = 2 * hid * hid + 2 * hid * kv + 3 * hid * c["ffn"]
    if path == "decode_layer":
        item = 2 if c["cache"] == "f16" else 4
        return {"bytes": 2 * weights + 2 * item * kv * (c["pos"] + 1) + 8 * hid,
                "flops": 2 * weights + 4 * hid * (c["pos"] + 1)}
    t = c["tokens"]
    item = 2 if c["acts"] == "f16" else 4
    return {"bytes": 2 * weights + 8 * t * hid + 2 * item * t * kv,
            "flops": 2 * t * weights + 2 * hid * t * (t + 1)}


def tolerance(case):
    """Relative 2-norm differences that another correct implementation at
    the same precision shows, about four times what was measured."""
    path = case["path"]
    if path == "gemm":
        if case["kind"] == "a16":
            return {"rel": 1e-3}  # f16 results
        if case["kind"] == "f16w":
            return {"rel": 1.5e-3}  # A may be rounded to f16 as it is staged
        return {"rel": 1e-5}  # f32 sums in any order
    if path == "decode_mlp":
        return {"rel": 1e-5}
    if path == "decode_layer":
        # an f16 cache entry may round the other way
        return {"rel": 1e-5 if case["cache"] == "f32" else 1e-3}
    if path == "attention":
        return {"rel": 1e-3 if case["dtype"] == "f16" else 1e-5}
    return {"rel": 2e-3}  # f16 activations in part; A rounded to f16 per product


# ------------------------------------------------------------------- exact


def _act(x, act):
    if act == "relu":
        return torch.relu(x)
    if act == "silu":
        return x * torch.sigmoid(x)
    if act == "gelu":
        return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))
    return x


def _norm(x, gain):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * gain.double()


def _mlp(x, residual, w):
    h = _act(x @ w["gate"].double(), "silu") * (x @ w["up"].double())
    return h @ w["down"].double() + residual


def _rope(x, table, pos):
    """x [T, heads, dh], interleaved pairs rotated by table[pos + t]."""
    cs = table[pos:pos + x.shape[0]].double()[:, None]
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * cs[..., 0] - b * cs[..., 1], a * cs[..., 1] + b * cs[..., 0]], dim=-1).reshape(x.shape)


def _causal(q, kt, v, pos):
    """q [H, T, dh], kt [H_kv, dh, S], v [H_kv, S, dh] -> [H, T, dh], one
    head at a time."""
    h, t, dh = q.shape
    group = h // kt.shape[0]
    i = torch.arange(t, device=q.device)[:, None] + pos
    mask = torch.arange(kt.shape[2], device=q.device)[None, :] > i
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for j in range(h):
        s = (q[j].double() @ kt[j // group].double()) / math.sqrt(dh)
        out[j] = torch.softmax(s.masked_fill(mask, -math.inf), dim=-1) @ v[j // group].double()
    return out


def exact(case, seed):
    c, path = case, case["path"]
    v = _values(case, seed)
    if path == "gemm":
        a, b = v["a"].double(), v["b"].double()
        r = a @ b if c["batch"] == 1 else torch.stack([x @ y for x, y in zip(a, b)])
        if c["bias"]:
            r = r + (v["bias"].double() if c["batch"] == 1 else v["bias"].double()[:, None, :])
        r = _act(r, c["act"])
        if c["binary"] == "add":
            r = r + 0.5 * v["d"].double()
        elif c["binary"] == "mul":
            r = r * v["d"].double()
        return r
    if path in ("decode_mlp", "prefill_mlp"):
        x = v["x"].double()
        for w in v["layers"]:
            x = _mlp(x, x, w)
        return x
    if path == "attention":
        return _causal(v["q"], v["kt"], v["v"], c["pos"])
    h, hkv, dh = c["heads"], c["kv_heads"], c["dh"]
    x = v["x"].double()
    xn = _norm(x, v["g1"])
    if path == "decode_layer":
        p = c["pos"]
        kt, vc = v["kt"].double(), v["vc"].double()
        q = _rope((xn @ v["q"].double()).view(1, h, dh), v["table"], p)
        kt[:, :, p] = _rope((xn @ v["k"].double()).view(1, hkv, dh), v["table"], p)[0]
        vc[:, p] = (xn @ v["v"].double()).view(hkv, dh)
        o = _causal(q.view(h, 1, dh), kt[:, :, :p + 1], vc[:, :p + 1], p).reshape(1, -1) @ v["o"].double() + x
        return {"y": _mlp(_norm(o, v["g2"]), o, v), "kt": kt, "v": vc}
    t, hid = c["tokens"], c["hidden"]
    qkv = xn @ v["qkv"].double()
    q = _rope(qkv[:, :hid].reshape(t, h, dh), v["table"], 0).permute(1, 0, 2)
    kt = _rope(qkv[:, hid:hid + hkv * dh].reshape(t, hkv, dh), v["table"], 0).permute(1, 2, 0).contiguous()
    vc = qkv[:, hid + hkv * dh:].reshape(t, hkv, dh).permute(1, 0, 2).contiguous()
    o = _causal(q, kt, vc, 0).permute(1, 0, 2).reshape(t, hid) @ v["o"].double() + x
    return {"y": _mlp(_norm(o, v["g2"]), o, v), "kt": kt, "v": vc}
