"""The calls that this library's speed is measured on.

Every case is one call, or the few calls that a program makes together, through
the public Python API (wpcg), at sizes that occur in use: the matrices of the
Qwen2.5-0.5B, Qwen3-4B, Qwen3-30B-A3B and Gemma-12B shapes that bench.py and
the tests run, and sizes around them.

Kinds:
  matvec    two quantized matrices of one shape, each times the same vector by
            a call of its own (Linear::matvec of gate, then of up)
  layer     the seven projections of consecutive decoder layers as four
            launches each, replayed as one captured graph
  gemm      a quantized matrix times a batch of activations
  moe       the routed-expert MLP of one layer
  decode    single steps of a decoder at a given position, logits to the host
  generate  a prompt, greedy tokens, then one more step's logits
  prefill   a prompt as one call, the last logits to the host
  verify    speculative verification of drafts, every row's logits

Models hold a few layers of their shape and a small vocabulary, so that the
layers, not the output head, are most of a step, as with all layers.
"""
import ctypes
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "wpc-engine_amd"))
import wpcg  # noqa: E402

BLOCK_BYTES = {3: 100, 4: 68}
STD = 0.02  # of the weights
EPS = 1e-6
THETA = 1e6

# layers' shapes: Qwen3-4B (dense) and Qwen3-30B-A3B (moe)
ARCH = {
    "dense": dict(hidden=2560, n_heads=32, n_kv_heads=8, head_dim=128, inter=9728, n_experts=0, top_k=0,
                  moe_inter=0, n_layers=4),
    "moe": dict(hidden=2048, n_heads=32, n_kv_heads=4, head_dim=128, inter=0, n_experts=128, top_k=8,
                moe_inter=768, n_layers=2),
}
VOCAB = 32768


def listed():
    return [
        # gate and up of a 0.5B model (4864x896): one small launch each, latency
        {"name": "matvec-v4-4864x896", "kind": "matvec", "mode": "fast", "scheme": 4, "rows": 4864, "cols": 896},
        # the projections of four decoder layers of a 4B model in the 6-bit
        # format, weights from HBM: the stream of weights of a decode
        {"name": "layers-v3-fast", "kind": "layer", "mode": "fast", "scheme": 3, "arch": "dense", "layers": 4},
        # the same in the bit-exact mode, the library's default, 4-bit format
        {"name": "layers-v4-exact", "kind": "layer", "mode": "exact", "scheme": 4, "arch": "dense", "layers": 4},
        # a handful of sequences decoded together (ragged batch, fp32 in)
        {"name": "gemm-v4-m6-f32", "kind": "gemm", "scheme": 4, "rows": 15360, "cols": 3840, "m": 6, "dtype": "f32"},
        # a full decode batch
        {"name": "gemm-v4-m64-bf16", "kind": "gemm", "scheme": 4, "rows": 3840, "cols": 15360, "m": 64,
         "dtype": "bf16"},
        # a prompt's rows through a projection, fp32 activations carried as two
        # bf16 terms, ragged
        {"name": "gemm-v3-m777-split", "kind": "gemm", "scheme": 3, "rows": 9728, "cols": 2560, "m": 777,
         "dtype": "split"},
        # a long prompt's rows or a training-size batch in bf16
        {"name": "gemm-v4-m1024-bf16", "kind": "gemm", "scheme": 4, "rows": 15360, "cols": 3840, "m": 1024,
         "dtype": "bf16"},
        # a chat turn on the MoE model: short prompt, greedy tokens
        {"name": "generate-moe-fast", "kind": "generate", "arch": "moe", "mode": "fast", "prompt": 48, "new": 48},
        # decode deep in a long context
        {"name": "decode-dense-fast-3000", "kind": "decode", "arch": "dense", "mode": "fast", "position": 3000,
         "steps": 4},
        # the default (bit-exact) mode end to end
        {"name": "generate-dense-exact", "kind": "generate", "arch": "dense", "mode": "exact", "prompt": 12,
         "new": 12},
        # an MoE prompt of one pass
        {"name": "prefill-moe-256", "kind": "prefill", "arch": "moe", "mode": "fast", "start": 0, "n": 256},
        # a long ragged prompt on the dense model
        {"name": "prefill-dense-1000", "kind": "prefill", "arch": "dense", "mode": "fast", "start": 0, "n": 1000},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["matvec", "layer", "gemm", "gemm", "moe", "decode", "generate", "prefill", "prefill", "verify"])
    mode = "fast" if rng.random() < 0.75 else "exact"
    scheme = rng.choice([3, 4])
    arch = rng.choice(["dense", "moe"])
    if kind == "matvec":
        return {"kind": kind, "mode": mode, "scheme": scheme, "rows": _log_int(rng, 128, 40000),
                "cols": 128 * _log_int(rng, 4, 96)}
    if kind == "layer":
        return {"kind": kind, "mode": mode, "scheme": scheme, "arch": "dense", "layers": rng.randint(1, 4)}
    if kind == "gemm":
        rows, cols = _log_int(rng, 512, 16000), 128 * _log_int(rng, 6, 96)
        m = _log_int(rng, 2, 1024)
        while rows * cols * m > 15360 * 3840 * 1024:
            m //= 2
        return {"kind": kind, "scheme": scheme, "rows": rows, "cols": cols, "m": max(2, m),
                "dtype": rng.choice(["bf16", "bf16", "f32", "split"])}
    if kind == "moe":
        return {"kind": kind, "mode": mode, "scheme": scheme, "experts": rng.choice([16, 64, 128]),
                "hidden": rng.choice([1024, 2048]), "inter": rng.choice([512, 768]), "top_k": rng.choice([2, 4, 8])}
    if kind == "decode":
        return {"kind": kind, "arch": arch, "mode": mode, "position": _log_int(rng, 16, 4000),
                "steps": rng.randint(2, 6)}
    if kind == "generate":
        return {"kind": kind, "arch": arch, "mode": mode, "prompt": _log_int(rng, 4, 24 if mode == "exact" else 400),
                "new": rng.randint(4, 16 if mode == "exact" else 48)}
    if kind == "prefill":
        return {"kind": kind, "arch": arch, "mode": "fast", "start": rng.choice([0, 0, _log_int(rng, 8, 900)]),
                "n": _log_int(rng, 5, 1000)}
    return {"kind": kind, "arch": arch, "mode": "fast", "start": _log_int(rng, 16, 1000), "n": rng.randint(2, 64)}


# ---- inputs ------------------------------------------------------------------

def _blocks(rng, scheme, rows, cols):
    """Random reference blocks: uniform codes, values in about +-2.7 STD."""
    n, bb = rows * (cols // 128), BLOCK_BYTES[scheme]
    out = np.empty((n, bb), np.uint8)
    span = rng.uniform(2.2, 3.2, n) * STD
    zp = (-span).astype(np.float16)
    sc = (2 * span / (15 if scheme == 4 else 63)).astype(np.float16)
    out[:, 0:2] = zp.view(np.uint8).reshape(n, 2)
    out[:, 2:4] = sc.view(np.uint8).reshape(n, 2)
    out[:, 4:] = np.frombuffer(rng.bytes(n * (bb - 4)), np.uint8).reshape(n, bb - 4)
    return out.reshape(-1)


def _activations(rng, *shape):
    """Normal values with a few channels of much larger ones, as hidden states have."""
    x = rng.standard_normal(shape, dtype=np.float32)
    hot = rng.integers(0, shape[-1], max(1, shape[-1] // 256))
    x[..., hot] *= np.float32(12.0)
    return x


_CTX = []


def _ctx():
    if not _CTX:
        _CTX.append(wpcg.Context(0))
    return _CTX[0]


class _Dev:
    """A torch tensor as the API's device buffer."""

    def __init__(self, t):
        self.t, self.ptr = t, ctypes.c_void_p(t.data_ptr())


def _up(a):
    return _Dev(torch.from_numpy(np.ascontiguousarray(a)).cuda())


def _out(*shape, dtype=torch.float32):
    return _Dev(torch.zeros(shape, dtype=dtype, device="cuda"))


def _mode(case):
    return wpcg.MODE_FAST if case["mode"] == "fast" else wpcg.MODE_EXACT


DTYPES = {"f32": wpcg.DTYPE_F32, "bf16": wpcg.DTYPE_BF16, "split": wpcg.DTYPE_F32_SPLIT}


def _layer_shapes(arch):
    c = ARCH[arch]
    qd, kvd = c["n_heads"] * c["head_dim"], c["n_kv_heads"] * c["head_dim"]
    h, i = c["hidden"], c["inter"]
    return [("q", qd, h), ("k", kvd, h), ("v", kvd, h), ("o", h, qd), ("gate", i, h), ("up", i, h), ("down", h, i)]


def _matvec_inputs(case, seed):
    rng = np.random.default_rng(seed)
    return [_blocks(rng, case["scheme"], case["rows"], case["cols"]) for _ in range(2)], _activations(rng, case["cols"])


def _layer_inputs(case, seed):
    """Per layer: {name: blocks} and the inputs of q/k/v, o, gate/up and down."""
    rng = np.random.default_rng(seed)
    c = ARCH[case["arch"]]
    qd = c["n_heads"] * c["head_dim"]
    for _ in range(case["layers"]):
        mats = {name: _blocks(rng, case["scheme"], r, k) for name, r, k in _layer_shapes(case["arch"])}
        yield mats, {n: _activations(rng, k) for n, k in (("hidden", c["hidden"]), ("attn", qd),
                                                           ("post", c["hidden"]), ("act", c["inter"]))}


def _bf16_bits(x):
    u = x.view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def _gemm_inputs(case, seed):
    rng = np.random.default_rng(seed)
    return _blocks(rng, case["scheme"], case["rows"], case["cols"]), _activations(rng, case["m"], case["cols"])


def _moe_inputs(case, seed):
    rng = np.random.default_rng(seed)
    h, i, s = case["hidden"], case["inter"], case["scheme"]
    router = rng.standard_normal((case["experts"], h), dtype=np.float32) * np.float32(STD)
    experts = [(_blocks(rng, s, i, h), _blocks(rng, s, i, h), _blocks(rng, s, h, i)) for _ in range(case["experts"])]
    return router, experts, rng.standard_normal(h, dtype=np.float32)


def _model_inputs(case, seed):
    """(config, tensors by name, token ids): 4-bit matrices, random norms."""
    rng = np.random.default_rng(seed)
    a = ARCH[case["arch"]]
    last = {"decode": lambda: case["position"] + case["steps"], "generate": lambda: case["prompt"] + case["new"] + 1,
            "prefill": lambda: case["start"] + case["n"], "verify": lambda: case["start"] + case["n"]}[case["kind"]]()
    cfg = dict(a, vocab=VOCAB, norm_topk=1, tied=0 if a["n_experts"] else 1, max_pos=min(4096, -(-last // 64) * 64),
               eps=EPS, rope_theta=THETA)
    h, hd = a["hidden"], a["head_dim"]
    qd, kvd = a["n_heads"] * hd, a["n_kv_heads"] * hd

    def norm(n):
        return (1.0 + 0.1 * rng.standard_normal(n)).astype(np.float32)

    t = {"model.embed_tokens.weight": _blocks(rng, 4, VOCAB, h), "model.norm.weight": norm(h)}
    if a["n_experts"]:
        t["lm_head.weight"] = _blocks(rng, 4, VOCAB, h)
    for l in range(a["n_layers"]):
        p = "model.layers.%d." % l
        t[p + "input_layernorm.weight"], t[p + "post_attention_layernorm.weight"] = norm(h), norm(h)
        t[p + "self_attn.q_norm.weight"], t[p + "self_attn.k_norm.weight"] = norm(hd), norm(hd)
        for n, r, k in (("q", qd, h), ("k", kvd, h), ("v", kvd, h), ("o", h, qd)):
            t[p + "self_attn.%s_proj.weight" % n] = _blocks(rng, 4, r, k)
        if a["n_experts"]:
            i = a["moe_inter"]
            t[p + "mlp.gate.weight"] = rng.standard_normal((a["n_experts"], h), dtype=np.float32) * np.float32(STD)
            # one draw of blocks for the layer, each expert its own part
            pool = _blocks(rng, 4, a["n_experts"] * 3 * i, h).reshape(a["n_experts"], 3, -1)
            for e in range(a["n_experts"]):
                for j, n in enumerate(("gate", "up", "down")):
                    t[p + "mlp.experts.%d.%s_proj.weight" % (e, n)] = pool[e, j]
        else:
            for n, r, k in (("gate", a["inter"], h), ("up", a["inter"], h), ("down", h, a["inter"])):
                t[p + "mlp.%s_proj.weight" % n] = _blocks(rng, 4, r, k)
    return cfg, t, rng.integers(0, VOCAB, last).astype(np.uint32)


# ---- a pass --------------------------------------------------------------------

def prepare(case, seed):
    ctx, kind = _ctx(), case["kind"]
    s = {"kind": kind}
    if kind == "matvec":
        blocks, x = _matvec_inputs(case, seed)
        s["lins"] = [wpcg.WpcLinear.from_blocks(ctx, case["scheme"], b, case["rows"], case["cols"]).set_mode(
            _mode(case)) for b in blocks]
        s["x"], s["ys"] = _up(x), [_out(case["rows"]) for _ in blocks]
    elif kind == "layer":
        layers = []
        for mats, xs in _layer_inputs(case, seed):
            lin = {n: wpcg.WpcLinear.from_blocks(ctx, case["scheme"], mats[n], r, k).set_mode(_mode(case))
                   for n, r, k in _layer_shapes(case["arch"])}
            x = {n: _up(v) for n, v in xs.items()}
            y = {n: _out(r) for n, r, k in _layer_shapes(case["arch"])}
            layers.append((lin, x, y))

        def launches():
            for lin, x, y in layers:
                wpcg.matvec_multi([lin["q"], lin["k"], lin["v"]], [x["hidden"]] * 3, [y["q"], y["k"], y["v"]])
                lin["o"].matvec_dev(x["attn"], y["o"])
                wpcg.matvec_multi([lin["gate"], lin["up"]], [x["post"]] * 2, [y["gate"], y["up"]])
                lin["down"].matvec_dev(x["act"], y["down"])

        torch.cuda.synchronize()
        s["graph"], s["layers"] = ctx.capture(launches), layers
        s["outs"] = [{n: b.t for n, b in y.items()} for _, _, y in layers]
    elif kind == "gemm":
        blocks, x = _gemm_inputs(case, seed)
        s["lin"] = wpcg.WpcLinear.from_blocks(ctx, case["scheme"], blocks, case["rows"], case["cols"])
        s["lin"].set_mode(wpcg.MODE_FAST)
        s["x"] = _up(_bf16_bits(x).view(np.int16) if case["dtype"] == "bf16" else x)
        s["y"], s["m"], s["dtype"] = _out(case["m"], case["rows"]), case["m"], DTYPES[case["dtype"]]
    elif kind == "moe":
        router, experts, x = _moe_inputs(case, seed)
        m = wpcg.MoeLayer(ctx, case["scheme"], case["experts"], case["hidden"], case["inter"], case["top_k"])
        m.set_router(router).set_mode(_mode(case))
        for e, (g, u, d) in enumerate(experts):
            m.set_expert(e, g, u, d)
        s["moe"], s["x"], s["y"] = m, _up(x), _out(case["hidden"])
        s["ids"], s["w"] = _out(case["top_k"], dtype=torch.int32), _out(case["top_k"])
    else:
        cfg, tensors, toks = _model_inputs(case, seed)
        m = wpcg.Model(ctx, wpcg.SCHEME_V4, wpcg.ModelConfig(**cfg))
        for name, a in tensors.items():
            m.set_tensor(name, a)
        m.set_mode(wpcg.MODE_FAST)
        s["model"], s["toks"] = m, toks
        if kind == "generate":
            s["prompt"], s["new"] = toks[:case["prompt"]], case["new"]
        else:
            # what the cache holds before the call
            s["start"] = case["position"] if kind == "decode" else case["start"]
            if s["start"]:
                m.prefill(toks[:s["start"]], want_logits=False)
        m.set_mode(_mode(case))
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "matvec":
        for lin, y in zip(s["lins"], s["ys"]):
            lin.matvec_dev(s["x"], y)
        return [y.t for y in s["ys"]]
    if kind == "layer":
        s["graph"].launch()
        return s["outs"]
    if kind == "gemm":
        s["lin"].gemm_dev(s["x"], s["m"], s["y"], s["dtype"])
        return s["y"].t
    if kind == "moe":
        s["moe"].forward_dev(s["x"], s["y"], s["ids"], s["w"])
        return {"y": s["y"].t, "ids": s["ids"].t, "weights": s["w"].t}
    m = s["model"]
    if kind == "generate":
        ids, _ = m.generate(s["prompt"], s["new"])
        return {"ids": ids.astype(np.int64), "logits": m.forward_token(int(ids[-1]))[0]}
    m.set_position(s["start"])
    if kind == "decode":
        return [m.forward_token(int(t))[0] for t in s["toks"][s["start"]:]]
    if kind == "prefill":
        return m.prefill(s["toks"][s["start"]:])[0]
    return m.verify(s["toks"][s["start"]:], want_logits=True)[1]


# ---- what a pass cannot do without ---------------------------------------------

def _matrix(scheme, rows, cols):
    return rows * (cols // 128) * BLOCK_BYTES[scheme]


def _model_work(arch, steps, first, logit_rows, batched):
    """`steps` positions from `first` on: the weights once per step, or once if
    the positions come as a batch; the cache, the embedding rows, the logits."""
    c = ARCH[arch]
    h, hd = c["hidden"], c["head_dim"]
    qd, kvd = c["n_heads"] * hd, c["n_kv_heads"] * hd
    att = qd * h + 2 * kvd * h + h * qd
    if c["n_experts"]:
        per = 3 * c["moe_inter"] * h
        used = min(c["n_experts"], c["top_k"] * steps) if batched else c["top_k"] * steps
        mlp_flops, mlp_values = 2 * c["top_k"] * per * steps, used * per
        router = c["n_experts"] * h
    else:
        per = 3 * c["inter"] * h
        mlp_flops, mlp_values, router = 2 * per * steps, per * (1 if batched else steps), 0
    reads = 1 if batched else steps
    positions = sum(first + i + 1 for i in range(steps))
    cache = 2 * kvd * 4 * ((first + steps) if batched else positions) + 2 * kvd * 4 * steps
    layer_bytes = (att * reads + mlp_values) / 128 * 68 + router * 4 * reads + cache
    layer_flops = 2 * att * steps + mlp_flops + 2 * router * steps + 4 * qd * positions
    head = VOCAB * h
    head_reads = 1 if batched else logit_rows
    return (c["n_layers"] * layer_bytes + head / 128 * 68 * head_reads + logit_rows * VOCAB * 4 + steps * h / 128 * 68,
            c["n_layers"] * layer_flops + 2 * head * logit_rows)


def work(case):
    kind = case["kind"]
    if kind == "matvec":
        r, k = case["rows"], case["cols"]
        return {"bytes": 2 * _matrix(case["scheme"], r, k) + 8 * r + 4 * k, "flops": 4 * r * k}
    if kind == "layer":
        sh = _layer_shapes(case["arch"])
        c = ARCH[case["arch"]]
        x = 2 * c["hidden"] + c["n_heads"] * c["head_dim"] + c["inter"]
        return {"bytes": case["layers"] * (sum(_matrix(case["scheme"], r, k) + 4 * r for _, r, k in sh) + 4 * x),
                "flops": case["layers"] * sum(2 * r * k for _, r, k in sh)}
    if kind == "gemm":
        r, k, m = case["rows"], case["cols"], case["m"]
        return {"bytes": _matrix(case["scheme"], r, k) + m * k * (2 if case["dtype"] == "bf16" else 4) + 4 * m * r,
                "flops": 2 * r * k * m}
    if kind == "moe":
        h, i, n, k = case["hidden"], case["inter"], case["experts"], case["top_k"]
        return {"bytes": n * h * 4 + k * 3 * _matrix(case["scheme"], i, h) + 8 * h + 8 * k,
                "flops": 2 * n * h + 2 * k * 3 * i * h}
    if kind == "decode":
        b, f = _model_work(case["arch"], case["steps"], case["position"], case["steps"], False)
    elif kind == "generate":
        if case["mode"] == "fast":
            b0, f0 = _model_work(case["arch"], case["prompt"], 0, 1, True)
            b1, f1 = _model_work(case["arch"], case["new"], case["prompt"], case["new"], False)
            b, f = b0 + b1, f0 + f1
        else:
            n = case["prompt"] + case["new"]
            b, f = _model_work(case["arch"], n, 0, n, False)
    else:
        b, f = _model_work(case["arch"], case["n"], case["start"], case["n"] if kind == "verify" else 1, True)
    return {"bytes": b, "flops": f}


def tolerance(case):
    """EXACT results are fixed bit for bit. FAST ones are 32-bit sums of exact
    weights; X in bf16 is the caller's choice and the same in every
    implementation; as two bf16 terms it is carried to 2^-18."""
    if case.get("mode") == "exact" and case["kind"] != "decode":
        return "exact"
    if case["kind"] in ("matvec", "layer", "moe"):
        return {"rel": 4e-6, "max": 1e-4}
    if case["kind"] == "gemm":
        return {"rel": 1.5e-5 if case["dtype"] == "split" else 8e-6, "max": 3e-4}
    return {"rel": 6e-5, "max": 1e-3}


# ---- the same in 64 bits -------------------------------------------------------

def _dequant(scheme, blocks, rows, cols):
    """float64 [rows][cols] on the GPU."""
    b = torch.from_numpy(np.ascontiguousarray(blocks)).cuda().reshape(rows * (cols // 128), BLOCK_BYTES[scheme])
    par = b[:, :4].contiguous().view(torch.float16).double()
    c = b[:, 4:]
    if scheme == 4:
        codes = torch.cat([c & 15, c >> 4], 1).double()
    else:
        g = c.reshape(-1, 32, 3).to(torch.int32)
        w = g[..., 0] | g[..., 1] << 8 | g[..., 2] << 16
        codes = torch.stack([w & 63, w >> 6 & 63, w >> 12 & 63, w >> 18 & 63], -1).reshape(-1, 128).double()
    return (par[:, 0:1] + codes * par[:, 1:2]).reshape(rows, cols)


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda().double()


def _silu(x):
    return x / (1 + torch.exp(-x))


def _top(scores, k):
    p = torch.softmax(scores, -1)
    w, ids = torch.topk(p, k, -1)
    return w / w.sum(-1, keepdim=True), ids


class _Exact:
    """The decoder in float64 over a whole sequence at once."""

    def __init__(self, cfg, tensors):
        self.c, self.t, self.kept = cfg, tensors, {}

    def w(self, name, rows, cols):
        if name not in self.kept:
            self.kept[name] = _dequant(4, self.t[name], rows, cols)
        return self.kept[name]

    def norm(self, x, name):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(EPS))) * _f64(self.t[name])

    def rope(self, x):
        n, half = x.shape[0], x.shape[-1] // 2
        inv = THETA ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / (2 * half))
        ang = torch.arange(n, dtype=torch.float64, device="cuda")[:, None] * inv
        cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def logits(self, toks, keep):
        """Logits of the last `keep` positions of the sequence."""
        c, t = self.c, self.t
        h, hd, nh, nkv = c["hidden"], c["head_dim"], c["n_heads"], c["n_kv_heads"]
        bb = h // 128 * 68
        rows = t["model.embed_tokens.weight"].reshape(-1, bb)[np.asarray(toks, np.int64)]
        x = _dequant(4, rows.reshape(-1), len(toks), h)
        n = len(toks)
        mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
        for l in range(c["n_layers"]):
            p = "model.layers.%d." % l
            y = self.norm(x, p + "input_layernorm.weight")
            a = p + "self_attn."
            q = (y @ self.w(a + "q_proj.weight", nh * hd, h).T).reshape(n, nh, hd)
            k = (y @ self.w(a + "k_proj.weight", nkv * hd, h).T).reshape(n, nkv, hd)
            v = (y @ self.w(a + "v_proj.weight", nkv * hd, h).T).reshape(n, nkv, hd)
            q, k = self.rope(self.norm(q, a + "q_norm.weight")), self.rope(self.norm(k, a + "k_norm.weight"))
            o = torch.empty(n, nh, hd, dtype=torch.float64, device="cuda")
            for i in range(nh):
                kv = i // (nh // nkv)
                sc = (q[:, i] @ k[:, kv].T.contiguous()) / hd ** 0.5
                o[:, i] = torch.softmax(sc.masked_fill(mask, float("-inf")), -1) @ v[:, kv]
            x = x + o.reshape(n, nh * hd) @ self.w(a + "o_proj.weight", h, nh * hd).T
            y = self.norm(x, p + "post_attention_layernorm.weight")
            if not c["n_experts"]:
                g = y @ self.w(p + "mlp.gate_proj.weight", c["inter"], h).T
                u = y @ self.w(p + "mlp.up_proj.weight", c["inter"], h).T
                x = x + (_silu(g) * u) @ self.w(p + "mlp.down_proj.weight", h, c["inter"]).T
                continue
            i = c["moe_inter"]
            w, ids = _top(y @ _f64(t[p + "mlp.gate.weight"]).T, c["top_k"])
            add = torch.zeros_like(x)
            for e in torch.unique(ids).tolist():
                at, slot = torch.nonzero(ids == e, as_tuple=True)
                q_ = p + "mlp.experts.%d." % e
                g, u = y[at] @ self.w(q_ + "gate_proj.weight", i, h).T, y[at] @ self.w(q_ + "up_proj.weight", i, h).T
                d = (_silu(g) * u) @ self.w(q_ + "down_proj.weight", h, i).T
                add.index_add_(0, at, d * w[at, slot][:, None])
            x = x + add
        x = self.norm(x[-keep:], "model.norm.weight")
        return x @ self.w("lm_head.weight" if c["n_experts"] else "model.embed_tokens.weight", VOCAB, h).T


def exact(case, seed):
    kind = case["kind"]
    if kind == "matvec":
        blocks, x = _matvec_inputs(case, seed)
        return [_dequant(case["scheme"], b, case["rows"], case["cols"]) @ _f64(x) for b in blocks]
    if kind == "layer":
        src = {"q": "hidden", "k": "hidden", "v": "hidden", "o": "attn", "gate": "post", "up": "post", "down": "act"}
        return [{n: _dequant(case["scheme"], mats[n], r, k) @ _f64(xs[src[n]])
                 for n, r, k in _layer_shapes(case["arch"])} for mats, xs in _layer_inputs(case, seed)]
    if kind == "gemm":
        blocks, x = _gemm_inputs(case, seed)
        x = _f64(x) if case["dtype"] == "split" else _f64((_bf16_bits(x).astype(np.uint32) << 16).view(np.float32))
        return x @ _dequant(case["scheme"], blocks, case["rows"], case["cols"]).T
    if kind == "moe":
        router, experts, x = _moe_inputs(case, seed)
        x, h, i, s = _f64(x), case["hidden"], case["inter"], case["scheme"]
        w, ids = _top(_f64(router) @ x, case["top_k"])
        y = torch.zeros(h, dtype=torch.float64, device="cuda")
        for j, e in enumerate(ids.tolist()):
            g, u, d = experts[e]
            y += w[j] * (_dequant(s, d, h, i) @ (_silu(_dequant(s, g, i, h) @ x) * (_dequant(s, u, i, h) @ x)))
        return {"y": y, "ids": ids.int(), "weights": w}
    cfg, tensors, toks = _model_inputs(case, seed)
    m = _Exact(cfg, tensors)
    if kind == "decode":
        return list(m.logits(toks, case["steps"]))
    if kind == "prefill":
        return m.logits(toks, 1)[0]
    if kind == "verify":
        return m.logits(toks, case["n"])
    seq = [int(t) for t in toks[:case["prompt"]]]
    for _ in range(case["new"]):
        seq.append(int(m.logits(seq, 1)[0].argmax()))
    return {"ids": None, "logits": m.logits(seq, 1)[0]}
