"""The engine's work in use, as cases that can be timed and compared.

A case is one call, or the few calls in a row, that a program on the engine
(metalium-rs_amd/miburn.py over include/miburn.h) makes: whole training steps
and a whole prompt, a decoder layer's decode step, and the single layers and
kernels they are made of.  Sizes are those of the repository's own workloads
(the 784-128-10 MLP, the 4-layer transformer, the SmolLM2-135M-shaped decoder,
the matmul sweep, the [8192, 8192] suite) and, in between, the sizes that real
batches and prompts have: not multiples of anything.

`listed()` names the cases, `draw(rng)` gives more of the same ranges,
`prepare(case, seed)` makes what a program holds before the call, `run(state)`
is one pass, `work(case)` its unavoidable bytes and operations,
`tolerance(case)` how far another correct implementation may be off, and
`exact(case, seed)` the outputs in 64 bits.

A result stays on the device, as it does in a program that feeds it to the
next call: `run` returns tensors that name their engine buffers and read them
back when they are looked at.  Every kernel of a pass is on the engine's
stream when `run` returns.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "metalium-rs_amd"))
import miburn  # noqa: E402
from miburn import BF16, F32  # noqa: E402

EPS = 1e-5
ROPE_THETA = 100000.0

# A decoder layer's shape: SmolLM2-135M's, and two generic ones beside it.
LAYERS = {"smollm2": dict(hidden=576, heads=9, kv=3, d=64, inter=1536),
          "wide": dict(hidden=1024, heads=16, kv=4, d=64, inter=2816),
          "mha": dict(hidden=512, heads=8, kv=8, d=64, inter=1408)}
ROW_OPS = ("softmax", "log_softmax", "layer_norm", "rms_norm", "gelu", "silu", "add", "row_sum", "col_sum")


def listed():
    return [
        # The MNIST-sized MLP's training step: some twenty tiny launches, the
        # smallest work a training loop on the engine has.
        dict(name="mlp_step", kind="mlp", batch=64, d_in=784, hidden=128, d_out=10),
        # The 4-layer transformer's training step, forward to SGD, F32.
        dict(name="transformer_step", kind="transformer", batch=16, seq=128, d=256, heads=4, ff=1024, layers=4,
             vocab=8192),
        # A prompt through the whole SmolLM2-135M-shaped decoder to the last
        # position's logits; 500 tokens, as prompts are not powers of two.
        dict(name="prefill_500", kind="prefill", batch=1, t=500, numerics="reference"),
        # One decoder layer of a decode step: one sequence (latency), and a
        # full batch of 32.
        dict(name="decode_layer_b1", kind="decode", shape="smollm2", batch=1, ctx=576, weights="bf16", cache="f32"),
        dict(name="decode_layer_b32", kind="decode", shape="smollm2", batch=32, ctx=576, weights="bf16", cache="f32"),
        # The attention of a batch of prompts.
        dict(name="attention_b4_t512", kind="attention", batch=4, t=512, pos0=0, heads=9, kv=3, d=64, cache="f32"),
        # The matmul sweep's headline size.
        dict(name="matmul_bf16_4096", kind="matmul", dtype="bf16", m=4096, n=4096, k=4096, ta=False, tb=False,
             out="f32"),
        # An F32 product of sizes that nothing divides.
        dict(name="matmul_f32_ragged", kind="matmul", dtype="f32", m=3001, n=2500, k=2047, ta=False, tb=False,
             out="f32"),
        # A Linear layer with bias and residual: F32 activations of a ragged
        # batch of tokens against a stored BF16 weight.
        dict(name="linear_1500", kind="linear", m=1500, n=3072, k=768, bias=True, residual=True),
        # The sweep's batched product.
        dict(name="batched_f32_512", kind="batched", dtype="f32", batch=16, m=512, n=512, k=512, ta=False, tb=False),
        # The suite's row softmax: bound by HBM.
        dict(name="softmax_8192", kind="rows", op="softmax", rows=8192, cols=8192),
        # A language model's head in training: LayerNorm, the vocabulary
        # product, cross-entropy, and the gradients back through all three.
        dict(name="lm_head_train", kind="lm_head", rows=2000, d=256, vocab=8192),
    ]


def _between(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm: odd ones as
    often as even, and one in three rounded to a multiple of 64 or 8."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    step = rng.choice((1, 1, 1, 1, 8, 64)) if hi > 64 else 1
    return min(hi, max(lo, v // step * step if v >= step else v))


def draw(rng):
    kind = rng.choice(("mlp", "transformer", "prefill", "decode", "decode", "attention", "matmul", "matmul", "linear",
                       "batched", "rows", "lm_head"))
    if kind == "mlp":
        return dict(kind=kind, batch=_between(rng, 16, 512), d_in=_between(rng, 100, 1024),
                    hidden=_between(rng, 32, 512), d_out=_between(rng, 10, 100))
    if kind == "transformer":
        heads = rng.choice((2, 4, 8))
        d = heads * rng.choice((16, 32, 64)) if heads < 8 else 256
        return dict(kind=kind, batch=_between(rng, 2, 16), seq=_between(rng, 17, 128), d=d, heads=heads, ff=4 * d,
                    layers=rng.randint(1, 4), vocab=_between(rng, 1000, 8192))
    if kind == "prefill":
        batch = rng.randint(1, 4)
        return dict(kind=kind, batch=batch, t=_between(rng, 33, 600 // batch),
                    numerics=rng.choice(("reference", "reference", "performance")))
    if kind == "decode":
        return dict(kind=kind, shape=rng.choice(("smollm2", "smollm2", "wide", "mha")), batch=_between(rng, 1, 32),
                    ctx=_between(rng, 16, 1000), weights=rng.choice(("bf16", "bf16", "bfp8")),
                    cache=rng.choice(("f32", "bf16")))
    if kind == "attention":
        heads, kv = rng.choice(((9, 3), (8, 8), (16, 4), (4, 2)))
        return dict(kind=kind, batch=_between(rng, 1, 8), t=_between(rng, 16, 512), pos0=rng.choice((0, 0, 64, 301)),
                    heads=heads, kv=kv, d=rng.choice((64, 64, 64, 32, 128)), cache=rng.choice(("f32", "f32", "bf16")))
    if kind == "matmul":
        m, n, k = (_between(rng, 64, 4096) for _ in range(3))
        dtype = rng.choice(("bf16", "f32"))
        return dict(kind=kind, dtype=dtype, m=m, n=n, k=k, ta=rng.random() < 0.25, tb=rng.random() < 0.4,
                    out=rng.choice(("f32", "f32", "bf16")) if dtype == "bf16" else "f32")
    if kind == "linear":
        return dict(kind=kind, m=_between(rng, 16, 4096), n=_between(rng, 256, 4096), k=_between(rng, 256, 3072),
                    bias=rng.random() < 0.5, residual=rng.random() < 0.5)
    if kind == "batched":
        m, n, k = (_between(rng, 32, 640) for _ in range(3))
        return dict(kind=kind, dtype=rng.choice(("bf16", "f32")), batch=rng.randint(2, 48), m=m, n=n, k=k,
                    ta=rng.random() < 0.25, tb=rng.random() < 0.5)
    if kind == "rows":
        rows, op = _between(rng, 64, 16384), rng.choice(ROW_OPS)
        most = (1 << 26) * 2 // (3 if op == "add" else 2)  # as many bytes as the largest listed
        return dict(kind=kind, op=op, rows=rows, cols=_between(rng, 64, min(16384, most // rows)))
    return dict(kind=kind, rows=_between(rng, 100, 4000), d=_between(rng, 64, 512), vocab=_between(rng, 500, 8192))


# ------------------------------------------------------------------ inputs


class _Draws:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, std=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std + mean

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device="cuda")

    def ids(self, hi, *shape):
        return torch.randint(0, hi, shape, generator=self.g, device="cuda", dtype=torch.int32)


def _rope_tables(n, d):
    half = d // 2
    freq = ROPE_THETA ** (-2.0 * np.arange(half) / d)
    ang = np.arange(n)[:, None] * freq[None, :]
    cos, sin = np.cos(ang), np.sin(ang)
    return (torch.from_numpy(np.concatenate([cos, cos], 1)).float().cuda(),
            torch.from_numpy(np.concatenate([-sin, sin], 1)).float().cuda())


def _max_ctx(case):
    return (case["ctx"] + 64) // 64 * 64 + 64


def _inputs(case, seed):
    """The case's input tensors, on the GPU: BF16 where the engine's buffer is."""
    r, kind = _Draws(seed), case["kind"]
    if kind == "mlp":
        return dict(x=r.uniform(case["batch"], case["d_in"]), y=r.ids(case["d_out"], case["batch"], 1))
    if kind == "transformer":
        rows = case["batch"] * case["seq"]
        return dict(tokens=r.ids(case["vocab"], rows, 1), targets=r.ids(case["vocab"], rows, 1))
    if kind == "prefill":
        return dict(ids=r.ids(miburn.SMOLLM2_135M["vocab"], case["batch"], case["t"]))
    if kind == "decode":
        s, b = LAYERS[case["shape"]], case["batch"]
        hid, d, rows = s["hidden"], s["d"], b * s["kv"] * _max_ctx(case)
        cos, sin = _rope_tables(_max_ctx(case), d)
        cache = torch.bfloat16 if case["cache"] == "bf16" else torch.float32

        def weight(n, k):
            return r.normal(n, k, std=0.02).bfloat16()
        return dict(x=r.normal(b, hid), g1=r.normal(1, hid, std=0.1, mean=1.0), g2=r.normal(1, hid, std=0.1, mean=1.0),
                    wqkv=weight((s["heads"] + 2 * s["kv"]) * d, hid), wo=weight(hid, s["heads"] * d),
                    wgu=weight(2 * s["inter"], hid), wdown=weight(hid, s["inter"]), cos=cos, sin=sin,
                    k=r.normal(rows, d).to(cache), v=r.normal(rows, d).to(cache))
    if kind == "attention":
        ctx, d = case["pos0"] + case["t"], case["d"]
        cache = torch.bfloat16 if case["cache"] == "bf16" else torch.float32
        rows = case["batch"] * case["kv"] * ctx
        return dict(q=r.normal(case["batch"] * case["t"], case["heads"] * d), k=r.normal(rows, d).to(cache),
                    v=r.normal(rows, d).to(cache))
    if kind in ("matmul", "batched"):
        m, n, k, b = case["m"], case["n"], case["k"], case.get("batch", 1)
        elem = torch.bfloat16 if case["dtype"] == "bf16" else torch.float32
        return dict(a=r.normal(*((b * k, m) if case["ta"] else (b * m, k))).to(elem),
                    b=r.normal(*((b * n, k) if case["tb"] else (b * k, n))).to(elem))
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        out = dict(x=r.normal(m, k), w=r.normal(n, k, std=0.02).bfloat16())
        if case["bias"]:
            out["bias"] = r.normal(1, n, std=0.02)
        if case["residual"]:
            out["residual"] = r.normal(m, n)
        return out
    if kind == "rows":
        out = dict(x=r.normal(case["rows"], case["cols"]))
        if case["op"] == "add":
            out["y"] = r.normal(case["rows"], case["cols"])
        if case["op"] in ("layer_norm", "rms_norm"):
            out["g"] = r.normal(1, case["cols"], std=0.1, mean=1.0)
        if case["op"] == "layer_norm":
            out["b"] = r.normal(1, case["cols"], std=0.1)
        return out
    rows, d, v = case["rows"], case["d"], case["vocab"]
    lim = 1.0 / math.sqrt(d)
    return dict(x=r.normal(rows, d), g=r.normal(1, d, std=0.1, mean=1.0), b=r.normal(1, d, std=0.1),
                w=(2 * r.uniform(d, v) - 1) * lim, bias=(2 * r.uniform(1, v) - 1) * lim, y=r.ids(v, rows, 1))


# ------------------------------------------------------------------- state

_ENGINE = None


def _engine():
    """The process's engine: a program attaches to the device once."""
    global _ENGINE
    if _ENGINE is None:
        _ENGINE = miburn.Engine(0)
    return _ENGINE


class Result(torch.Tensor):
    """A result on the device: reading it in any way reads its buffer back."""

    @staticmethod
    def of(read):
        t = torch.empty(0).as_subclass(Result)
        t.read = read
        return t

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        def real(v):
            return v.read() if isinstance(v, Result) else v
        return func(*[real(a) for a in args], **{k: real(v) for k, v in (kwargs or {}).items()})


class State:
    """What a program holds: input buffers, a model if it has one, and the
    buffers of the last pass's results (freed when the next pass replaces
    them, as a loop's temporaries are)."""

    def __init__(self, case):
        self.case, self.eng = case, _engine()
        self.ids, self.out, self.results, self.model = {}, {}, {}, None

    def upload(self, name, t):
        host = t.cpu()
        if t.dtype == torch.bfloat16:
            self.ids[name] = self.eng.upload_bf16(host.view(torch.int16).numpy().view(np.uint16))
        elif t.dtype == torch.int32:
            self.ids[name] = self.eng.upload_i32(host.numpy())
        else:
            self.ids[name] = self.eng.upload(host.numpy())

    def download(self, id_):
        host = self.eng.download(id_)
        if host.dtype == np.uint16:
            return torch.from_numpy(host.view(np.int16)).view(torch.bfloat16)
        return torch.from_numpy(host)

    def result(self, name, read=None):
        self.results[name] = Result.of(read or (lambda: self.download(self.out[name])))

    def give(self, **out):
        """The pass's results, in the place of the last one's."""
        for id_ in self.out.values():
            self.eng.free(id_)
        self.out = out
        return self.results

    def __del__(self):
        if self.eng.ctx:
            for id_ in list(self.out.values()) + list(self.ids.values()):
                self.eng.free(id_)
            if self.model is not None:
                self.model.close()


def _transformer_config(case):
    return dict(vocab=case["vocab"], d_model=case["d"], heads=case["heads"], d_ff=case["ff"], layers=case["layers"],
                eps=EPS)


def _model(case, seed):
    """The model of a case, its weights drawn by the engine from the seed."""
    eng = _engine()
    if case["kind"] == "mlp":
        return miburn.Mlp(eng, case["d_in"], case["hidden"], case["d_out"], lcg_seed=seed + 1)
    if case["kind"] == "transformer":
        return miburn.Transformer(eng, _transformer_config(case), seed=seed)
    return miburn.Llama(eng, miburn.SMOLLM2_135M, max_ctx=case["t"], max_batch=case["batch"], seed=seed,
                        numerics=case["numerics"])


MLP_LR, TRANSFORMER_LR = 0.01, 0.05
OUTPUTS = {"decode": ("attn", "out"), "attention": ("out",), "matmul": ("out",), "batched": ("out",),
           "linear": ("out",), "rows": ("out",), "prefill": ("logits",), "mlp": ("loss",), "transformer": ("loss",),
           "lm_head": ("logp", "dw", "dbias", "dx", "dg", "db")}


def prepare(case, seed):
    s, kind = State(case), case["kind"]
    inputs = _inputs(case, seed)
    if kind == "prefill":
        s.tokens = inputs["ids"].cpu().numpy()  # a prompt comes from the host
    else:
        for name, t in inputs.items():
            s.upload(name, t)
    for name in OUTPUTS[kind]:
        s.result(name)
    if kind in ("mlp", "transformer", "prefill"):
        s.model = m = _model(case, seed)
    if kind == "mlp":  # the updated weights are the step's outputs too
        for i, name in enumerate(("w1", "b1", "w2", "b2")):
            s.result(name, lambda i=i: torch.from_numpy(m.param(i)))
    if kind == "transformer":
        for name in ("embed", "head_w", "head_b"):
            s.result(name, lambda name=name: torch.from_numpy(m.param(name)))
        for name in miburn.TRANSFORMER_LAYER_PARAMS:
            s.result(name, lambda name=name: torch.stack([torch.from_numpy(m.param(name, i))
                                                          for i in range(case["layers"])]))
    if kind == "decode":
        if case["weights"] == "bfp8":
            for name in ("wqkv", "wo", "wgu", "wdown"):
                bf = s.ids[name]
                s.ids[name] = s.eng.cast_bfp(bf)
                s.eng.free(bf)
        for name in ("k", "v"):  # the caches with the step's row in them
            s.result(name, lambda name=name: s.download(s.ids[name]))
    return s


# -------------------------------------------------------------------- run


def run(s):
    c, e, i = s.case, s.eng, s.ids
    kind = c["kind"]
    if kind == "mlp":
        return s.give(loss=s.model.train_step_ids(i["x"], i["y"], MLP_LR))
    if kind == "transformer":
        return s.give(loss=s.model.train_step_ids(i["tokens"], i["targets"], c["batch"], c["seq"], TRANSFORMER_LR))
    if kind == "prefill":
        s.model.reset()
        return s.give(logits=s.model.forward(s.tokens))
    if kind == "decode":
        w = LAYERS[c["shape"]]
        span = (c["ctx"] + 64) // 64 * 64
        x1 = e.norm_qkv_attention_o(i["x"], i["g1"], EPS, i["wqkv"], i["cos"], i["sin"], w["heads"], w["kv"], 0, c["ctx"],
                                    span, i["k"], i["v"], w["d"] ** -0.5, i["wo"])
        h = e.norm_matvec(x1, i["g2"], EPS, i["wgu"], 0, True)
        x2 = e.norm_matvec(h, 0, 0.0, i["wdown"], x1, False)
        e.free(h)
        return s.give(attn=x1, out=x2)
    if kind == "attention":
        return s.give(out=e.attention_rows(i["q"], i["k"], i["v"], c["batch"], c["t"], c["heads"], c["kv"], c["pos0"],
                                           c["d"] ** -0.5))
    if kind == "matmul":
        return s.give(out=e.matmul_dram(i["a"], c["ta"], i["b"], c["tb"], BF16 if c["out"] == "bf16" else F32))
    if kind == "batched":
        return s.give(out=e.matmul_dram_batched(i["a"], c["ta"], i["b"], c["tb"], c["batch"], c["m"], c["k"], c["n"]))
    if kind == "linear":
        return s.give(out=e.linear(i["x"], i["w"], True, i.get("bias", 0), i.get("residual", 0)))
    if kind == "rows":
        op, x = c["op"], i["x"]
        if op in ("softmax", "log_softmax"):
            return s.give(out=e.softmax_rows(x, log=op == "log_softmax"))
        if op == "layer_norm":
            return s.give(out=e.layer_norm(x, i["g"], i["b"], EPS))
        if op == "rms_norm":
            return s.give(out=e.rms_norm(x, i["g"], EPS))
        if op == "row_sum":
            return s.give(out=e.reduce(x, miburn.R_SUM, miburn.AXIS_COLS))
        if op == "col_sum":
            return s.give(out=e.reduce(x, miburn.R_SUM, miburn.AXIS_ROWS))
        return s.give(out=e.eltwise_op_as(op.upper(), x, i.get("y", 0)))
    n = e.layer_norm(i["x"], i["g"], i["b"], EPS)
    z = e.linear(n, i["w"], False, i["bias"])
    logp, dz = e.log_softmax_ce(z, i["y"], 1.0 / c["rows"])
    dw = e.matmul_dram(n, True, dz, False)
    dbias = e.reduce(dz, miburn.R_SUM, miburn.AXIS_ROWS)
    dn = e.matmul_dram(dz, False, i["w"], True)
    dx, dg, db = e.layer_norm_backward(i["x"], i["g"], dn, 0, EPS)
    for t in (n, z, dz, dn):
        e.free(t)
    return s.give(logp=logp, dw=dw, dbias=dbias, dx=dx, dg=dg, db=db)


# ------------------------------------------------------------ work, tolerance


def work(case):
    c, kind = case, case["kind"]
    if kind == "mlp":
        params = c["d_in"] * c["hidden"] + c["hidden"] + c["hidden"] * c["d_out"] + c["d_out"]
        macs = c["batch"] * (2 * c["d_in"] * c["hidden"] + 3 * c["hidden"] * c["d_out"])
        return dict(bytes=4 * (2 * params + c["batch"] * (c["d_in"] + 1)), flops=2 * macs)
    if kind == "transformer":
        rows, d = c["batch"] * c["seq"], c["d"]
        layer = 4 * d * d + 2 * d * c["ff"]
        macs = rows * (c["layers"] * (layer + 2 * c["seq"] * d) + d * c["vocab"])
        params = c["layers"] * (layer + 9 * d + c["ff"]) + (d + 1) * c["vocab"]
        return dict(bytes=8 * (params + min(rows, c["vocab"]) * d), flops=6 * macs)
    if kind == "prefill":
        m, rows = miburn.SMOLLM2_135M, c["batch"] * c["t"]
        layer = (m["heads"] + 2 * m["kv_heads"]) * 64 * m["hidden"] + m["hidden"] ** 2 + 3 * m["intermediate"] * m["hidden"]
        head = m["vocab"] * m["hidden"]
        attn = 2 * rows * (c["t"] + 1) * 64 * m["heads"] * m["layers"]
        cache = 4 if c["numerics"] == "reference" else 2
        return dict(bytes=2 * (m["layers"] * layer + head) + cache * 2 * rows * m["layers"] * m["kv_heads"] * 64
                    + 4 * c["batch"] * m["vocab"],
                    flops=2 * rows * m["layers"] * layer + attn + 2 * c["batch"] * head)
    if kind == "decode":
        w, b = LAYERS[c["shape"]], c["batch"]
        weights = (2 * w["heads"] + 2 * w["kv"]) * w["d"] * w["hidden"] + 3 * w["inter"] * w["hidden"]
        kv = 2 * b * w["kv"] * c["ctx"] * w["d"]
        return dict(bytes=weights * (2 if c["weights"] == "bf16" else 17 / 16) + kv * (4 if c["cache"] == "f32" else 2)
                    + 12 * b * w["hidden"],
                    flops=2 * b * weights + 4 * b * w["heads"] * w["d"] * (c["ctx"] + 1))
    if kind == "attention":
        b, t, ctx = c["batch"], c["t"], c["pos0"] + c["t"]
        pairs = b * c["heads"] * (t * c["pos0"] + t * (t + 1) // 2)
        return dict(bytes=8 * b * t * c["heads"] * c["d"] + 2 * b * c["kv"] * ctx * c["d"] * (4 if c["cache"] == "f32" else 2),
                    flops=4 * pairs * c["d"])
    if kind in ("matmul", "batched"):
        m, n, k, b = c["m"], c["n"], c["k"], c.get("batch", 1)
        return dict(bytes=b * ((m * k + k * n) * (2 if c["dtype"] == "bf16" else 4)
                               + m * n * (2 if c.get("out") == "bf16" else 4)), flops=2 * b * m * n * k)
    if kind == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=4 * m * k + 2 * n * k + 4 * m * n * (2 if c["residual"] else 1), flops=2 * m * n * k)
    if kind == "rows":
        n = c["rows"] * c["cols"]
        out = c["rows"] if c["op"] == "row_sum" else c["cols"] if c["op"] == "col_sum" else n
        return dict(bytes=4 * (n * (2 if c["op"] == "add" else 1) + out), flops=0)
    rows, d, v = c["rows"], c["d"], c["vocab"]
    return dict(bytes=4 * (2 * rows * d + 2 * d * v + v + 2 * rows), flops=6 * rows * d * v)


def tolerance(case):
    """About four times the distance from `exact` that the engine shows, which
    is what F32 sums in another order, or a BF16 rounding that falls the other
    way, give; `max` is 40 times `rel` where it is not said."""
    kind = case["kind"]
    if kind in ("matmul", "batched") and case.get("out") == "bf16":
        return {"rel": 3e-3, "max": 2e-2}  # one rounding to 8 bits
    if kind in ("matmul", "batched"):
        # From 2^33 multiply-adds an F32 operand is taken as two BF16 parts
        # (2^-18 a product); below that, and for BF16 operands, F32 sums.
        macs = case["m"] * case["n"] * case["k"] * case.get("batch", 1)
        return {"rel": 2e-5 if case["dtype"] == "f32" and macs >= 1 << 33 else 3e-6}
    if kind == "linear":  # F32 activations as two BF16 parts
        return {"rel": 2e-5}
    if kind == "prefill":  # 30 layers on two BF16 parts, or on BF16 operands
        return {"rel": 3e-5 if case["numerics"] == "reference" else 1e-2}
    if kind == "decode":  # a BF16 cache's new row is rounded once
        return {"rel": 1e-6, "max": 1e-4} if case["cache"] == "f32" else {"rel": 2e-4, "max": 2e-2}
    return {"rel": {"mlp": 1e-6, "transformer": 5e-6, "lm_head": 5e-6}.get(kind, 2e-6)}


# ------------------------------------------------------------------ 64 bits


def _rms(x, g):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * g


def _layer_norm(x, g, b):
    mu = x.mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + EPS) * g + b


def _rope(x, cos, sin):
    """x [..., positions, heads, d] at the tables' rows [positions, d]."""
    half = x.shape[-1] // 2
    return x * cos[:, None, :] + torch.cat([x[..., half:], x[..., :half]], -1) * sin[:, None, :]


def _attend(q, k, v, pos0):
    """q [b, t, heads, d] against caches k, v [b, kv, ctx, d], causal from pos0."""
    b, t, heads, d = q.shape
    group = heads // k.shape[1]
    out = torch.empty_like(q)
    hidden = torch.arange(k.shape[2], device=q.device)[None, :] > pos0 + torch.arange(t, device=q.device)[:, None]
    for j in range(b):
        for h in range(heads):
            s = (q[j, :, h] @ k[j, h // group].T.contiguous()) * d ** -0.5
            out[j, :, h] = torch.softmax(s.masked_fill(hidden, -math.inf), -1) @ v[j, h // group]
    return out


def _exact_mlp(case, seed, inp):
    m = _model(case, seed)
    p = [torch.from_numpy(m.param(i)).cuda().double().requires_grad_() for i in range(4)]
    m.close()
    z = torch.relu(inp["x"].double() @ p[0] + p[1]) @ p[2] + p[3]
    loss = torch.nn.functional.cross_entropy(z, inp["y"].long().reshape(-1))
    loss.backward()
    out = {n: (t - MLP_LR * t.grad).detach() for n, t in zip(("w1", "b1", "w2", "b2"), p)}
    return dict(out, loss=loss.detach().reshape(1, 1))


def _exact_transformer(case, seed, inp):
    m = _model(case, seed)
    top = {n: torch.from_numpy(m.param(n)).cuda().double().requires_grad_() for n in ("embed", "head_w", "head_b")}
    layers = [{n: torch.from_numpy(m.param(n, i)).cuda().double().requires_grad_()
               for n in miburn.TRANSFORMER_LAYER_PARAMS} for i in range(case["layers"])]
    m.close()
    b, s, d, heads = case["batch"], case["seq"], case["d"], case["heads"]

    def split(t):
        return t.reshape(b, s, heads, d // heads).transpose(1, 2).contiguous()
    x = top["embed"][inp["tokens"].long().reshape(-1)]
    for p in layers:
        n1 = _layer_norm(x, p["ln1_g"], p["ln1_b"])
        q, k, v = (split(n1 @ p[w] + p[c]) for w, c in (("wq", "bq"), ("wk", "bk"), ("wv", "bv")))
        a = torch.softmax(q @ k.transpose(-1, -2).contiguous() * (d // heads) ** -0.5, -1) @ v
        x = x + a.transpose(1, 2).reshape(b * s, d) @ p["wo"] + p["bo"]
        n2 = _layer_norm(x, p["ln2_g"], p["ln2_b"])
        x = x + torch.nn.functional.gelu(n2 @ p["w1"] + p["b1"]) @ p["w2"] + p["b2"]
    loss = torch.nn.functional.cross_entropy(x @ top["head_w"] + top["head_b"], inp["targets"].long().reshape(-1))
    loss.backward()
    out = {n: (t - TRANSFORMER_LR * t.grad).detach() for n, t in top.items()}
    for n in miburn.TRANSFORMER_LAYER_PARAMS:
        out[n] = torch.stack([(p[n] - TRANSFORMER_LR * p[n].grad).detach() for p in layers])
    return dict(out, loss=loss.detach().reshape(1, 1))


def _exact_prefill(case, seed, inp):
    if case["numerics"] != "reference":
        return None  # its roundings to BF16 are part of what it computes
    m, cfg, b, t = _model(case, seed), miburn.SMOLLM2_135M, case["batch"], case["t"]
    heads, kv, d = cfg["heads"], cfg["kv_heads"], cfg["head_dim"]

    def weight(name, layer=0):
        id_ = m.param(name, layer)
        host = m.eng.download(id_)
        m.eng.free(id_)
        if host.dtype == np.uint16:
            host = miburn.bf16_to_f32(host)
        return torch.from_numpy(host).cuda().double()
    cos, sin = (c.double() for c in _rope_tables(t, d))
    embed = weight("embed")
    x = embed[inp["ids"].long()]
    for layer in range(cfg["layers"]):
        n = _rms(x, weight("attn_norm", layer))
        q = _rope((n @ weight("wq", layer).T).reshape(b, t, heads, d), cos, sin)
        k = _rope((n @ weight("wk", layer).T).reshape(b, t, kv, d), cos, sin).transpose(1, 2).contiguous()
        v = (n @ weight("wv", layer).T).reshape(b, t, kv, d).transpose(1, 2).contiguous()
        x = x + _attend(q, k, v, 0).reshape(b, t, heads * d) @ weight("wo", layer).T
        n = _rms(x, weight("mlp_norm", layer))
        x = x + (torch.nn.functional.silu(n @ weight("wgate", layer).T) * (n @ weight("wup", layer).T)) @ weight("wdown", layer).T
    logits = _rms(x[:, -1], weight("final_norm")) @ embed.T
    m.close()
    return dict(logits=logits)


def _exact_decode(case, inp):
    w, b, ctx = LAYERS[case["shape"]], case["batch"], case["ctx"]
    heads, kv, d, inter = w["heads"], w["kv"], w["d"], w["inter"]
    p = {n: t.double() for n, t in inp.items()}
    if case["weights"] == "bfp8":  # the weights as the engine stores them
        eng = _engine()
        for n in ("wqkv", "wo", "wgu", "wdown"):
            bf = eng.upload(inp[n].float().cpu().numpy())
            q = eng.cast_bfp(bf)
            p[n] = torch.from_numpy(eng.download(q)).cuda().double()
            eng.free(bf)
            eng.free(q)
    qkv = _rms(p["x"], p["g1"]) @ p["wqkv"].T
    cos, sin = p["cos"][ctx:ctx + 1], p["sin"][ctx:ctx + 1]
    q = _rope(qkv[:, :heads * d].reshape(b, 1, heads, d), cos, sin)
    k_new = _rope(qkv[:, heads * d:(heads + kv) * d].reshape(b, 1, kv, d), cos, sin)[:, 0]
    v_new = qkv[:, (heads + kv) * d:].reshape(b, kv, d)
    k, v = (p[n].reshape(b, kv, -1, d).clone() for n in ("k", "v"))
    k[:, :, ctx], v[:, :, ctx] = k_new, v_new
    rounded = torch.bfloat16 if case["cache"] == "bf16" else torch.float64  # attention reads the stored row
    ka, va = k[:, :, :ctx + 1].clone(), v[:, :, :ctx + 1].clone()
    ka[:, :, ctx], va[:, :, ctx] = k_new.to(rounded).double(), v_new.to(rounded).double()
    attn = p["x"] + _attend(q, ka, va, ctx).reshape(b, heads * d) @ p["wo"].T
    gu = _rms(attn, p["g2"]) @ p["wgu"].T
    out = attn + (torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]) @ p["wdown"].T
    return dict(attn=attn, out=out, k=k.reshape(-1, d), v=v.reshape(-1, d))


def _exact_rows(op, p):
    x = p["x"]
    if op in ("softmax", "log_softmax"):
        return getattr(torch, op)(x, -1)
    if op == "layer_norm":
        return _layer_norm(x, p["g"], p["b"])
    if op == "rms_norm":
        return _rms(x, p["g"])
    if op == "add":
        return x + p["y"]
    if op == "row_sum":
        return x.sum(1, keepdim=True)
    if op == "col_sum":
        return x.sum(0, keepdim=True)
    return getattr(torch.nn.functional, op)(x)


def exact(case, seed):
    kind, inp = case["kind"], _inputs(case, seed)
    if kind == "mlp":
        return _exact_mlp(case, seed, inp)
    if kind == "transformer":
        return _exact_transformer(case, seed, inp)
    if kind == "prefill":
        return _exact_prefill(case, seed, inp)
    if kind == "decode":
        return _exact_decode(case, inp)
    p = {n: t.double() if t.is_floating_point() else t for n, t in inp.items()}
    if kind == "attention":
        b, t, d = case["batch"], case["t"], case["d"]
        k, v = (p[n].reshape(b, case["kv"], -1, d) for n in ("k", "v"))
        return dict(out=_attend(p["q"].reshape(b, t, -1, d), k, v, case["pos0"]).reshape(b * t, -1))
    if kind in ("matmul", "batched"):
        out, b = [], case.get("batch", 1)
        for x, y in zip(p["a"].chunk(b), p["b"].chunk(b)):
            out.append((x.T if case["ta"] else x) @ (y.T if case["tb"] else y))
        return dict(out=torch.cat(out))
    if kind == "linear":
        y = p["x"] @ p["w"].T
        if case["bias"]:
            y = y + p["bias"]
        return dict(out=y + p["residual"] if case["residual"] else y)
    if kind == "rows":
        return dict(out=_exact_rows(case["op"], p))
    x, g, b, w, bias = (p[n].requires_grad_() for n in ("x", "g", "b", "w", "bias"))
    logp = torch.log_softmax(_layer_norm(x, g, b) @ w + bias, -1).gather(1, p["y"].long())
    (-logp.mean()).backward()
    return dict(logp=logp.detach(), dw=w.grad, dbias=bias.grad, dx=x.grad, dg=g.grad, db=b.grad)
