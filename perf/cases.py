"""What this library is timed on: the calls that a training loop or a decoder
makes, through the public submit_* entry points (dataflow_lib_amd.api).

A case is a dict with a `kind` and the kind's sizes, storage type and options:

  decode    one decoding step's native ops for `tokens` sequences: RMSNorm,
            RoPE with the KV-cache scatter, SwiGLU
  prefill   the same block over a packed batch of prompts of uneven lengths,
            with the embedding gather in front
  norm      RMSNorm forward and backward (the fused exact gradient, or the
            split bwd_x / bwd_w pair)
  rope      RoPE forward on Q, K and backward on dQ, dK of packed sequences
  swiglu    SwiGLU forward and backward
  loss      fused softmax + cross-entropy of a batch of logits
  softmax   row softmax out of place (sampling and scoring); fp8 logits give
            16-bit probabilities
  fp8       a block with fp8 forward and 16-bit backward tensors: RMSNorm
            forward, bwd_x and bwd_w, RoPE, SwiGLU forward and backward
  head      submit_transformer_head: norm, output projection and softmax
            (inference) or the whole loss path with its gradients (training)

Buffers are torch tensors on the GPU, filled before the call; the ops run on
the handle's own stream 0.
"""
import math

import numpy as np
import torch

from dataflow_lib_amd import api

EPS = 1e-5
THETA = 500000
TYPES = {"fp32": (api.DATAFLOW_FP32, torch.float32, 4), "fp16": (api.DATAFLOW_FP16, torch.float16, 2),
         "bf16": (api.DATAFLOW_BF16, torch.bfloat16, 2), "fp8e4m3": (api.DATAFLOW_FP8E4M3, torch.float8_e4m3fn, 1),
         "fp8e5m2": (api.DATAFLOW_FP8E5M2, torch.float8_e5m2, 1)}

_handle = None


def handle():
    """The program's one handle: native ops and the matmul registered once."""
    global _handle
    if _handle is None:
        torch.zeros(1, device="cuda")
        _handle = api.Handle(0, num_streams=2, matmul=True)
    return _handle


def listed():
    return [
        # one decoding step of a small serving batch, Llama-3-8B sizes: three short launches
        dict(name="decode_8", kind="decode", tokens=8, hidden=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, context=512, dtype="bf16"),
        # a packed prompt batch that is no multiple of anything
        dict(name="prefill_1531", kind="prefill", tokens=1531, hidden=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, vocab=32000, dtype="bf16"),
        # the training norm of Llama-3-8B at 8192 tokens
        dict(name="norm_8192x4096", kind="norm", rows=8192, cols=4096, dtype="bf16", split=False),
        # a small model trained in fp32, with the separate dX and dW ops
        dict(name="norm_split_3000x1000_fp32", kind="norm", rows=3000, cols=1000, dtype="fp32", split=True),
        # rotary embedding of a small model with as many K as Q heads, fp16
        dict(name="rope_4099x16x64_fp16", kind="rope", tokens=4099, heads=16, kv_heads=16, head_dim=64, dtype="fp16"),
        # the training MLP of Llama-3-8B at 8192 tokens
        dict(name="swiglu_8192x14336", kind="swiglu", rows=8192, cols=14336, dtype="bf16"),
        # the training loss at the Llama-3 vocabulary (the largest case)
        dict(name="loss_4096x128256", kind="loss", rows=4096, vocab=128256, dtype="bf16"),
        # a vocabulary that is odd, as byte-pair vocabularies often are: rows are not 16-byte aligned
        dict(name="loss_1024x50257", kind="loss", rows=1024, vocab=50257, dtype="bf16"),
        # a vocabulary whose rows exceed the register-row limit
        dict(name="loss_1024x151936", kind="loss", rows=1024, vocab=151936, dtype="bf16"),
        # next-token probabilities of a serving batch
        dict(name="sample_16x128256", kind="softmax", rows=16, vocab=128256, dtype="bf16"),
        # an fp8 training block of 2048 tokens
        dict(name="fp8_2048", kind="fp8", tokens=2048, hidden=4096, heads=32, kv_heads=8, head_dim=128, ffn=14336, dtype="fp8e4m3", grad="bf16"),
        # the whole loss path with its gradients
        dict(name="head_train_1024", kind="head", tokens=1024, hidden=2048, vocab=32000, dtype="bf16", train=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng):
    """a vocabulary size: half of them odd, half a multiple of 8"""
    v = _log(rng, 1000, 200000)
    return v | 1 if rng.random() < 0.5 else v & ~7


def _block(rng):
    """the sizes of a transformer block"""
    hidden = rng.choice([1024, 2048, 3072, 4096, 5120, 8192])
    head_dim = 64 if hidden <= 1024 else 128
    heads = hidden // head_dim
    return dict(hidden=hidden, heads=heads, kv_heads=heads // rng.choice([1, 2, 4, 8]), head_dim=head_dim,
                ffn=8 * int(rng.uniform(2.6, 4.0) * hidden / 8))


def draw(rng):
    """One more case of the same ranges; its bytes are at most the largest
    listed case's, and a quarter of those where rows are unaligned."""
    while True:
        kind = rng.choice(["decode", "prefill", "norm", "rope", "swiglu", "loss", "loss", "softmax", "softmax", "fp8", "head"])
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        if kind == "decode":
            c = dict(tokens=_log(rng, 1, 64), context=_log(rng, 64, 512), dtype=dtype, **_block(rng))
        elif kind == "prefill":
            c = dict(tokens=_log(rng, 65, 8192), vocab=32000, dtype=dtype, **_block(rng))
        elif kind == "norm":
            c = dict(rows=_log(rng, 16, 16384), cols=8 * _log(rng, 64, 1024), dtype=dtype, split=rng.random() < 0.5)
        elif kind == "rope":
            head_dim = rng.choice([64, 96, 128, 128, 256])
            heads = rng.choice([8, 16, 24, 32, 40, 64])
            c = dict(tokens=_log(rng, 16, 16384), heads=heads, kv_heads=heads // rng.choice([1, 2, 4, 8]), head_dim=head_dim, dtype=dtype)
        elif kind == "swiglu":
            c = dict(rows=_log(rng, 1, 8192), cols=_log(rng, 1000, 28672), dtype=dtype)
        elif kind == "loss":
            c = dict(rows=_log(rng, 16, 8192), vocab=_vocab(rng), dtype=dtype)
        elif kind == "softmax":
            c = dict(rows=_log(rng, 1, 2048), vocab=_vocab(rng), dtype=rng.choice([dtype, dtype, "fp8e4m3"]))
        elif kind == "fp8":
            c = dict(tokens=_log(rng, 64, 8192), dtype=rng.choice(["fp8e4m3", "fp8e5m2"]), grad=rng.choice(["bf16", "fp16"]), **_block(rng))
        else:
            train = rng.random() < 0.5
            c = dict(tokens=_log(rng, 64, 1024) if train else _log(rng, 1, 64), hidden=rng.choice([1024, 2048, 4096]),
                     vocab=8 * _log(rng, 500, 6000), dtype=rng.choice(["bf16", "fp16"]), train=train)
        c = dict(kind=kind, **c)
        odd = c.get("vocab", 0) % 8 or c.get("cols", 0) % 8
        if work(c)["bytes"] <= 2.1e9 / (4 if odd else 1) and work(c)["flops"] <= 4.5e11:
            return c


# ---------------- inputs ----------------

class _Maker:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, shape, dtype, mean=0.0, std=1.0):
        t = torch.empty(shape, dtype=torch.float32 if TYPES[dtype][2] == 1 else TYPES[dtype][1], device="cuda")
        return t.normal_(mean, std, generator=self.g).to(TYPES[dtype][1])

    def ints(self, shape, high):
        return torch.randint(0, high, shape, generator=self.g, device="cuda", dtype=torch.int32)

    def logits(self, rows, vocab, dtype):
        """logits of a part-trained model: the row's spread is 2.5, its offset varies"""
        x = self.normal((rows, vocab), dtype, std=2.5)
        if TYPES[dtype][2] > 1:
            x += self.normal((rows, 1), dtype, std=2.0)
        return x


def _lengths(tokens):
    """uneven prompt lengths that add up to `tokens`"""
    out, n, k = [], tokens, 0
    while n > 0:
        take = min(n, (37, 512, 129, 1000, 2048, 301)[k % 6])
        out.append(take)
        n -= take
        k += 1
    return out


def _packed_positions(tokens):
    return torch.cat([torch.arange(n, dtype=torch.int32) for n in _lengths(tokens)]).cuda()


def _data(case, seed):
    """The tensors that a program has before the call, by name."""
    m, k, dt = _Maker(seed), case["kind"], case["dtype"]
    d = {}
    if k in ("decode", "prefill", "fp8"):
        t, h, kv, f = case["tokens"], case["hidden"], case["kv_heads"] * case["head_dim"], case["ffn"]
        d["x"], d["w"] = m.normal((t, h), dt), m.normal((h,), dt, 1.0, 0.1)
        d["q"], d["k"] = m.normal((t, h), dt), m.normal((t, kv), dt)
        d["gate"], d["up"] = m.normal((t, f), dt, std=2.0), m.normal((t, f), dt)
        if k == "prefill":
            d["table"], d["ids"] = m.normal((case["vocab"], h), dt), m.ints((t,), case["vocab"])
        if k == "fp8":
            g = case["grad"]
            d["pos"] = _packed_positions(t)
            d["dy"], d["dx"] = m.normal((t, h), g), m.normal((t, h), g)
            d["dw"], d["dout"] = m.normal((h,), g), m.normal((t, f), g)
            x = d["x"].double()
            d["rstd"] = torch.rsqrt(x.square().mean(1) + EPS).float()
            d["wsum"] = (x * d["w"].double()).sum(1).float()
        else:
            d["v"] = m.normal((t, kv), dt)
            if k == "decode":
                sizes = torch.full((t,), case["context"], dtype=torch.int32)
                d["pos"] = m.ints((t,), case["context"])
                first = torch.arange(t, dtype=torch.int64) * 2 * case["context"]
            else:
                lens = _lengths(t)
                sizes = torch.cat([torch.full((n,), n, dtype=torch.int32) for n in lens])
                d["pos"] = _packed_positions(t)
                first = torch.cat([torch.full((n,), 2 * sum(lens[:i]), dtype=torch.int64) for i, n in enumerate(lens)])
            rows = 2 * (t * case["context"] if k == "decode" else t)
            d["cache"] = torch.zeros((rows, kv), dtype=TYPES[dt][1], device="cuda")
            d["ctx_size"], d["ctx_row"] = sizes.cuda(), first.cuda()
    elif k == "norm":
        r, c = case["rows"], case["cols"]
        d["x"], d["w"], d["dy"] = m.normal((r, c), dt), m.normal((c,), dt, 1.0, 0.1), m.normal((r, c), dt)
        d["dx"], d["dw"] = m.normal((r, c), dt), m.normal((c,), dt if case["split"] else "fp32")
    elif k == "rope":
        t, qd, kd = case["tokens"], case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
        d["pos"] = _packed_positions(t)
        for n, w in (("q", qd), ("k", kd), ("dq", qd), ("dk", kd)):
            d[n] = m.normal((t, w), dt)
    elif k == "swiglu":
        s = (case["rows"], case["cols"])
        d["gate"], d["up"], d["dout"] = m.normal(s, dt, std=2.0), m.normal(s, dt), m.normal(s, dt)
    elif k == "loss":
        d["logits"], d["labels"] = m.logits(case["rows"], case["vocab"], dt), m.ints((case["rows"],), case["vocab"])
    elif k == "softmax":
        d["logits"] = m.logits(case["rows"], case["vocab"], dt)
    else:
        t, h, v = case["tokens"], case["hidden"], case["vocab"]
        d["x"], d["w"] = m.normal((t, h), dt), m.normal((h,), dt, 1.0, 0.1)
        d["w_head"] = m.normal((v, h), dt, std=2.0 * h ** -0.5)
        if case["train"]:
            d["labels"] = m.ints((t,), v)
            d["dw_head"], d["dw"], d["dx"] = m.normal((v, h), dt, std=0.01), m.normal((h,), "fp32", std=0.01), m.normal((t, h), dt, std=0.01)
    return d


def prepare(case, seed):
    hd, k = handle(), case["kind"]
    d = _data(case, seed)
    dt, tt, _ = TYPES[case["dtype"]]
    new = lambda shape, t=tt: torch.empty(shape, dtype=t, device="cuda")  # noqa: E731
    f32 = torch.float32
    p = lambda n: d[n].data_ptr()  # noqa: E731
    calls, outs = [], []

    def call(f, *args):
        calls.append((f, (hd, 0) + args))

    if k in ("decode", "prefill", "norm"):
        r, c = d["x"].shape
        d["y"], d["ws"], d["rs"] = new((r, c)), new((r,), f32), new((r,), f32)
        if k == "prefill":
            call(api.submit_embedding, dt, r, c, p("ids"), p("table"), p("x"))
            outs.append("x")
        call(api.submit_rms_norm, dt, r, c, EPS, p("w"), p("x"), p("y"), p("ws"), p("rs"))
        outs += ["y", "ws", "rs"]
    if k in ("decode", "prefill"):
        kv = case["kv_heads"] * case["head_dim"]
        d["ctx"] = d["cache"].data_ptr() + d["ctx_row"] * (kv * d["cache"].element_size())
        call(api.submit_rope_copy_to_seq_context, dt, r * c, c, case["head_dim"], case["kv_heads"], THETA, p("pos"), p("q"), p("k"), p("v"),
             p("ctx"), p("ctx_size"))
        d["act"] = new((r, case["ffn"]))
        call(api.submit_swiglu, dt, r, case["ffn"], p("gate"), p("up"), p("act"))
        outs += ["q", "k", "cache", "act"]
    elif k == "norm":
        if case["split"]:
            call(api.submit_rms_norm_bwd_x, dt, dt, r, c, EPS, p("ws"), p("rs"), p("w"), p("x"), p("dy"), p("dx"))
            call(api.submit_rms_norm_bwd_w, dt, dt, r, c, EPS, p("rs"), p("x"), p("dy"), p("dw"))
        else:
            call(api.submit_rms_norm_bwd, dt, dt, r, c, EPS, p("rs"), p("w"), p("x"), p("dy"), p("dx"), p("dw"))
        outs += ["dx", "dw"]
    elif k == "rope":
        t, qd = d["q"].shape
        call(api.submit_rope, dt, t * qd, qd, case["head_dim"], case["kv_heads"], THETA, p("pos"), p("q"), p("k"))
        call(api.submit_rope_bwd_x, dt, t * qd, qd, case["head_dim"], case["kv_heads"], THETA, p("pos"), p("dq"), p("dk"))
        outs = ["q", "k", "dq", "dk"]
    elif k == "swiglu":
        r, c = d["gate"].shape
        d["act"], d["dgate"], d["dup"] = new((r, c)), new((r, c)), new((r, c))
        call(api.submit_swiglu, dt, r, c, p("gate"), p("up"), p("act"))
        call(api.submit_swiglu_bwd_x, dt, dt, r, c, p("gate"), p("up"), p("dout"), p("dgate"), p("dup"))
        outs = ["act", "dgate", "dup"]
    elif k == "loss":
        r, c = d["logits"].shape
        d["loss"], d["mean"] = new((r,), f32), new((1,), f32)
        call(api.submit_softmax_cross_entropy_loss, dt, r, c, p("logits"), p("labels"), p("loss"), p("mean"))
        outs = ["logits", "loss", "mean"]
    elif k == "softmax":
        r, c = d["logits"].shape
        ot = "bf16" if case["dtype"].startswith("fp8") else case["dtype"]
        d["probs"] = new((r, c), TYPES[ot][1])
        call(api.submit_softmax, dt, TYPES[ot][0], r, c, p("logits"), p("probs"))
        outs = ["probs"]
    elif k == "fp8":
        gt = TYPES[case["grad"]][0]
        r, c = d["x"].shape
        d["y"], d["ss"], d["act"] = new((r, c)), new((r,), f32), new((r, case["ffn"]))
        d["dgate"], d["dup"] = torch.empty_like(d["dout"]), torch.empty_like(d["dout"])
        call(api.submit_rms_norm, dt, r, c, EPS, p("w"), p("x"), p("y"), None, p("ss"))
        call(api.submit_rope, dt, r * c, c, case["head_dim"], case["kv_heads"], THETA, p("pos"), p("q"), p("k"))
        call(api.submit_swiglu, dt, r, case["ffn"], p("gate"), p("up"), p("act"))
        call(api.submit_swiglu_bwd_x, dt, gt, r, case["ffn"], p("gate"), p("up"), p("dout"), p("dgate"), p("dup"))
        call(api.submit_rms_norm_bwd_x, dt, gt, r, c, EPS, p("wsum"), p("rstd"), p("w"), p("x"), p("dy"), p("dx"))
        call(api.submit_rms_norm_bwd_w, dt, gt, r, c, EPS, p("rstd"), p("x"), p("dy"), p("dw"))
        outs = ["y", "ss", "q", "k", "act", "dgate", "dup", "dx", "dw"]
    else:
        t, h = d["x"].shape
        v, F32 = case["vocab"], api.DATAFLOW_FP32
        d["norm"], d["ws"], d["rs"], d["out"] = new((t, h)), new((t,), f32), new((t,), f32), new((t, v))
        d["space"] = torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
        cfg = api.EmbeddingConfig(v, h)
        head = api.TransformerHead(dt, dt, F32, EPS, cfg, None, p("w"), p("w_head"))
        acts = api.TransformerHeadActivations(t, None, p("norm"), p("ws"), p("rs"), p("out"), p("space"), 32 << 20)
        block = api.TransformerBlockTransition(None, p("x"))
        if case["train"]:
            d["loss"], d["dnorm"] = new((t + 1,), f32), new((t, h))
            mo = api.TransformerModelOutput(None, None, p("labels"), None, p("loss"), 0.0)
            ghead = api.TransformerHead(dt, dt, F32, EPS, cfg, None, p("dw"), p("dw_head"))
            gacts = api.TransformerHeadActivations(t, None, p("dnorm"), None, None, None, p("space"), 32 << 20)
            calls.append((api.submit_transformer_head, (hd, 0, 0, block, head, acts, mo, ghead, gacts, api.TransformerBlockTransition(None, p("dx")), None)))
            outs = ["norm", "out", "loss", "dnorm", "dw_head", "dw", "dx"]
        else:
            d["probs"] = new((t, v))
            mo = api.TransformerModelOutput(None, None, None, p("probs"), None, 0.0)
            calls.append((api.submit_transformer_head, (hd, 0, 0, block, head, acts, mo)))
            outs = ["norm", "out", "probs"]
    # the ops run on the handle's non-blocking stream, which does not wait for torch's
    torch.cuda.synchronize()
    return {"calls": calls, "outputs": {n: d[n] for n in outs}, "data": d}


def run(state):
    for f, args in state["calls"]:
        if f(*args) != 0:
            raise RuntimeError("%s failed" % f.__name__)
    return state["outputs"]


# ---------------- what a pass cannot do without ----------------

def work(case):
    k, e = case["kind"], TYPES[case["dtype"]][2]
    if k in ("decode", "prefill", "fp8"):
        t, h, kv, f = case["tokens"], case["hidden"], case["kv_heads"] * case["head_dim"], case["ffn"]
        if k == "fp8":
            g = TYPES[case["grad"]][2]
            n = 2 * t * h * e + 2 * t * (h + kv) * e + 3 * t * f * e + t * f * (2 * e + 3 * g)      # norm, rope, swiglu, its backward
            n += t * h * (e + 3 * g) + t * h * (e + g)                                              # bwd_x (dX read and written), bwd_w
            return {"bytes": n + 20 * t + 4 * h, "flops": t * (14 * h + 6 * (h + kv) + 24 * f)}
        n = 2 * t * h * e + 2 * t * (h + kv) * e + 3 * t * kv * e + 3 * t * f * e                   # norm, rope, cache rows (V read, K and V written), swiglu
        if k == "prefill":
            n += 2 * t * h * e
        return {"bytes": n + 24 * t + h * e, "flops": t * (6 * h + 6 * (h + kv) + 8 * f)}
    if k == "norm":
        r, c = case["rows"], case["cols"]
        n = 2 * r * c * e + 4 * r * c * e + (2 * r * c * e if case["split"] else 0)                 # forward; X, dY, dX, dX (bwd_w: X, dY again)
        return {"bytes": n + 16 * r + 6 * c * e, "flops": 16.0 * r * c}
    if k == "rope":
        n = case["tokens"] * (case["heads"] + case["kv_heads"]) * case["head_dim"]
        return {"bytes": 4 * n * e + 8 * case["tokens"], "flops": 6.0 * n}
    if k == "swiglu":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n * e, "flops": 20.0 * n}
    if k in ("loss", "softmax"):
        n = case["rows"] * case["vocab"]
        return {"bytes": (n * (e + max(e, 2)) if k == "softmax" else 2 * n * e + 8 * case["rows"]), "flops": 8.0 * n}
    t, h, v = case["tokens"], case["hidden"], case["vocab"]
    g = 2.0 * t * h * v
    if not case["train"]:
        return {"bytes": e * (2 * t * h + v * h + 2 * t * v), "flops": g}
    return {"bytes": e * (6 * t * h + 3 * v * h + t * v), "flops": 3 * g}


# ---------------- how exact, and against what ----------------

# Relative 2-norm and largest difference between two correct programs at one
# precision: sums in another order, so a stored value may be its neighbour.
# Against exact() the outputs are off by 1.7e-3 (bf16), 2.1e-4 (fp16), 2e-7
# (fp32) and 2.5e-2 (fp8e4m3), which is the rounding of the stored value.
_TOL = {"fp32": {"rel": 4e-6, "max": 4e-5}, "fp16": {"rel": 5e-4, "max": 4e-3}, "bf16": {"rel": 4e-3, "max": 2e-2},
        "fp8e4m3": {"rel": 1e-2, "max": 0.15}, "fp8e5m2": {"rel": 2e-2, "max": 0.3}}


def tolerance(case):
    if case["kind"] == "head":   # logits rounded to 16 bits pass through the loss and two products
        return {"rel": 8e-3, "max": 0.1}
    if case["kind"] == "softmax" and case["dtype"].startswith("fp8"):
        return dict(_TOL["bf16"])
    return dict(_TOL[case["dtype"]])


def _rope_exact(x, pos, head_dim, sign):
    """pairs (2p, 2p + 1) of each head turned by fl32(pos * angle_p), angle_p in fp32 as the op defines it"""
    t, half = x.shape[0], head_dim // 2
    expo = [-(np.float32(2 * p) / np.float32(head_dim)) for p in range(half)]
    ang = torch.tensor([float(np.float32(float(THETA) ** float(e))) for e in expo], dtype=torch.float32, device="cuda")
    arg = (pos.float()[:, None] * ang[None, :]).double()
    c, s = torch.cos(arg)[:, None, :], sign * torch.sin(arg)[:, None, :]
    v = x.double().view(t, -1, half, 2)
    return torch.stack((c * v[..., 0] - s * v[..., 1], c * v[..., 1] + s * v[..., 0]), -1).view(t, -1)


def _softmax_exact(x, diff_dtype):
    """softmax with x - max rounded to the storage type, as the op defines it, a few rows at a time"""
    y = torch.empty(x.shape, dtype=torch.float64, device="cuda")
    loss_sum = torch.empty(x.shape[0], dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // x.shape[1])
    for i in range(0, x.shape[0], step):
        v = x[i:i + step].double()
        v = v - v.amax(1, keepdim=True)
        loss_sum[i:i + step] = torch.logsumexp(v, 1)
        e = torch.exp(v.to(diff_dtype).double())
        y[i:i + step] = e / e.sum(1, keepdim=True)
    return y, loss_sum


def _norm_exact(x, w):
    x, w = x.double(), w.double()
    r = torch.rsqrt(x.square().mean(1) + EPS)
    return x * r[:, None] * w, (x * w).sum(1), r


def _norm_bwd_exact(x, w, dy, r):
    x, g = x.double(), dy.double() * w.double()
    return r[:, None] * g - x * (r ** 3 * (g * x).mean(1))[:, None]


def _bwd_x_exact(x, w, dy, r, ws):
    return dy.double() * (w.double() * r[:, None] - x.double() * (r ** 3 * ws / x.shape[1])[:, None])


def _swiglu_exact(d):
    g, u = d["gate"].double(), d["up"].double()
    s = torch.sigmoid(g)
    out = {"act": g * s * u}
    if "dout" in d:
        do = d["dout"].double()
        out["dgate"], out["dup"] = do * u * s * (1 + g * (1 - s)), do * g * s
    return out


def exact(case, seed):
    k, d = case["kind"], _data(case, seed)
    if k in ("decode", "prefill"):
        o = {}
        x = d["x"]
        if k == "prefill":
            o["x"] = x = d["table"][d["ids"].long()]
        y, ws, r = _norm_exact(x, d["w"])
        o.update(y=y, ws=ws, rs=r, q=_rope_exact(d["q"], d["pos"], case["head_dim"], 1.0), k=_rope_exact(d["k"], d["pos"], case["head_dim"], 1.0))
        o["cache"] = d["cache"].double()
        at = d["ctx_row"] + d["pos"].long()
        o["cache"][at] = o["k"]
        o["cache"][at + d["ctx_size"].long()] = d["v"].double()
        o.update(_swiglu_exact(d))
        return o
    if k == "norm":
        y, ws, r = _norm_exact(d["x"], d["w"])
        bwd = _bwd_x_exact(d["x"], d["w"], d["dy"], r, ws) if case["split"] else _norm_bwd_exact(d["x"], d["w"], d["dy"], r)
        dw = d["dw"].double() + (d["dy"].double() * d["x"].double() * r[:, None]).sum(0)
        return {"y": y, "ws": ws, "rs": r, "dx": d["dx"].double() + bwd, "dw": dw}
    if k == "rope":
        f = lambda n, s: _rope_exact(d[n], d["pos"], case["head_dim"], s)  # noqa: E731
        return {"q": f("q", 1.0), "k": f("k", 1.0), "dq": f("dq", -1.0), "dk": f("dk", -1.0)}
    if k == "swiglu":
        return _swiglu_exact(d)
    if k == "loss":
        x, lab = d["logits"], d["labels"].long()
        y, lse = _softmax_exact(x, x.dtype)
        at = torch.arange(x.shape[0], device="cuda")
        y[at, lab] -= 1.0
        loss = lse + x.amax(1).double() - x[at, lab].double()
        return {"logits": y, "loss": loss, "mean": loss.mean().view(1)}
    if k == "softmax":
        return {"probs": _softmax_exact(d["logits"], torch.bfloat16 if case["dtype"].startswith("fp8") else d["logits"].dtype)[0]}
    if k == "fp8":
        x = d["x"].double()
        y, _, _ = _norm_exact(d["x"], d["w"])
        r = d["rstd"].double()
        o = {"y": y, "ss": x.square().sum(1)}
        o["q"], o["k"] = _rope_exact(d["q"].float(), d["pos"], case["head_dim"], 1.0), _rope_exact(d["k"].float(), d["pos"], case["head_dim"], 1.0)
        o.update(_swiglu_exact(d))
        o["dx"] = d["dx"].double() + _bwd_x_exact(x, d["w"], d["dy"], r, d["wsum"].double())
        o["dw"] = d["dw"].double() + (d["dy"].double() * x * r[:, None]).sum(0)
        return o
    y, _, r = _norm_exact(d["x"], d["w"])
    w = d["w_head"].double()
    z = y @ w.T
    if not case["train"]:
        return {"norm": y, "out": z, "probs": torch.softmax(z, 1)}
    at, lab = torch.arange(z.shape[0], device="cuda"), d["labels"].long()
    loss = torch.logsumexp(z, 1) - z[at, lab]
    g = torch.softmax(z, 1)
    g[at, lab] -= 1.0
    dn = g @ w
    return {"norm": y, "out": g, "loss": torch.cat((loss, loss.mean().view(1))), "dnorm": dn, "dw_head": d["dw_head"].double() + g.T @ y,
            "dw": d["dw"].double() + (dn * d["x"].double() * r[:, None]).sum(0),
            "dx": d["dx"].double() + _norm_bwd_exact(d["x"], d["w"], dn, r)}
