"""Performance cases of the decode engine: what a program that uses it has it do, through its public entry points.

Kinds of a case
  attn      one decode attention (moert.attn_decode_noalloc) over fp16 K/V rows in the caller's device buffers
  block     one MoE block, one position (GpuBlock.forward): host vector in, host vector out
  batch     one MoE block, m positions at once (GpuBlock.forward_batched)
  decode    forced tokens one step at a time (GpuModel.step) after `ctx` cached positions, logits of every step;
            with `pool`, the experts are served from an HBM pool of that share of them over the pinned host store
  generate  a new sequence: prompt, then greedy tokens (GpuModel.generate), and the logits of the last one
  prefill   `n` tokens after `ctx` cached positions (GpuModel.prefill), logits and hidden state of the last one; for
            a new sequence also the last layer's K/V rows, which depend on every layer at every position, as a program
            that keeps a prompt's rows reads them; mode 1 runs the grouped integer products (GpuModel.batched_mode)

Shapes are the two Granite ones of the package (moert.GRANITE_1B / GRANITE_3B: "1b", "3b"). Layers are independent of
each other in cost, so that the prefill and pool cases take a few of them; weights are random, of the package's own
synthetic models, and each case's exceed the last-level cache as a whole model's do, where weights are streamed.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "lastro-rust_amd"))
import moert  # noqa: E402

SHAPES = {"1b": moert.GRANITE_1B, "3b": moert.GRANITE_3B}
DTYPES = {"q8_0": moert.Q8_0, "q4_0": moert.Q4_0, "f32": moert.F32}
STD = 0.02


def listed():
    return [
        # the attention of a short chat turn: launches and latency only
        dict(name="attn_short_1b", kind="attn", shape="1b", ctx=100, max_len=512, splits=8),
        # the attention of a long document, a length that fills no tile
        dict(name="attn_long_3b", kind="attn", shape="3b", ctx=16001, max_len=16384, splits=64),
        # the smallest unit of work of a program that runs blocks itself: one token's experts
        dict(name="block_1b", kind="block", shape="1b", dtype="q8_0"),
        # sixteen sequences decoding together, skewed expert loads: the batch of the package's benchmark
        dict(name="batch16_3b", kind="batch", shape="3b", m=16, zipf=1.1),
        # a ragged batch near the limit of one step
        dict(name="batch29_1b", kind="batch", shape="1b", m=29, zipf=0.0),
        # a short chat on the small model, f32 head as the decode benchmark has it
        dict(name="generate_1b", kind="generate", shape="1b", layers=24, dtype="q8_0", embed="f32", n=19, new=24),
        # decode of the large model after 4096 positions: the package's headline benchmark
        dict(name="decode_3b_4096", kind="decode", shape="3b", layers=32, dtype="q8_0", embed="q8_0", ctx=4096, n=4,
             splits=32, pool=0.0),
        # a model that does not fit its share of HBM: a quarter of the experts in the pool
        dict(name="decode_3b_pool", kind="decode", shape="3b", layers=8, dtype="q4_0", embed="q4_0", ctx=300, n=8,
             splits=32, pool=0.25),
        # a short question read at the start of a chat, 4-bit weights
        dict(name="prefill37_1b_q4", kind="prefill", shape="1b", layers=6, dtype="q4_0", embed="q4_0", ctx=0, n=37,
             splits=32, mode=0),
        # a page of text read at the start of a sequence
        dict(name="prefill512_3b", kind="prefill", shape="3b", layers=4, dtype="q8_0", embed="q8_0", ctx=0, n=512,
             splits=32, mode=0),
        # the next turn of a long chat
        dict(name="prefill70_3b_4096", kind="prefill", shape="3b", layers=4, dtype="q8_0", embed="q8_0", ctx=4096,
             n=70, splits=32, mode=0),
        # a page after retrieved text, through the integer products
        dict(name="prefill300_3b_grouped", kind="prefill", shape="3b", layers=4, dtype="q8_0", embed="q8_0", ctx=1000,
             n=300, splits=32, mode=1),
    ]


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    shape = rng.choice(["1b", "3b"])
    kind = rng.choice(["attn", "block", "batch", "generate", "decode", "prefill", "prefill", "prefill"])
    if kind == "attn":
        ctx = _log(rng, 1, 16384)
        return dict(kind=kind, shape=shape, ctx=ctx, max_len=64 * rng.randint(-(-ctx // 64), 256),
                    splits=rng.choice([8, 32, 64]))
    if kind == "block":
        return dict(kind=kind, shape=shape, dtype=rng.choice(["q8_0", "q4_0", "f32"]))
    if kind == "batch":
        return dict(kind=kind, shape=shape, m=rng.randint(1, 32), zipf=rng.choice([0.0, 1.1]))
    dtype = rng.choice(["q8_0", "q8_0", "q4_0"])
    embed = rng.choice([dtype, "f32"])
    layers = rng.randint(3, 8)
    if kind == "generate":
        return dict(kind=kind, shape=shape, layers=layers, dtype=dtype, embed=embed, n=_log(rng, 1, 64),
                    new=rng.randint(1, 32))
    if kind == "decode":
        return dict(kind=kind, shape=shape, layers=layers, dtype=dtype, embed=embed, ctx=_log(rng, 1, 6000),
                    n=rng.randint(1, 6), splits=rng.choice([8, 32, 64]), pool=rng.choice([0.0, 0.0, 0.25]))
    mode = 1 if dtype == "q8_0" and rng.random() < 0.4 else 0
    ctx = rng.choice([0, _log(rng, 1, 4096)])
    return dict(kind=kind, shape=shape, layers=rng.randint(3, 4), dtype=dtype, embed=embed, ctx=ctx,
                n=_log(rng, 1, 512 if ctx < 1024 else 200), splits=rng.choice([8, 32, 64]), mode=mode)


# ---- inputs ----------------------------------------------------------------------------------------------------
def _config(case):
    s = dict(SHAPES[case["shape"]])
    s["layers"] = case.get("layers", 1)
    return moert.Config(**s)


def _max_len(case):
    return -(-(case.get("ctx", 0) + case["n"] + case.get("new", 0) + 64) // 64) * 64


def _tokens(case, seed, vocab):
    return np.random.default_rng(seed + 7).integers(0, vocab, case["n"]).astype(np.int32)


def _model(case, seed):
    return moert.SynthModel(_config(case), seed=seed + 1, wdtype=DTYPES[case["dtype"]],
                            embed_dtype=DTYPES[case["embed"]], std=STD)


def _block_data(case, seed):
    c = _config(case)
    dt = DTYPES[case.get("dtype", "q8_0")]
    router = moert.synth_quantized(seed, 1, c.experts * c.hidden, STD, dt)
    gate_up = moert.synth_quantized(seed, 2, c.experts * 2 * c.inter * c.hidden, STD, dt)
    down = moert.synth_quantized(seed, 3, c.experts * c.hidden * c.inter, STD, dt)
    bias = moert.zipf_bias(c.experts, seed, case["zipf"]) if case.get("zipf") else None
    x = np.random.default_rng(seed + 3).standard_normal((case.get("m", 1), c.hidden)).astype(np.float32)
    return c, dt, router, gate_up, down, bias, x


def _attn_data(case, seed):
    c = _config(case)
    g = torch.Generator(device="cuda").manual_seed(seed + 5)
    q = 4.0 * torch.randn(c.heads, 64, generator=g, device="cuda")
    k, v = (torch.randn(c.kv_heads, case["max_len"], 64, generator=g, device="cuda").half() for _ in range(2))
    return c, q, k, v


def prepare(case, seed):
    kind = case["kind"]
    if kind == "attn":
        c, q, k, v = _attn_data(case, seed)
        return dict(case=case, c=c, q=q, k=k, v=v, out=torch.empty_like(q),
                    tps=moert.tiles_per_split(case["max_len"], case["splits"]))
    if kind in ("block", "batch"):
        c, dt, router, gate_up, down, bias, x = _block_data(case, seed)
        b = moert.GpuBlock(c.hidden, c.inter, c.experts, c.top_k, router, gate_up, down, dt, bias)
        return dict(case=case, block=b, x=x)
    m = _model(case, seed)
    slots = int(m.cfg.layers * m.cfg.experts * case["pool"]) if case.get("pool") else None
    g = moert.GpuModel(m, _max_len(case), attn_splits=case.get("splits", 32), cache_slots=slots)
    if case.get("mode"):
        g.batched_mode(case["mode"])
    ctx = case.get("ctx", 0)
    if ctx:
        for l in range(m.cfg.layers):
            g.kv_prefill(l, *moert.kv_prefill_data(m.cfg, seed, l, ctx))
    return dict(case=case, model=g, tokens=_tokens(case, seed, m.cfg.vocab))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        c = state["c"]
        moert.attn_decode_noalloc(state["q"].data_ptr(), state["k"].data_ptr(), state["v"].data_ptr(), c.heads,
                                  c.kv_heads, case["max_len"], case["ctx"], c.attention_multiplier, state["tps"],
                                  state["out"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        return state["out"]
    if kind == "block":
        return state["block"].forward(state["x"][0])
    if kind == "batch":
        return state["block"].forward_batched(state["x"])
    g, tokens = state["model"], state["tokens"]
    if kind == "generate":
        g.reset()
        out = g.generate(tokens, case["new"])
        return dict(tokens=out, logits=g.read_logits())
    g.set_position(case["ctx"])  # back to the end of what is cached: the same turn again
    if kind == "decode":
        return [g.step(int(t))[:3] for t in tokens]
    logits, _ = g.prefill(tokens)
    out = dict(logits=logits, hidden=g.hidden())
    if not case["ctx"]:
        k, v = g.read_kv(g.cfg.layers - 1, case["n"])
        out.update(k=k.view(np.float16), v=v.view(np.float16))
    return out


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def _distinct(experts, k, n):
    """Experts that n positions of k experts each are expected to use."""
    return experts * (1.0 - (1.0 - k / experts) ** n)


def work(case):
    c = _config(case)
    H, I, k, kv, qd = c.hidden, c.inter, c.top_k, c.kv_heads * 64, c.heads * 64
    if case["kind"] == "attn":
        n = case["ctx"]
        return dict(bytes=4 * n * kv + 8 * qd, flops=4 * qd * n)
    dt = DTYPES[case.get("dtype", "q8_0")]
    expert = moert.dtype_bytes(dt, 3 * I * H)
    router = moert.dtype_bytes(dt, c.experts * H)
    if case["kind"] in ("block", "batch"):
        m = case.get("m", 1)
        return dict(bytes=int(_distinct(c.experts, k, m) * expert + router + m * (8 * H + 8 * k)),
                    flops=2 * m * (k * 3 * I * H + c.experts * H))
    attn = (qd + 2 * kv) * H + H * qd
    head = moert.dtype_bytes(DTYPES[case["embed"]], c.vocab * H)
    ctx, n = case.get("ctx", 0), case["n"]
    token = 2 * (attn + k * 3 * I * H + c.experts * H)
    if case["kind"] == "prefill":
        layer = moert.dtype_bytes(dt, attn) + router + int(_distinct(c.experts, k, n) * expert) + 8 * H
        rows = sum(range(ctx + 1, ctx + n + 1))
        return dict(bytes=c.layers * (layer + 4 * kv * (ctx + 2 * n)) + head + 4 * c.vocab,
                    flops=c.layers * (n * token + 4 * qd * rows) + 2 * c.vocab * H)
    steps = n + (case["new"] - 1 if case["kind"] == "generate" else 0)
    total = sum(moert.step_bytes(c, dt, DTYPES[case["embed"]], ctx + i + 1) for i in range(steps))
    rows = sum(range(ctx + 1, ctx + steps + 1))
    return dict(bytes=total, flops=c.layers * (steps * token + 4 * qd * rows) + 2 * steps * c.vocab * H)


def tolerance(case):
    if case["kind"] == "attn":
        return {"rel": 1e-6, "max": 4e-6}  # f32 sums: 2.7e-7 and 9e-7 against 64 bits
    if case["kind"] == "block":
        return {"rel": 1e-6, "max": 4e-6}  # f32 sums: 2.1e-7 and 7e-7
    if case["kind"] == "batch":
        return {"rel": 2e-4, "max": 1e-3}  # 15-bit codes of the activations: 4.6e-5 and 2.4e-4
    # K/V rows are fp16: an entry that rounds the other way differs by 9.8e-4 of itself and travels through the layers
    # and steps that follow; 1.2e-4 and 5.5e-4 of the logits against 64 bits over 43 steps of 24 layers, 1.0e-4 and
    # 9.8e-4 of K and V rows through the integer products
    return {"rel": 5e-4, "max": 4e-3, "differ": 0.02}


# ---- the same in 64 bits -------------------------------------------------------------------------------------------
def _dequant(raw, dtype, rows, cols, lo=0, hi=None):
    """Rows [lo, hi) of a matrix of GGML blocks, in 64 bits, on the GPU."""
    hi = rows if hi is None else hi
    if dtype == moert.F32:
        return torch.from_numpy(raw.reshape(rows, cols)[lo:hi]).cuda().double()
    size = 34 if dtype == moert.Q8_0 else 18
    b = torch.from_numpy(raw.reshape(rows, cols // 32, size)[lo:hi]).cuda()
    d = b[:, :, :2].contiguous().view(torch.float16).double()
    if dtype == moert.Q8_0:
        q = b[:, :, 2:].contiguous().view(torch.int8).double()
    else:
        n = b[:, :, 2:]
        q = torch.cat([n & 15, n >> 4], 2).double() - 8.0
    return (q * d).reshape(hi - lo, cols)


def _experts64(xn, logits, k, inter, gate_up, down):
    """y [n, H], ids, weights of the top k experts of each row; gate_up(e), down(e) give an expert's matrices."""
    n = xn.shape[0]
    top = torch.sort(logits, dim=1, descending=True, stable=True)
    ids = top.indices[:, :k]
    w = torch.softmax(top.values[:, :k], dim=1)
    y = torch.zeros_like(xn)
    for e in torch.unique(ids).tolist():
        p, j = torch.nonzero(ids == e, as_tuple=True)
        gu = xn[p] @ gate_up(e).T.contiguous()
        act = torch.nn.functional.silu(gu[:, :inter]) * gu[:, inter:]
        y[p] += w[p, j, None] * (act @ down(e).T.contiguous())
    return y, ids, w


def _block64(case, seed):
    c, dt, router, gate_up, down, bias, x = _block_data(case, seed)
    H, I, E = c.hidden, c.inter, c.experts
    xd = torch.from_numpy(x).cuda().double()
    logits = xd @ _dequant(router, dt, E, H).T.contiguous()
    if bias is not None:
        logits = logits + torch.from_numpy(bias).cuda().double()
    y, ids, w = _experts64(xd, logits, c.top_k, I,
                           lambda e: _dequant(gate_up, dt, E * 2 * I, H, e * 2 * I, (e + 1) * 2 * I),
                           lambda e: _dequant(down, dt, E * H, I, e * H, (e + 1) * H))
    out = y.cpu().numpy(), ids.to(torch.int32).cpu().numpy(), w.cpu().numpy()
    return tuple(a[0] for a in out) if case["kind"] == "block" else out


def _softmax_attend(q, k, v, scale, first):
    """q [n, heads, 64] at positions first, first + 1, ..; k, v [kv, len, 64]."""
    n, heads, _ = q.shape
    group = heads // k.shape[0]
    out = torch.empty_like(q)
    pos = torch.arange(k.shape[1], device=q.device)[None, :]
    hide = pos > (first + torch.arange(n, device=q.device))[:, None]
    for h in range(heads):
        s = (q[:, h] @ k[h // group].T.contiguous()) * scale
        out[:, h] = torch.softmax(s.masked_fill(hide, -math.inf), dim=1) @ v[h // group]
    return out


class _Model64:
    """The model in 64 bits; K and V rows are kept in fp16, as the model's cache is defined, and the rotary angles
    in f32."""

    def __init__(self, case, seed):
        self.m = _model(case, seed)
        c = self.c = self.m.cfg
        self.kv = []
        for l in range(c.layers):
            if case.get("ctx"):
                kv = [torch.from_numpy(a.view(np.float16)).cuda() for a in
                      moert.kv_prefill_data(c, seed, l, case["ctx"])]
            else:
                kv = [torch.empty(c.kv_heads, 0, 64, dtype=torch.float16, device="cuda") for _ in range(2)]
            self.kv.append(kv)
        self.norm = torch.from_numpy(self.m.arrays["norm"]).cuda().double()

    def mat(self, l, name, rows, cols, lo=0, hi=None):
        return _dequant(self.m.arrays[f"{l}.{name}"], self.m.wdtype, rows, cols, lo, hi)

    def rms(self, x, w):
        return x * torch.rsqrt((x * x).mean(1, keepdim=True) + self.c.eps) * w

    def forward(self, tokens):
        """(logits of the last position, ids and weights of every layer at it); its hidden state in self.last."""
        c, a = self.c, self.m.arrays
        H, I, E, qd, kvd = c.hidden, c.inter, c.experts, c.heads * 64, c.kv_heads * 64
        n, pos0 = len(tokens), self.kv[0][0].shape[1]
        ed = self.m.embed_dtype
        h = torch.cat([_dequant(a["embed"], ed, c.vocab, H, int(t), int(t) + 1) for t in tokens])
        h = h * c.embedding_multiplier
        inv = torch.from_numpy(c.inv_freq())
        ang = (torch.arange(pos0, pos0 + n, dtype=torch.float32)[:, None] * inv[None, :]).double().cuda()
        cos, sin = torch.cos(ang)[:, None, :], torch.sin(ang)[:, None, :]

        def rot(x):
            x1, x2 = x[..., :32], x[..., 32:]
            return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], 2)

        ids, wts = [], []
        for l in range(c.layers):
            f64 = lambda name: torch.from_numpy(a[f"{l}.{name}"]).cuda().double()  # noqa: E731
            xn = self.rms(h, f64("ln_attn"))
            q = rot((xn @ self.mat(l, "q", qd, H).T.contiguous()).reshape(n, c.heads, 64))
            k = rot((xn @ self.mat(l, "k", kvd, H).T.contiguous()).reshape(n, c.kv_heads, 64))
            v = (xn @ self.mat(l, "v", kvd, H).T.contiguous()).reshape(n, c.kv_heads, 64)
            for i, new in ((0, k), (1, v)):
                self.kv[l][i] = torch.cat([self.kv[l][i], new.transpose(0, 1).half()], 1)
            att = _softmax_attend(q, self.kv[l][0].double(), self.kv[l][1].double(), c.attention_multiplier, pos0)
            h = h + c.residual_multiplier * (att.reshape(n, qd) @ self.mat(l, "o", H, qd).T.contiguous())
            xn = self.rms(h, f64("ln_moe"))
            logits = xn @ self.mat(l, "router", E, H).T.contiguous()
            y, i, w = _experts64(xn, logits, c.top_k, I,
                                 lambda e: self.mat(l, "gate_up", E * 2 * I, H, e * 2 * I, (e + 1) * 2 * I),
                                 lambda e: self.mat(l, "down", E * H, I, e * H, (e + 1) * H))
            h = h + c.residual_multiplier * y
            ids.append(i[-1])
            wts.append(w[-1])
        self.last = h[-1].cpu().numpy()
        xn = self.rms(h[-1:], self.norm)[0]
        if not hasattr(self, "head"):
            self.head = _dequant(a["embed"], ed, c.vocab, H)
        out = (self.head @ xn) / c.logits_scaling
        return (out.cpu().numpy(), torch.stack(ids).to(torch.int32).cpu().numpy(), torch.stack(wts).cpu().numpy())


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn":
        c, q, k, v = _attn_data(case, seed)
        n = case["ctx"]
        return _softmax_attend(q.double()[None], k[:, :n].double(), v[:, :n].double(), c.attention_multiplier,
                               n - 1)[0]
    if kind in ("block", "batch"):
        return _block64(case, seed)
    m = _Model64(case, seed)
    tokens = _tokens(case, seed, m.c.vocab)
    if kind == "decode":
        return [m.forward([t]) for t in tokens]
    if kind == "generate":
        out = []
        logits = m.forward(tokens)[0]
        for i in range(case["new"]):
            if i:
                logits = m.forward(out[-1:])[0]
            # the engine's greedy choice: the last index of equal maxima
            out.append(int(logits.size - 1 - np.argmax(logits[::-1])))
        return dict(tokens=np.array(out, np.int32), logits=logits)
    out = dict(logits=m.forward(tokens)[0], hidden=m.last)
    if not case["ctx"]:
        k, v = (a.cpu().numpy() for a in m.kv[-1])
        out.update(k=k, v=v)
    return out
