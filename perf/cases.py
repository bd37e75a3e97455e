"""The work that this framework is used for, as cases that can be timed.

listed() names the cases, draw(rng) gives more of the same ranges. prepare()
makes what a program holds before the call (weights uploaded, the KV pool, the
plan's host arrays), run() makes one call through the public Python API, work()
counts the bytes and flops the call cannot do without, and exact() restates the
call in float64 with plain torch.

Three kinds of call:
  linear     Context.linear: y[M,N] = x[M,K] . deq(W), every weight form, the
             three activation forms (f32, the f16 hi + lo pair that a step's
             producers write, f16 operands).
  attention  Context.paged_attention: one ragged launch over a paged f16 cache,
             decode rows (extent 1) and prefill chunks.
  step       Context.step: a whole batched forward pass that returns its logits.
The widths are those of the 0.6B, 8B and 32B configurations in bench.py.
"""
import math
import random

import numpy as np
import torch

import tgo_amd

DH = 128
FORMS = {"f16": tgo_amd.FORM_F16, "i8": tgo_amd.FORM_I8, "i4tgo": tgo_amd.FORM_I4_TGO,
         "i4sym": tgo_amd.FORM_I4_SYM}
DTYPES = {"f32": tgo_amd.F32, "f16": tgo_amd.F16, "x2": tgo_amd.F16X2}
MODELS = {
    "0.6b": dict(hidden=1024, heads=16, kv_heads=8, ffn=3072),
    "8b": dict(hidden=4096, heads=32, kv_heads=8, ffn=12288),
}
EPS, THETA = 1e-6, 1e6
# The projections of the three configurations, [K, N] as a layer runs them
# (QKV and gate/up fused): 0.6B, 8B, 32B.
SHAPES = [(1024, 4096), (2048, 1024), (1024, 6144), (3072, 1024),
          (4096, 6144), (4096, 4096), (4096, 12288), (4096, 24576), (12288, 4096),
          (5120, 10240), (8192, 5120), (25600, 5120)]
LARGEST_LINEAR = 1152 * 4096 * 24576


def listed():
    return [
        # one sequence decoding: the fused QKV of an 8B layer, the smallest call
        dict(name="linear_1_int4", kind="linear", form="i4sym", m=1, k=4096, n=6144, x="f32", y="f32"),
        # eight sequences decoding over int8 weights: the fused QKV of a 32B layer
        dict(name="linear_8_int8", kind="linear", form="i8", m=8, k=5120, n=10240, x="f32", y="f32"),
        # three decode rows and a 64-token chunk: the gate/up of a 0.6B f16 layer
        dict(name="linear_67_f16", kind="linear", form="f16", m=67, k=1024, n=6144, x="x2", y="f32"),
        # a batch of 128 decoding sequences: the down projection of an 8B layer
        dict(name="linear_128_int4", kind="linear", form="i4sym", m=128, k=12288, n=4096, x="x2", y="f32"),
        # a ragged mixed batch over tgo's own int4 pack, f32 activations
        dict(name="linear_353_tgo4", kind="linear", form="i4tgo", m=353, k=4096, n=12288, x="f32", y="f32"),
        # 128 decode rows beside two 512-token chunks: the gate/up of an 8B layer
        dict(name="linear_1152_int4", kind="linear", form="i4sym", m=1152, k=4096, n=24576, x="x2", y="f32"),
        # prefill in the f16-operand arithmetic
        dict(name="linear_1024_f16ops", kind="linear", form="i4sym", m=1024, k=4096, n=12288, x="f16", y="f16"),
        # the attention of a decode-only step: 128 sequences, lognormal contexts
        dict(name="attn_decode_128", kind="attention", decodes=128, dist="lognormal", lo=16, hi=8192,
             chunks=0, chunk=0, heads=32, kv_heads=8, q="f32", lens=11),
        # a mixed ragged launch: 56 decode rows and 8 chunks of up to 256 tokens
        dict(name="attn_mixed_64", kind="attention", decodes=56, dist="uniform", lo=1, hi=4096,
             chunks=8, chunk=256, heads=32, kv_heads=8, q="f32", lens=12),
        # prefill alone with f16 queries: four 512-token chunks
        dict(name="attn_prefill_f16", kind="attention", decodes=0, dist="uniform", lo=512, hi=4096,
             chunks=4, chunk=512, heads=32, kv_heads=8, q="f16", lens=13),
        # a small model's whole step: 0.6B widths and depth, f16 weights, three
        # decodes at contexts 37, 300 and 511 beside a fresh 64-token chunk
        dict(name="step_06b_f16", kind="step", model="0.6b", layers=28, vocab=151936, form="f16",
             contexts="37,300,511", decodes=3, chunks=1, chunk=64, fresh=True, ports="packed", lens=14),
        # the serving step at 8B widths (four of its layers, a short vocabulary):
        # 128 decodes beside two 512-token chunks, ports derived on the device
        dict(name="step_8b_int4", kind="step", model="8b", layers=4, vocab=8192, form="i4sym",
             contexts="", decodes=128, chunks=2, chunk=512, fresh=False, ports="derived", lens=15),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["attention"] * 3 + ["step"])
    if kind == "linear":
        form = rng.choice(["i4sym", "i4sym", "i4tgo", "i8", "f16"])
        k, n = rng.choice(SHAPES)
        if rng.random() < 0.25:  # other widths a checkpoint may have
            k, n = 64 * _log_int(rng, 8, 160), 128 * _log_int(rng, 8, 160)
        m = _log_int(rng, 1, 1353)
        m = max(1, min(m, LARGEST_LINEAR // (k * n)))
        x = rng.choice(["x2", "x2", "f32", "f16"])
        return dict(kind="linear", form=form, m=m, k=k, n=n, x=x, y="f16" if x == "f16" else "f32")
    if kind == "attention":
        decodes, chunks = rng.choice([(1, 0), (0, 1), (1, 1)])
        decodes *= _log_int(rng, 1, 128)
        chunks *= rng.randint(1, 8)
        heads, kv = rng.choice([(16, 8), (32, 8), (64, 8)])
        dist = rng.choice(["uniform", "lognormal"])
        return dict(kind="attention", decodes=decodes, dist=dist, lo=rng.randint(1, 512),
                    hi=_log_int(rng, 1024, 4096), chunks=chunks, chunk=_log_int(rng, 16, 512) if chunks else 0,
                    heads=heads, kv_heads=kv, q=rng.choice(["f32", "f32", "f16"]), lens=rng.randint(0, 1 << 20))
    model = rng.choice(["0.6b", "8b"])
    return dict(kind="step", model=model, layers=rng.randint(4, 12) if model == "0.6b" else rng.randint(1, 3),
                vocab=8192, form=rng.choice(["f16", "i8", "i4tgo", "i4sym", "i4sym"]), contexts="",
                decodes=_log_int(rng, 1, 128), chunks=rng.randint(0, 2), chunk=_log_int(rng, 16, 512),
                fresh=False, ports=rng.choice(["packed", "derived"]), lens=rng.randint(0, 1 << 20))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _weight(form, k, n, g):
    """A random weight's stored planes, on the device: (plane, scales, zeros)."""
    if form == "f16":
        return (torch.randn(k, n, device="cuda", generator=g) * 0.02).half(), None, None

    def scales(count, mid):
        return ((torch.rand(count, device="cuda", generator=g) + 0.5) * mid).half()

    def words(count):
        w = torch.randint(0, 1 << 32, (count,), device="cuda", generator=g, dtype=torch.int64)
        return torch.where(w >= 1 << 31, w - (1 << 32), w).to(torch.int32)

    if form == "i8":
        q = torch.randint(-127, 128, (k, n), device="cuda", generator=g, dtype=torch.int8)
        return q, scales(k * n // 32, 2.7e-4), None
    if form == "i4sym":
        return words(k * n // 8), scales(k // 32 * n, 4.3e-3), None
    zeros = torch.randint(6, 10, (k * n // 128,), device="cuda", generator=g).half()
    return words(k * n // 8), scales(k * n // 128, 4.3e-3), zeros


def _dequant(form, k, n, plane, scales, zeros, dtype=torch.float64):
    """The weight's values [K, N]."""
    if form == "f16":
        return plane.to(dtype)
    if form == "i8":
        return (plane.reshape(-1, 32).to(dtype) * scales.to(dtype)[:, None]).reshape(k, n)
    shift = torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)
    if form == "i4sym":
        q = ((plane.reshape(k // 8, 1, n) >> shift[None, :, None]) & 15).reshape(k // 32, 32, n)
        return ((q - 8).to(dtype) * scales.reshape(k // 32, 1, n).to(dtype)).reshape(k, n)
    q = ((plane[:, None] >> shift[None, :]) & 15).reshape(-1, 128).to(dtype)
    return ((q - zeros.to(dtype)[:, None]) * scales.to(dtype)[:, None]).reshape(k, n)


def _host(w):
    return [None if t is None else t.cpu() for t in w]


_ctx = None


def _context():
    """The op-level calls' context: one per process, as a program keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = tgo_amd.Context(0)
        _ctx.set_stream(torch.cuda.current_stream().cuda_stream)
    return _ctx


class Linear:
    def __init__(self, case, seed):
        self.ctx = _context()
        g = _gen(seed)
        self.m, k, n = case["m"], case["k"], case["n"]
        self.handle = self.ctx.weight_upload(FORMS[case["form"]], k, n, *_host(_weight(case["form"], k, n, g)))
        x, self.x = _activation(case, g)
        self.y = torch.empty(self.m, n, device="cuda", dtype=torch.float16 if case["y"] == "f16" else torch.float32)
        self.xd, self.yd = DTYPES[case["x"]], DTYPES[case["y"]]

    def run(self):
        self.ctx.linear(self.handle, self.x, self.m, self.y, x_dtype=self.xd, y_dtype=self.yd)
        return self.y

    def __del__(self):
        if getattr(self, "handle", None) is not None and self.ctx.h:
            self.ctx.weight_free(self.handle)


def _activation(case, g):
    """(the values in float64, the stored activation) of a projection's input."""
    x = torch.randn(case["m"], case["k"], device="cuda", generator=g)
    if case["x"] == "f32":
        return x.double(), x
    hi = x.half()
    if case["x"] == "f16":
        return hi.double(), hi
    lo = (x - hi.float()).half()
    return hi.double() + lo.double(), torch.stack([hi, lo])


def _lengths(case):
    """Lengths and extents of the members: the decoding sequences, then the chunks."""
    r = random.Random(case["lens"])
    if case["kind"] == "step":
        lo, hi, dist = 16, 8192 if case["decodes"] > 64 else 4096, "lognormal"
    else:
        lo, hi, dist = case["lo"], case["hi"], case["dist"]

    def one():
        v = r.randint(lo, hi) if dist == "uniform" else round(math.exp(math.log(1024) + r.gauss(0, 1)))
        return max(lo, min(hi, int(v)))

    given = [int(v) + 1 for v in case["contexts"].split(",") if v] if case["kind"] == "step" else []
    L = given or [one() for _ in range(case["decodes"])]
    ext = [1] * len(L)
    for _ in range(case["chunks"]):
        n = case["chunk"]
        if case["kind"] == "step":
            L.append(n if case["fresh"] else n + one() // 2)
        else:
            L.append(max(1, one()))
            n = min(n, L[-1])
        ext.append(n)
    return np.array(L, np.int64), np.array(ext, np.int64)


def _pages(L, block, rng):
    """Each sequence's block table: a slice of a permutation of the pool."""
    need = (L + block - 1) // block
    perm = rng.permutation(int(need.sum()))
    pages = np.zeros((len(L), int(need.max())), np.uint32)
    at = 0
    for s, c in enumerate(need):
        pages[s, :c] = perm[at:at + c]
        at += c
    return pages, int(need.sum()) * block


BLOCK = 16


class Attention:
    def __init__(self, case, seed):
        self.ctx = _context()
        self.H, self.Hkv = case["heads"], case["kv_heads"]
        L, ext = _lengths(case)
        pages, self.cap = _pages(L, BLOCK, np.random.default_rng(seed))
        self.maxp = pages.shape[1]
        self.L, self.ext, self.pages = L.astype(np.uint32), ext.astype(np.uint32), pages.ravel()
        self.T = int(ext.sum())
        self.q, self.k, self.v = _qkv(case, seed, self.T, self.cap)
        self.dt = DTYPES[case["q"]]
        self.out = torch.empty_like(self.q)
        self.scale = 1.0 / math.sqrt(DH)

    def run(self):
        self.ctx.paged_attention(self.q, self.T, self.H, self.Hkv, self.k, self.v, self.cap, self.L, self.ext,
                                 self.pages, self.maxp, BLOCK, self.scale, self.out, q_dtype=self.dt,
                                 out_dtype=self.dt)
        return self.out


def _qkv(case, seed, T, cap):
    g = _gen(seed)
    k = torch.randn(cap, case["kv_heads"], DH, device="cuda", generator=g).half()
    v = torch.randn(cap, case["kv_heads"], DH, device="cuda", generator=g).half()
    q = torch.randn(T, case["heads"], DH, device="cuda", generator=g)
    return (q.half() if case["q"] == "f16" else q), k, v


def _model(case):
    m = MODELS[case["model"]]
    d, qw, kw, f = m["hidden"], m["heads"] * DH, m["kv_heads"] * DH, m["ffn"]
    ports = [("wq", d, qw), ("wk", d, kw), ("wv", d, kw), ("wo", qw, d), ("wgate", d, f), ("wup", d, f),
             ("wdown", f, d)]
    return m, ports


def _gain(width, g):
    return torch.rand(width, device="cuda", generator=g) + 0.5


def _model_weights(case, seed):
    """The step's weights in the order they are made: (port, form, K, N, planes) or (port, gain)."""
    m, ports = _model(case)
    g = _gen(seed)
    d, v = m["hidden"], case["vocab"]
    form = case["form"]
    eform = "f16" if form == "f16" else "i8"
    yield "embed", eform, v, d, _weight(eform, v, d, g)
    yield "lm_head", form, d, v, _weight(form, d, v, g)
    yield "final_norm", _gain(d, g)
    for l in range(case["layers"]):
        for name, width in (("attn_norm", d), ("ffn_norm", d), ("qnorm", DH), ("knorm", DH)):
            yield "%d.%s" % (l, name), _gain(width, g)
        for name, k, n in ports:
            yield "%d.%s" % (l, name), form, k, n, _weight(form, k, n, g)


class _Pool:
    """A device pool as torch sees it (f16 [layers, positions, kv_heads, head_dim])."""

    def __init__(self, address, shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f2", data=(address, False), version=2)


def _pool_layers(case, seed, cap):
    """The cached context's K and V of each layer."""
    m = MODELS[case["model"]]
    g = _gen(seed + 1)
    for _ in range(case["layers"]):
        yield tuple(torch.randn(cap, m["kv_heads"], DH, device="cuda", generator=g).half() for _ in "kv")


def _step_inputs(case, seed):
    rng = np.random.default_rng(seed)
    L, ext = _lengths(case)
    pages, cap = _pages(L, BLOCK, rng)
    ids = rng.integers(0, case["vocab"], int(ext.sum()))
    return L, ext, pages, cap, ids


class Step:
    def __init__(self, case, seed):
        m, _ = _model(case)
        self.ctx = c = tgo_amd.Context(0)
        c.set_stream(torch.cuda.current_stream().cuda_stream)
        c.config(case["layers"], m["hidden"], m["heads"], m["kv_heads"], DH, m["ffn"], case["vocab"], EPS, THETA,
                 BLOCK)
        L, ext, pages, cap, ids = _step_inputs(case, seed)
        c.kv_alloc(cap)
        kp, vp, _ = c.kv_pointers()
        shape = (case["layers"], cap, m["kv_heads"], DH)
        pools = [torch.as_tensor(_Pool(p, shape), device="cuda") for p in (kp, vp)]
        for l, kv in enumerate(_pool_layers(case, seed, cap)):
            for pool, t in zip(pools, kv):
                pool[l].copy_(t)
        for w in _model_weights(case, seed):
            if len(w) == 2:
                c.gain(w[0], w[1].cpu().numpy())
            else:
                c.weight(w[0], FORMS[w[1]], w[2], w[3], *_host(w[4]))
        cu = np.concatenate([[0], np.cumsum(ext)])
        if case["ports"] == "packed":
            members = [(ids[cu[b]:cu[b + 1]], int(L[b] - ext[b]), list(pages[b, :-(-int(L[b]) // BLOCK)]))
                       for b in range(len(L))]
            self.st = tgo_amd.new_batch_step(case["vocab"], m["heads"], m["kv_heads"], int(ext.sum()), members,
                                             BLOCK, cap)
        else:
            self.st = dict(ids=ids, posq=None, posk=None, slots=None, lengths=L, extents=ext, last=cu[1:] - 1)
        self.pages, self.maxp = pages.ravel(), pages.shape[1]

    def run(self):
        logits, _, _ = self.ctx.step(self.st, self.pages, self.maxp, want_logits=True, want_argmax=False)
        return logits

    def __del__(self):
        if getattr(self, "ctx", None) is not None:
            self.ctx.close()


KINDS = {"linear": Linear, "attention": Attention, "step": Step}


def prepare(case, seed):
    return KINDS[case["kind"]](case, seed)


def run(state):
    return state.run()


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

PER_WEIGHT = {"f16": 2.0, "i8": 1 + 2 / 32, "i4tgo": 0.5 + 4 / 128, "i4sym": 0.5 + 2 / 32}


def _attention_work(L, ext, heads, kv_heads, qbytes):
    kv = float(L.sum()) * kv_heads * DH * 2 * 2
    pairs = float(sum(n * (l - n) + n * (n + 1) / 2 for l, n in zip(L.tolist(), ext.tolist())))
    return kv + float(ext.sum()) * heads * DH * 2 * qbytes, 4.0 * DH * heads * pairs


def work(case):
    if case["kind"] == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        xb, yb = (2 if case["x"] == "f16" else 4), (2 if case["y"] == "f16" else 4)
        return dict(bytes=k * n * PER_WEIGHT[case["form"]] + m * k * xb + m * n * yb, flops=2.0 * m * k * n)
    L, ext = _lengths(case)
    if case["kind"] == "attention":
        b, f = _attention_work(L, ext, case["heads"], case["kv_heads"], 2 if case["q"] == "f16" else 4)
        return dict(bytes=b, flops=f)
    md, ports = _model(case)
    rows, members = float(ext.sum()), len(L)
    per_layer = float(sum(k * n for _, k, n in ports))
    head = float(md["hidden"] * case["vocab"])
    kv, f = _attention_work(L, ext, md["heads"], md["kv_heads"], 0)
    # the weights, the cached context and the new rows of it, the rows' embeddings, the logits
    by = (case["layers"] * (per_layer * PER_WEIGHT[case["form"]] + kv + rows * md["kv_heads"] * DH * 4) +
          head * PER_WEIGHT[case["form"]] + rows * md["hidden"] * (2 if case["form"] == "f16" else 1.0625) +
          members * case["vocab"] * 4.0)
    return dict(bytes=by, flops=case["layers"] * (2.0 * rows * per_layer + f) + 2.0 * members * head)


def tolerance(case):
    """About four times the largest error against float64 that each path shows."""
    if case["kind"] == "linear":
        # f16 out: 2.1e-4 seen, its own rounding; f32 out: 1.2e-7 to 4.6e-7
        # seen, an f32 sum of up to 25600 products of 22-bit activations
        return {"rel": 1e-3, "max": 4e-3} if case["x"] == "f16" else {"rel": 2e-6, "max": 4e-5}
    if case["kind"] == "attention":
        # f16: 2.9e-4 seen, probabilities and output rounded to f16; f32: 4.5e-6
        # to 7.4e-6 seen, 22-bit queries inside the exponential
        return {"rel": 1.2e-3, "max": 2e-2} if case["q"] == "f16" else {"rel": 3e-5, "max": 1e-3}
    # a whole step: 8e-5 to 5e-4 seen. K and V are rounded to f16 on the way into
    # the pool, so an f32 rounding can move a cached value by 2^-11 of itself
    return {"rel": 2e-3, "max": 3e-2}


# ---------------------------------------------------------------------------
# the same call in float64
# ---------------------------------------------------------------------------

def exact(case, seed):
    with torch.no_grad():
        return {"linear": _exact_linear, "attention": _exact_attention, "step": _exact_step}[case["kind"]](case, seed)


def _exact_linear(case, seed):
    g = _gen(seed)
    k, n = case["k"], case["n"]
    planes = _weight(case["form"], k, n, g)
    x, _ = _activation(case, g)
    w = _dequant(case["form"], k, n, *planes)
    if case["x"] == "f16":
        w = w.half().double()  # f16 operands: the weight is rounded once, too
    return x @ w


def _attend(q, k, v, scale, first):
    """q [n, H, d] at positions first.., k/v [L, Hkv, d]: causal attention in float64."""
    n, H, _ = q.shape
    Lk, Hkv, _ = k.shape
    G = H // Hkv
    qh = q.reshape(n, Hkv, G, DH).permute(1, 2, 0, 3).reshape(Hkv, G * n, DH).contiguous()
    kt, vh = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    mask = torch.arange(Lk, device="cuda")[None, :] > (first + torch.arange(n, device="cuda"))[:, None]
    out = []
    for h in range(Hkv):
        s = (qh[h] @ kt[h]).reshape(G, n, Lk) * scale
        p = torch.softmax(s.masked_fill(mask[None], -math.inf), -1)
        out.append((p.reshape(G * n, Lk) @ vh[h]).reshape(G, n, DH))
    return torch.stack(out).permute(2, 0, 1, 3).reshape(n, H, DH)


def _slots(pages_row, length):
    p = torch.arange(int(length), device="cuda")
    return torch.from_numpy(pages_row.astype(np.int64)).cuda()[p // BLOCK] * BLOCK + p % BLOCK


def _exact_attention(case, seed):
    L, ext = _lengths(case)
    pages, cap = _pages(L, BLOCK, np.random.default_rng(seed))
    q, k, v = _qkv(case, seed, int(ext.sum()), cap)
    out, at = [], 0
    scale = float(np.float32(1.0 / math.sqrt(DH)))
    for b in range(len(L)):
        n, sl = int(ext[b]), _slots(pages[b], L[b])
        out.append(_attend(q[at:at + n].double(), k[sl].double(), v[sl].double(), scale, int(L[b]) - n))
        at += n
    return torch.cat(out)


def _norm(x, gain):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + float(np.float32(EPS))) * gain


def _rope(x, pos):
    inv = THETA ** (-2.0 * torch.arange(DH // 2, device="cuda", dtype=torch.float64) / DH)
    a = pos.double()[:, None, None] * inv
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * a.cos() - x1 * a.sin(), x1 * a.cos() + x0 * a.sin()], -1).reshape(x.shape)


def _exact_step(case, seed):
    m, _ = _model(case)
    L, ext, pages, cap, ids = _step_inputs(case, seed)
    cu = np.concatenate([[0], np.cumsum(ext)])
    T, H, Hkv = int(cu[-1]), m["heads"], m["kv_heads"]
    W = {}
    weights = iter(_model_weights(case, seed))

    def take(count):
        for _ in range(count):
            w = next(weights)
            W[w[0].split(".")[-1]] = w[1].double() if len(w) == 2 else w[1:]

    def mat(name):
        form, k, n, planes = W[name]
        return _dequant(form, k, n, *planes)

    take(3)
    rows = torch.from_numpy(ids.astype(np.int64)).cuda()
    ef, ek, en, (ep, es, _) = W["embed"]
    h = ep[rows].double()
    if ef == "i8":
        h = (h.reshape(T, en // 32, 32) * es.reshape(ek, en // 32)[rows].double()[:, :, None]).reshape(T, en)
    pos = torch.cat([torch.arange(int(L[b] - ext[b]), int(L[b]), device="cuda") for b in range(len(L))])
    scale = float(np.float32(1.0 / math.sqrt(DH)))
    sl = [_slots(pages[b], L[b]) for b in range(len(L))]
    pools = _pool_layers(case, seed, cap)
    for l in range(case["layers"]):
        take(11)
        kc, vc = next(pools)
        x = _norm(h, W["attn_norm"])
        q = _rope(_norm((x @ mat("wq")).reshape(T, H, DH), W["qnorm"]), pos)
        k = _rope(_norm((x @ mat("wk")).reshape(T, Hkv, DH), W["knorm"]), pos).half()
        v = (x @ mat("wv")).reshape(T, Hkv, DH).half()
        out = []
        for b in range(len(L)):
            a, z, n = int(cu[b]), int(cu[b + 1]), int(ext[b])
            kb, vb = kc[sl[b]].double(), vc[sl[b]].double()
            kb[len(kb) - n:], vb[len(vb) - n:] = k[a:z].double(), v[a:z].double()
            out.append(_attend(q[a:z], kb, vb, scale, int(L[b]) - n))
        h = h + torch.cat(out).reshape(T, H * DH) @ mat("wo")
        x = _norm(h, W["ffn_norm"])
        h = h + (torch.nn.functional.silu(x @ mat("wgate")) * (x @ mat("wup"))) @ mat("wdown")
    last = torch.from_numpy(cu[1:] - 1).cuda()
    return _norm(h[last], W["final_norm"]) @ mat("lm_head")
