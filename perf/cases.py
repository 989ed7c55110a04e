"""What the speed of this framework is judged on: the work that a Qwen3 program has it do through its public entry
points, on one GPU.

A case is a dict with a "kind":

    linear      one wcomp.gemvc1 (1 token) or wcomp.gemvc_tc (2-16 tokens) call on the host's stream
    layers      decoder layers over 1-16 tokens behind a filled cache (gemvc1 / gemvc_tc and attn.RopeAttn), replayed
                from one HIP graph as the reference engine's program does
    engine      engine.Engine.process over a whole model, and the logits of the same tokens
    head        wcomp.greedy over a vocabulary: ids and logits
    prefill     prefill.layer over a block of prompt tokens
    matrix      prefill.matrix over a block of prompt tokens
    compress    wcomp.compress of a bf16 matrix
    rows        wcomp.decode_rows of a compressed matrix

Weights are N(0, 0.02) in bf16, in the single-matrix kinds with one row in a thousand 20 times larger (the outliers a
trained matrix has; for compress see _trained); activations are N(0, 1) with one channel in 200 ten times larger; caches hold what a normed key
and a projected value look like.  Every value is drawn on the GPU from the seed.
"""
import math
from types import SimpleNamespace

import torch

from ai_amd import prefill, wcomp
from ai_amd.attn import RopeAttn
from ai_amd.engine import Engine
from ai_amd.model import QWEN3

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
EPS = 1e-6
LARGEST = 51200 * 5120 * 4096  # multiply-adds of the largest listed case
MODELS = ["0.6b", "8b", "32b"]  # those whose heads the attention takes (1, 2, 4 or 8 query heads per key head)


def listed():
    return [
        # the smallest call of a decode step, the attention output of Qwen3-0.6B, from a program without a graph:
        # launches and host work
        dict(name="linear-0.6b-o", kind="linear", n=1024, k=2048, t=1, mode=1, norm=False),
        # one generated token of Qwen3-0.6B in a short chat: 28 layers and the tied head, bound by its launches
        dict(name="engine-0.6b-token", kind="engine", model="0.6b", t=1, pos=128, maxt=256, kv="f32"),
        # generating with Qwen3-8B behind a 2048-token prompt, the cache in bf16
        dict(name="decode-8b-2k", kind="layers", model="8b", layers=2, t=1, pos=2100, maxt=2304, kv="bf16"),
        # checking 8 speculated tokens with Qwen3-32B behind a long prompt
        dict(name="verify8-32b-4k", kind="layers", model="32b", layers=1, t=8, pos=4096, maxt=4352, kv="bf16"),
        # a chunk of 16 prompt tokens with Qwen3-8B, the default way through a prompt, with the default cache type
        dict(name="chunk16-8b", kind="layers", model="8b", layers=1, t=16, pos=496, maxt=1024, kv="f32"),
        # the next token of Qwen3-8B over its vocabulary
        dict(name="head-8b", kind="head", n=151936, k=4096, t=1, norm=True),
        # the next tokens of 5 speculated ones over the tied vocabulary of Qwen3-0.6B, to be sampled from
        dict(name="head5-0.6b", kind="head", n=151936, k=1024, t=5, norm=True),
        # a 2048-token prompt through a layer of Qwen3-8B
        dict(name="prefill-8b-2048", kind="prefill", model="8b", t=2048, start=0, maxt=2304, kv="bf16"),
        # a short, ragged prompt block behind earlier turns, Qwen3-0.6B with the default cache type
        dict(name="prefill-0.6b-301", kind="prefill", model="0.6b", t=301, start=77, maxt=512, kv="f32"),
        # the widest matrix (gate and up of Qwen3-32B) over a 4096-token prompt: the largest call
        dict(name="matrix-32b-gu-4096", kind="matrix", n=51200, k=5120, t=4096, add=False, norm=True),
        # loading: the compression of one matrix (qkv of Qwen3-8B)
        dict(name="compress-8b-qkv", kind="compress", n=6144, k=4096),
        # the exact rows back, as the reference's blocked prefill and its CPU head read them (down of Qwen3-8B)
        dict(name="rows-8b-down", kind="rows", n=4096, k=12288, first=0, last=4096, dtype="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "layers", "layers", "engine", "head", "prefill", "prefill", "matrix",
                       "compress", "rows"])
    model = rng.choice(MODELS)
    kv = rng.choice(sorted(DTYPES))
    if kind == "linear":
        mode = rng.choice([0, 0, 1, 2])
        return dict(kind=kind, n=_log(rng, 256, 32768), k=256 * _log(rng, 3, 68), t=rng.choice([1, 1, rng.randint(2, 16)]),
                    mode=mode, norm=mode == 0 and rng.random() < 0.6)
    if kind == "layers":
        t = rng.choice([1, 1, rng.randint(2, 16)])
        pos = _log(rng, 1, 4000)
        return dict(kind=kind, model=model, layers=1, t=t, pos=pos, maxt=pos + t + rng.randint(1, 300), kv=kv)
    if kind == "engine":
        t = rng.choice([1, rng.randint(2, 16)])
        pos = _log(rng, 16, 400)
        return dict(kind=kind, model="0.6b", t=t, pos=pos, maxt=pos + t + rng.randint(1, 100), kv="f32")
    if kind == "head":
        return dict(kind=kind, n=_log(rng, 32000, 151936), k=rng.choice([1024, 2048, 4096, 5120]), t=rng.randint(1, 16),
                    norm=rng.random() < 0.8)
    if kind == "prefill":
        model = rng.choice(["0.6b", "0.6b", "8b"])
        t = _log(rng, 17, 2048)
        start = rng.choice([0, rng.randint(1, 600)])
        return dict(kind=kind, model=model, t=t, start=start, maxt=start + t + rng.randint(0, 300), kv=kv)
    if kind == "matrix":
        n, k = _log(rng, 512, 32768), 256 * _log(rng, 3, 68)
        t = _log(rng, 17, min(4096, LARGEST // (n * k)))
        add = rng.random() < 0.5
        return dict(kind=kind, n=n, k=k, t=t, add=add, norm=not add)
    n, k = _log(rng, 256, 16384), 256 * _log(rng, 3, 50)
    if kind == "compress":
        return dict(kind=kind, n=n, k=k)
    first = rng.choice([0, rng.randint(0, n // 2)])
    return dict(kind=kind, n=n, k=k, first=first, last=rng.choice([n, rng.randint(first + 1, n)]),
                dtype=rng.choice(sorted(DTYPES)))


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _weights(g, n, k, outliers=True):
    w = torch.randn(n, k, generator=g, device="cuda").mul_(0.02)
    if outliers:
        w[torch.randint(0, n, (max(1, n // 1000),), generator=g, device="cuda")] *= 20.0
    return w.to(torch.bfloat16)


def _trained(g, n, k):
    """A matrix to compress: one weight in 6553 far below its row's exponents, the others within 11 of them, so that
    every matrix of a size has as many exceptions (about as many as N(0, 0.02) has)."""
    w = torch.randn(n, k, generator=g, device="cuda").mul_(0.02)
    w = torch.copysign(w.abs().clamp_(2.0 ** -14, 0.124), w)
    at = torch.arange(0, n * k - 6552, 6553, device="cuda")
    w.view(-1)[at + torch.randint(0, 6553, at.shape, generator=g, device="cuda")] = 2.0 ** -30
    return w.to(torch.bfloat16)


def _acts(g, t, k):
    x = torch.randn(t, k, generator=g, device="cuda")
    x[:, torch.randint(0, k, (max(1, k // 200),), generator=g, device="cuda")] *= 10.0
    return x


def _norm_weight(g, k):
    return (1.0 + 0.1 * torch.randn(k, generator=g, device="cuda")).to(torch.bfloat16)


def _dims(model):
    c = QWEN3[model]
    return SimpleNamespace(D=c["hidden_size"], L=c["num_hidden_layers"], H=c["num_attention_heads"],
                           KV=c["num_key_value_heads"], HD=c["head_dim"], FF=c["intermediate_size"],
                           V=c["vocab_size"], theta=c["rope_theta"], eps=EPS)


def _shapes(d):
    return {"qkv": ((d.H + 2 * d.KV) * d.HD, d.D), "o": (d.D, d.H * d.HD), "gu": (2 * d.FF, d.D), "down": (d.D, d.FF)}


def _inv(d):
    return (1.0 / (d.theta ** (torch.arange(0, d.HD, 2, dtype=torch.float32) / d.HD))).cuda()


def _layer(g, d):
    """A layer's matrices and norm weights."""
    w = {name: _weights(g, n, k, outliers=False) for name, (n, k) in _shapes(d).items()}
    w.update(ln1=_norm_weight(g, d.D), ln2=_norm_weight(g, d.D), qn=_norm_weight(g, d.HD), kn=_norm_weight(g, d.HD))
    return w


def _caches(g, d, maxt, filled, kv):
    """A layer's caches, `filled` positions of them used."""
    c = torch.zeros(2, d.KV, maxt, d.HD, device="cuda")
    c[:, :, :filled] = torch.randn(2, d.KV, filled, d.HD, generator=g, device="cuda")
    return c.to(DTYPES[kv]).unbind(0)


class _Checkpoint:
    """A model of random weights, with what engine.Engine asks a checkpoint for."""

    def __init__(self, model, seed):
        self.__dict__.update(vars(_dims(model)))
        self.seed, self.tied, self.eos = seed, True, set()

    def head_name(self):
        return "model.embed_tokens.weight"

    def layer_params(self):
        return _shapes(self)

    def layer(self, i, device="cuda"):
        return {k: v.to(device) for k, v in _layer(_gen(self.seed * 1000 + i + 1), self).items()}

    def t(self, name, device="cuda"):
        g = _gen(self.seed * 1000)
        norm = _norm_weight(g, self.D)
        return (norm if name == "model.norm.weight" else _weights(g, self.V, self.D, outliers=False)).to(device)


def _tokens(case, g, vocab):
    return torch.randint(0, vocab, (case["t"],), generator=g, device="cuda").tolist()


def _raw(case, seed):
    """The inputs of the kinds that hold no engine: plain tensors."""
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("linear", "head", "matrix"):
        n, k, t = case["n"], case["k"], case["t"]
        mode = case.get("mode", 0)
        r = dict(w=_weights(g, n, k), x=_acts(g, t, 2 * k if mode == 2 else k),
                 lnw=_norm_weight(g, k) if case["norm"] else None)
        # the residual row that an accumulating call adds to
        r["y"] = torch.randn(t, n, generator=g, device="cuda") if mode or case.get("add") else torch.zeros(t, n, device="cuda")
        return r
    if kind in ("layers", "prefill"):
        d = _dims(case["model"])
        pos = case["pos"] if kind == "layers" else case["start"]
        ls = []
        for _ in range(case.get("layers", 1)):
            w = _layer(g, d)
            w["kc"], w["vc"] = _caches(g, d, case["maxt"], pos, case["kv"])
            ls.append(w)
        return dict(d=d, layers=ls, x=_acts(g, case["t"], d.D))
    return dict(w=(_trained if kind == "compress" else _weights)(g, case["n"], case["k"]))


MATS = ("qkv", "o", "gu", "down")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "engine":
        ck = _Checkpoint(case["model"], seed)
        eng = Engine(ck, maxt=case["maxt"], kv_dtype=DTYPES[case["kv"]], prefill="legacy")
        g = _gen(seed * 1000 + 999)
        fill = [_caches(g, eng, case["maxt"], case["pos"], case["kv"]) for _ in range(eng.L)]
        toks = _tokens(case, g, eng.V)
        eng.process(toks, case["pos"])  # records the graph of this pass size
        for i, (k, v) in enumerate(fill):
            eng.Kc[i].copy_(k)
            eng.Vc[i].copy_(v)
        return dict(case=case, eng=eng, toks=toks, ids=torch.zeros(16, dtype=torch.int64, device="cuda"),
                    logits=torch.zeros(case["t"], eng.V, device="cuda"))
    r = _raw(case, seed)
    s = dict(case=case)
    if kind == "compress":
        return dict(s, w=r["w"])
    if kind in ("linear", "head", "matrix", "rows"):
        s["c"] = wcomp.compress(r["w"])
        s.update({k: r[k] for k in ("x", "y", "lnw") if k in r})
        s["ids"] = torch.zeros(16, dtype=torch.int64, device="cuda")
        return s
    d = r["d"]
    s["eng"] = SimpleNamespace(**vars(d), inv=_inv(d), small=[])
    s["w"], s["kc"], s["vc"] = [], [], []
    for w in r["layers"]:
        s["w"].append({n: wcomp.compress(w[n]) for n in MATS})
        s["eng"].small.append({"ln1": w["ln1"], "ln2": w["ln2"], "qn": w["qn"].float(), "kn": w["kn"].float()})
        s["kc"].append(w["kc"])
        s["vc"].append(w["vc"])
    s["x0"] = r["x"]
    if kind == "layers":
        _record(s, d)
    return s


def _record(s, d):
    """The layers' calls as one HIP graph: what a decoding program keeps."""
    case = s["case"]
    t = case["t"]
    s["x"] = torch.empty_like(s["x0"])
    qkv = torch.empty(t, (d.H + 2 * d.KV) * d.HD, device="cuda")
    att = torch.empty(t, d.H * d.HD, device="cuda")
    gu = torch.empty(t, 2 * d.FF, device="cuda")
    pos = torch.full((1,), case["pos"], dtype=torch.int64, device="cuda")
    attn = RopeAttn(d.H, d.KV, d.HD, case["maxt"], DTYPES[case["kv"]], EPS, "cuda")
    s["keep"] = (qkv, att, gu, pos, attn)

    def one(l, x):
        w, sm = s["w"][l], s["eng"].small[l]
        kc, vc, inv = s["kc"][l], s["vc"][l], s["eng"].inv
        if t == 1:
            wcomp.gemvc1(x, w["qkv"], qkv, 0, lnw=sm["ln1"], eps=EPS)
            attn(qkv, sm["qn"], sm["kn"], inv, pos, kc, vc, att)
            wcomp.gemvc1(att, w["o"], x, 1)
            wcomp.gemvc1(x, w["gu"], gu, 0, lnw=sm["ln2"], eps=EPS)
            wcomp.gemvc1(gu, w["down"], x, 2)
        else:
            wcomp.gemvc_tc(x, w["qkv"], qkv, 0, t, lnw=sm["ln1"], eps=EPS)
            attn.batch(qkv, sm["qn"], sm["kn"], inv, pos, kc, vc, att, t)
            wcomp.gemvc_tc(att, w["o"], x, 1, t)
            wcomp.gemvc_tc(x, w["gu"], gu, 0, t, lnw=sm["ln2"], eps=EPS)
            wcomp.gemvc_tc(gu, w["down"], x, 2, t)

    def step():
        s["x"].copy_(s["x0"])  # the embedding rows of the tokens
        for l in range(len(s["w"])):
            one(l, s["x"])

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()  # workspaces get allocated
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        step()


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["t"] == 1:
            wcomp.gemvc1(s["x"], s["c"], s["y"], case["mode"], lnw=s["lnw"], eps=EPS)
        else:
            wcomp.gemvc_tc(s["x"], s["c"], s["y"], case["mode"], case["t"], lnw=s["lnw"], eps=EPS)
        return s["y"]
    if kind == "layers":
        s["graph"].replay()
        return dict(x=s["x"], k=list(s["kc"]), v=list(s["vc"]))
    if kind == "engine":
        eng, t = s["eng"], case["t"]
        ids = eng.process(s["toks"], case["pos"])
        wcomp.greedy(eng.xb[:t], eng.head, t, s["ids"], lnw=eng.norm, eps=eng.eps, logits=s["logits"])
        return dict(ids=ids, logits=s["logits"], x=eng.xb[:t], k=[eng.Kc[0], eng.Kc[-1]], v=[eng.Vc[0], eng.Vc[-1]])
    if kind == "head":
        wcomp.greedy(s["x"], s["c"], case["t"], s["ids"], lnw=s["lnw"], eps=EPS, logits=s["y"])
        return dict(ids=s["ids"], logits=s["y"])
    if kind == "prefill":
        x = s["x0"].clone()  # the embedding rows of the prompt
        prefill.layer(s["eng"], 0, s["w"][0], x, case["start"], s["kc"][0], s["vc"][0])
        return dict(x=x, k=s["kc"][0], v=s["vc"][0])
    if kind == "matrix":
        prefill.matrix(s["x"], s["c"], s["y"], add=case["add"], lnw=s["lnw"], eps=EPS)
        return s["y"]
    if kind == "compress":
        c = wcomp.compress(s["w"])
        return {k: c[k] for k in ("base", "rp", "er", "ec", "ev") + wcomp.PACKED}
    return wcomp.decode_rows(s["c"], case["first"], case["last"], DTYPES[case["dtype"]])


# ------------------------------------------------------------------ what a pass cannot do without
def _linear_work(n, k, t, acc=False, xs=1):
    return 1.5 * n * k + 4 * n + 4 * t * k * xs + 4 * t * n * (2 if acc else 1), 2.0 * t * n * k


def _layer_work(d, t, pos, kv):
    b = f = 0.0
    for name, (n, k) in _shapes(d).items():
        lb, lf = _linear_work(n, k, t, acc=name in ("o", "down"), xs=2 if name == "down" else 1)
        b, f = b + lb, f + lf
    eb = 2 if kv == "bf16" else 4
    b += 2.0 * (pos + t) * d.KV * d.HD * eb
    f += 4.0 * d.H * d.HD * (t * pos + t * (t + 1) / 2)
    return b, f


def work(case):
    kind = case["kind"]
    if kind in ("linear", "head", "matrix"):
        mode = case.get("mode", 0)
        b, f = _linear_work(case["n"], case["k"], case["t"], acc=bool(mode or case.get("add")), xs=2 if mode == 2 else 1)
    elif kind in ("layers", "prefill"):
        b, f = _layer_work(_dims(case["model"]), case["t"], case.get("pos", case.get("start")), case["kv"])
        b, f = b * case.get("layers", 1), f * case.get("layers", 1)
    elif kind == "engine":
        d = _dims(case["model"])
        b, f = _layer_work(d, case["t"], case["pos"], case["kv"])
        hb, hf = _linear_work(d.V, d.D, case["t"])
        b, f = b * d.L + 2 * hb, f * d.L + 2 * hf  # the ids by process(), the logits by greedy()
    elif kind == "compress":
        b, f = 3.5 * case["n"] * case["k"], 0.0
    else:
        rows = case["last"] - case["first"]
        b, f = rows * case["k"] * (1.5 + (2 if case["dtype"] == "bf16" else 4)), 0.0
    return {"bytes": b, "flops": f}


def tolerance(case):
    kind = case["kind"]
    if kind in ("compress", "rows"):
        return "exact"
    if kind in ("linear", "head", "matrix"):  # seen against 64 bits: 1.3e-7 to 7.8e-7
        return {"rel": 4e-6}
    if kind == "engine":  # 1.8e-6, over 28 layers
        return {"rel": 1e-5}
    if case["kv"] == "f32":  # 1e-7 to 2e-7 behind caches of the default type, more where a layer adds up its parts
        return {"rel": 4e-6}
    # 6e-7 to 9e-6; a key or value that falls on the other side of a bf16 rounding differs by 2^-8
    return {"rel": 5e-5, "max": 1e-2}


# ------------------------------------------------------------------ the same in 64 bits, on the CPU
def _f(t):
    return t.cpu().double()


def _mm(x, w):
    """x . w^T in float64, w (bf16 on the GPU) taken in slices of rows."""
    w = w.cpu()
    return torch.cat([x @ w[i:i + 8192].double().t() for i in range(0, w.shape[0], 8192)], 1)


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * _f(w)


def _rope(x, pos, inv):
    a = (pos.float()[:, None] * inv.cpu()[None]).double()  # the angle is a float32 product, as the model defines it
    c, s = a.cos()[:, None], a.sin()[:, None]
    h = x.shape[-1] // 2
    return torch.cat([x[..., :h] * c - x[..., h:] * s, x[..., h:] * c + x[..., :h] * s], -1)


def _exact_layer(d, w, x, p0, kc, vc):
    t = x.shape[0]
    qkv = _mm(_rms(x, w["ln1"]), w["qkv"]).view(t, d.H + 2 * d.KV, d.HD)
    pos = torch.arange(p0, p0 + t)
    inv = _inv(d)
    q = _rope(_rms(qkv[:, :d.H], w["qn"]), pos, inv)
    k = _rope(_rms(qkv[:, d.H:d.H + d.KV], w["kn"]), pos, inv)
    kc, vc = kc.cpu(), vc.cpu()
    kc[:, p0:p0 + t] = k.transpose(0, 1).to(kc.dtype)
    vc[:, p0:p0 + t] = qkv[:, d.H + d.KV:].transpose(0, 1).to(vc.dtype)
    att = torch.empty(t, d.H, d.HD, dtype=torch.float64)
    hidden = torch.arange(p0 + t)[None] > pos[:, None]
    for h in range(d.H):
        g = h // (d.H // d.KV)
        s = (q[:, h] @ kc[g, :p0 + t].double().t()) * d.HD ** -0.5
        att[:, h] = torch.softmax(s.masked_fill_(hidden, -math.inf), -1) @ vc[g, :p0 + t].double()
    x = x + _mm(att.view(t, -1), w["o"])
    gu = _mm(_rms(x, w["ln2"]), w["gu"])
    x = x + _mm(torch.nn.functional.silu(gu[:, :d.FF]) * gu[:, d.FF:], w["down"])
    return x, kc, vc


def exact(case, seed):
    kind = case["kind"]
    if kind == "compress":
        return None  # whole numbers and bytes
    if kind == "engine":
        ck = _Checkpoint(case["model"], seed)
        g = _gen(seed * 1000 + 999)
        fill = [_caches(g, ck, case["maxt"], case["pos"], case["kv"]) for _ in range(ck.L)]
        toks = _tokens(case, g, ck.V)
        emb = ck.t(ck.head_name(), "cuda")
        x = _f(emb[toks])
        caches = []
        for i in range(ck.L):
            x, kc, vc = _exact_layer(ck, ck.layer(i), x, case["pos"], *fill[i])
            caches.append((kc, vc))
        logits = _mm(_rms(x, ck.t("model.norm.weight")), emb)
        return dict(ids=[None] * case["t"], logits=logits, x=x, k=[caches[0][0], caches[-1][0]],
                    v=[caches[0][1], caches[-1][1]])
    r = _raw(case, seed)
    if kind == "rows":
        return _f(r["w"][case["first"]:case["last"]])
    if kind in ("linear", "head", "matrix"):
        x = _f(r["x"])
        if case.get("mode") == 2:
            x = torch.nn.functional.silu(x[:, :case["k"]]) * x[:, case["k"]:]
        if case["norm"]:
            x = _rms(x, r["lnw"])
        y = _mm(x, r["w"])
        if case.get("mode") or case.get("add"):
            y += _f(r["y"])
        return dict(ids=None, logits=y) if kind == "head" else y
    x, ks, vs = _f(r["x"]), [], []
    p0 = case["pos"] if kind == "layers" else case["start"]
    for w in r["layers"]:
        x, kc, vc = _exact_layer(r["d"], w, x, p0, w["kc"], w["vc"])
        # which side of a tie a bf16 cache value falls on is not the precision of the path
        ks.append(kc if case["kv"] == "f32" else None)
        vs.append(vc if case["kv"] == "f32" else None)
    return dict(x=x, k=ks, v=vs) if kind == "layers" else dict(x=x, k=ks[0], v=vs[0])
