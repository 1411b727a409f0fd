"""Performance cases of evk_amd: what programs on this framework have it do.

Each case is one pass through the public Python entry points, at the sizes of
the benchmark configurations and of the reference's own language model, or at
generic ones: single layers (a projection, an MLP, attention, the embedding
and the head of a language model) forward and, where training uses them,
backward, and two whole calls of the decode model (prefill and greedy decode).

  listed()            the named cases
  draw(rng)           one more case of the same ranges
  prepare(case, seed) inputs, weights, outputs and caches on the GPU
  run(state)          one pass; returns the outputs
  exact(case, seed)   the same outputs in 64 bits with plain torch
  work(case)          bytes and flops that the path cannot do without
  tolerance(case)     how far a correct result may be from another one
"""
import math

import torch

import evk_amd as evk

F16 = torch.float16
F64 = torch.float64


def listed():
    return [
        # one token through a large projection: the matrix-vector product of decoding
        dict(name="linear_m1", kind="linear", m=1, n=11008, k=4096),
        # the same projection for a batch of sequences decoded together, or a short prompt
        dict(name="linear_m40", kind="linear", m=40, n=11008, k=4096),
        # feature sizes that are no multiple of anything (a class count, a concatenation)
        dict(name="linear_ragged", kind="linear", m=1000, n=1001, k=777),
        # the QKV projection of a long prompt: the largest matrix product
        dict(name="linear_qkv", kind="linear", m=8192, n=12288, k=4096),
        # the MLP of a transformer block in training: forward, weight and input gradients
        dict(name="mlp_train", kind="mlp_train", t=2560, d=768, h=3072),
        # causal attention of a prompt batch (inference)
        dict(name="attention_s1024", kind="attention", b=4, s=1024, heads=8, dh=64, causal=True),
        # the attention of the reference's training program: one head of 256
        dict(name="attention_train_d256", kind="attention_train", b=16, s=160, heads=1, dh=256, causal=True),
        # training attention over a longer, ragged sequence with heads of 128
        dict(name="attention_train_long", kind="attention_train", b=2, s=2000, heads=8, dh=128, causal=True),
        # one decode step's attention over the caches of a batch, the reference's
        # decode shape: the smallest call
        dict(name="decode_attention", kind="decode_attention", b=16, pos=159, max_seq=160, heads=1, dh=256),
        # embedding and head of a language model in training: gather, norm, logits,
        # loss, and the gradients of both tables
        dict(name="lm_ends", kind="lm_ends", t=2560, d=768, vocab=32000),
        # a prompt through the 12-layer decode model
        dict(name="prefill", kind="prefill", layers=12, d=768, heads=12, hidden=3072, vocab=32000, max_seq=1056, n=1000),
        # greedy decode of 32 tokens behind a 1024-token context
        dict(name="decode", kind="decode", layers=12, d=768, heads=12, hidden=3072, vocab=32000, max_seq=1056, pos=1024, steps=32),
    ]


def _log(rng, lo, hi, step=1):
    """A size from lo to hi, spread over its logarithm, a multiple of step."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(lo, min(hi, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear_odd", "mlp_train", "attention", "attention_train", "attention_train",
                       "decode_attention", "lm_ends", "prefill", "decode"])
    if kind == "linear":  # any token count against feature counts that are multiples of 8
        while True:
            m, n, k = _log(rng, 1, 8192), _log(rng, 256, 12288, 8), _log(rng, 256, 8192, 8)
            if 2.0 * m * n * k <= 4e11:
                return dict(kind="linear", m=m, n=n, k=k)
    if kind == "linear_odd":  # feature counts of any kind
        while True:
            m, n, k = _log(rng, 8, 4096), _log(rng, 33, 3000), _log(rng, 33, 3000)
            if 2.0 * m * n * k <= 8e9 and (n % 8 or k % 8):
                return dict(kind="linear", m=m, n=n, k=k)
    if kind == "mlp_train":
        d = _log(rng, 128, 1024, 32)
        return dict(kind=kind, t=_log(rng, 200, 6000), d=d, h=d * rng.choice([2, 3, 4]))
    if kind in ("attention", "attention_train"):
        dh = rng.choice([32, 64, 64, 128, 256])
        heads = rng.choice([1, 2, 4, 8, 12]) if dh < 256 else rng.choice([1, 2])
        while True:
            b, s = _log(rng, 1, 16), _log(rng, 64, 4096)
            if 1e7 <= float(b) * heads * dh * s * s <= 3e10:
                return dict(kind=kind, b=b, s=s, heads=heads, dh=dh, causal=rng.random() < 0.8)
    if kind == "decode_attention":
        dh = rng.choice([32, 64, 128, 256])
        heads = rng.choice([1, 2, 4, 8, 12]) if dh < 256 else rng.choice([1, 2, 4])
        while True:
            b, pos = _log(rng, 1, 64), _log(rng, 32, 4000)
            if b * pos * heads * dh <= 64 << 20:
                return dict(kind=kind, b=b, pos=pos, max_seq=pos + 1 + rng.randrange(200), heads=heads, dh=dh)
    if kind == "lm_ends":
        while True:
            t, d, v = _log(rng, 160, 4096), _log(rng, 128, 1024, 32), _log(rng, 144, 32000, 8)
            if 2.0 * t * d * v <= 1.3e11:
                return dict(kind=kind, t=t, d=d, vocab=v)
    if kind == "prefill":
        heads = rng.choice([4, 8, 12, 16])
        n = _log(rng, 16, 1024)
        return dict(kind=kind, layers=rng.randint(2, 12), d=64 * heads, heads=heads, hidden=64 * heads * rng.choice([2, 4]),
                    vocab=_log(rng, 144, 32000, 8), max_seq=n + rng.randrange(64), n=n)
    heads = rng.choice([8, 12])
    pos = _log(rng, 16, 1024)
    return dict(kind="decode", layers=rng.randint(2, 12), d=64 * heads, heads=heads, hidden=256 * heads,
                vocab=_log(rng, 1024, 32000, 8), max_seq=1056, pos=pos, steps=rng.choice([1, 8, 32]))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _Draw:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.empty(*shape, dtype=F16, device="cuda").normal_(0.0, std, generator=self.g)

    def uniform(self, *shape):
        return torch.empty(*shape, dtype=F16, device="cuda").uniform_(-1.0, 1.0, generator=self.g)

    def ids(self, count, vocab):
        """Token ids with the frequencies of text: the k-th most frequent one about 1 / k as often as the first."""
        u = torch.rand(count, device="cuda", generator=self.g)
        return (float(vocab) ** u).long().clamp_(1, vocab - 1).to(torch.int16)


def _empty(*shape, dtype=F16):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _model_cfg(c):
    return evk.model_cfg(vocab=c["vocab"], d=c["d"], heads=c["heads"], layers=c["layers"], hidden=c["hidden"], max_seq=c["max_seq"])


def _inputs(c, seed):
    """The inputs of a case, by name (those that exact() reads too)."""
    g = _Draw(seed)
    kind = c["kind"]
    if kind == "linear":
        return dict(x=g.uniform(c["m"], c["k"]), w=g.uniform(c["k"], c["n"]))
    if kind == "mlp_train":
        t, d, h = c["t"], c["d"], c["h"]
        return dict(x=g.normal(t, d), w1=g.normal(d, h, std=0.02), w2=g.normal(h, d, std=0.02), dy=g.normal(t, d))
    if kind in ("attention", "attention_train"):
        b, s, dh = c["b"], c["s"], c["dh"]
        i = dict(q=g.normal(b, s, c["heads"] * dh), k=g.normal(b, s, dh), v=g.normal(b, s, dh))
        if kind == "attention_train":
            i["do"] = g.normal(b, s, c["heads"] * dh)
        return i
    if kind == "decode_attention":
        b, d = c["b"], c["heads"] * c["dh"]
        return dict(q=g.normal(b, 1, d), k=g.normal(b, 1, d), v=g.normal(b, 1, d), kc=g.normal(b, c["max_seq"], d),
                    vc=g.normal(b, c["max_seq"], d))
    if kind == "lm_ends":
        t, d, v = c["t"], c["d"], c["vocab"]
        targets = g.ids(t, v)
        targets[159::160] = 0  # the end of each sequence has no next token
        return dict(emb=g.normal(v, d, std=0.02), wout=g.normal(d, v, std=0.02), ids=g.ids(t, v), targets=targets)
    cfg = _model_cfg(c)
    i = dict(w=g.normal(evk.model_weight_elems(cfg), std=0.02))
    if kind == "prefill":
        i.update(cache=torch.zeros(evk.model_cache_elems(cfg), dtype=F16, device="cuda"), tokens=g.ids(c["n"], c["vocab"]))
    else:  # rows of an earlier prefill: about the spread that normalised rows times such weights have
        i.update(cache=g.normal(evk.model_cache_elems(cfg), std=0.02 * math.sqrt(c["d"])), token=g.ids(1, c["vocab"]))
    return i


def prepare(case, seed):
    c = case
    s = dict(_inputs(c, seed), case=c)
    kind = c["kind"]
    if kind == "linear":
        s["y"] = _empty(c["m"], c["n"])
    elif kind == "mlp_train":
        t, d, h = c["t"], c["d"], c["h"]
        s.update(a=_empty(t, h), g=_empty(t, h), y=_empty(t, d), dg=_empty(t, h), da=_empty(t, h), dx=_empty(t, d),
                 dw1=_empty(d, h), dw2=_empty(h, d))
    elif kind in ("attention", "attention_train"):
        s.update(o=torch.empty_like(s["q"]), lse=_empty(c["b"], c["heads"], c["s"], dtype=torch.float32))
        if kind == "attention_train":
            s.update(dq=torch.empty_like(s["q"]), dk=torch.empty_like(s["k"]), dv=torch.empty_like(s["v"]))
    elif kind == "decode_attention":
        s["o"] = torch.empty_like(s["q"])
    elif kind == "lm_ends":
        t, d, v = c["t"], c["d"], c["vocab"]
        s.update(x=_empty(t, d), xn=_empty(t, d), logits=_empty(t, v), dlogits=_empty(t, v), loss=_empty(1), dxn=_empty(t, d),
                 dx=_empty(t, d), dwout=_empty(d, v), demb=_empty(v, d))
    else:
        s.update(cfg=_model_cfg(c), logits=_empty(c["vocab"]))
        if kind == "prefill":
            s["next"] = torch.zeros(1, dtype=torch.int16, device="cuda")
        else:
            s["packed"] = _empty(evk.model_packed_elems(s["cfg"]))
            evk.model_pack(s["cfg"], s["w"], s["packed"])
            s["io"] = torch.zeros(c["steps"] + 1, dtype=torch.int16, device="cuda")
            s["io"][0] = s["token"][0]
            del s["w"]
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "linear":
        evk.matmul(s["x"], s["w"], s["y"])
        return s["y"]
    if kind == "mlp_train":
        evk.matmul(s["x"], s["w1"], s["a"])
        evk.gelu(s["a"], s["g"])
        evk.matmul(s["g"], s["w2"], s["y"])
        # backward; gradients accumulate, so they are cleared for each step
        for k in ("da", "dw1", "dw2"):
            s[k].zero_()
        evk.matmul(s["g"], s["dy"], s["dw2"], transpose_a=True, acc_c=True)
        evk.matmul(s["dy"], s["w2"], s["dg"], transpose_b=True)
        evk.gelu_backward(s["dg"], s["a"], s["da"])
        evk.matmul(s["x"], s["da"], s["dw1"], transpose_a=True, acc_c=True)
        evk.matmul(s["da"], s["w1"], s["dx"], transpose_b=True)
        return {k: s[k] for k in ("y", "dx", "dw1", "dw2")}
    if kind == "attention":
        evk.flash_attention(s["q"], s["k"], s["v"], s["o"], causal=c["causal"], lse=s["lse"])
        return {k: s[k] for k in ("o", "lse")}
    if kind == "attention_train":
        evk.flash_attention(s["q"], s["k"], s["v"], s["o"], causal=c["causal"], lse=s["lse"])
        evk.flash_attention_bwd(s["q"], s["k"], s["v"], s["o"], s["do"], s["dq"], s["dk"], s["dv"], causal=c["causal"], lse=s["lse"])
        return {k: s[k] for k in ("o", "lse", "dq", "dk", "dv")}
    if kind == "decode_attention":
        evk.kv_cache_write(s["k"], s["kc"], c["pos"])
        evk.kv_cache_write(s["v"], s["vc"], c["pos"])
        evk.single_query_attention(s["q"], s["kc"], s["vc"], s["o"], c["pos"] + 1, c["heads"])
        return {k: s[k] for k in ("o", "kc", "vc")}
    if kind == "lm_ends":
        evk.embed(s["emb"], s["ids"], s["x"])
        evk.rms_norm(s["x"], s["xn"])
        evk.matmul(s["xn"], s["wout"], s["logits"])
        evk.cross_entropy_loss(s["logits"], s["targets"], s["dlogits"], s["loss"])
        for k in ("dx", "dwout", "demb"):
            s[k].zero_()
        evk.matmul(s["xn"], s["dlogits"], s["dwout"], transpose_a=True, acc_c=True)
        evk.matmul(s["dlogits"], s["wout"], s["dxn"], transpose_b=True)
        evk.rms_norm_backward(s["x"], s["dxn"], s["dx"])
        evk.embed_backward(s["dx"], s["ids"], s["demb"])
        return {k: s[k] for k in ("loss", "logits", "dwout", "demb")}
    if kind == "prefill":
        evk.model_prefill(s["cfg"], s["w"], s["cache"], s["tokens"], 0, s["next"], s["logits"])
        return {k: s[k] for k in ("logits", "cache")}
    evk.model_decode_packed(s["cfg"], s["packed"], s["cache"], s["io"], c["steps"], c["pos"], s["logits"])
    return {k: s[k] for k in ("logits", "io", "cache")}


# ---------------------------------------------------------------------------
# 64 bits
# ---------------------------------------------------------------------------
def _rms(x, eps=1e-4):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


def _attend(q, k, v, heads, causal):
    """One sequence: q (S, H * Dh); k, v (S, Dh) shared by the heads.  Per-head rows: (H, S, ...)."""
    n, dh = k.shape
    qh = q.reshape(n, heads, dh).transpose(0, 1)
    sc = torch.stack([qh[h] @ k.t() for h in range(heads)]) / math.sqrt(dh)
    if causal:
        sc = sc.masked_fill(torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    lse = torch.logsumexp(sc, -1)
    p = torch.exp(sc - lse[..., None])
    o = torch.stack([p[h] @ v for h in range(heads)])
    return qh, p, lse, o


def _exact_attention(c, i):
    out = {k: [] for k in ("o", "lse", "dq", "dk", "dv")}
    heads, dh = c["heads"], c["dh"]
    flat = lambda t: t.transpose(0, 1).reshape(c["s"], heads * dh)  # noqa: E731
    for b in range(c["b"]):
        q, k, v = (i[n][b].to(F64) for n in ("q", "k", "v"))
        qh, p, lse, o = _attend(q, k, v, heads, c["causal"])
        out["o"].append(flat(o))
        out["lse"].append(lse)
        if c["kind"] == "attention":
            continue
        do = i["do"][b].to(F64).reshape(c["s"], heads, dh).transpose(0, 1)
        delta = (do * o).sum(-1, keepdim=True)
        dq, dk, dv = torch.empty_like(qh), torch.zeros_like(k), torch.zeros_like(v)
        for h in range(heads):
            ds = p[h] * (do[h] @ v.t() - delta[h]) / math.sqrt(dh)
            dq[h] = ds @ k
            dk += ds.t() @ qh[h]
            dv += p[h].t() @ do[h]
        out["dq"].append(flat(dq))
        out["dk"].append(dk)
        out["dv"].append(dv)
    return {k: torch.stack(v) for k, v in out.items() if v}


def _exact_model(c, i, ids, pos0):
    """The decode model on tokens `ids` at positions pos0...: the last row's logits and the cache."""
    d, hid, heads, n = c["d"], c["hidden"], c["heads"], len(ids)
    dh = d // heads
    w, at = i["w"], 0

    def take(rows, cols):
        nonlocal at
        m = w[at:at + rows * cols].reshape(rows, cols).to(F64)
        at += rows * cols
        return m

    half = torch.arange(dh // 2, device="cuda", dtype=F64)
    ang = torch.arange(pos0, pos0 + n, device="cuda", dtype=F64)[:, None] * 10000.0 ** (-2.0 * half / dh)
    cs, sn = torch.cos(ang)[:, None], torch.sin(ang)[:, None]

    def rope(t):
        t = t.reshape(n, heads, dh // 2, 2)
        return torch.stack([t[..., 0] * cs - t[..., 1] * sn, t[..., 0] * sn + t[..., 1] * cs], -1).reshape(n, heads, dh)

    cache = i["cache"].to(F64).reshape(c["layers"], 2, c["max_seq"], d).clone()
    x = take(c["vocab"], d)[ids.long()]
    seen = torch.arange(pos0 + n, device="cuda")[None] > torch.arange(pos0, pos0 + n, device="cuda")[:, None]
    for layer in range(c["layers"]):
        wqkv, wo, w1, w2 = take(d, 3 * d), take(d, d), take(d, hid), take(hid, d)
        q, k, v = (_rms(x) @ wqkv).split(d, -1)
        q = rope(q)
        cache[layer, 0, pos0:pos0 + n] = rope(k).reshape(n, d)
        cache[layer, 1, pos0:pos0 + n] = v
        ks, vs = (cache[layer, j, :pos0 + n].reshape(pos0 + n, heads, dh) for j in (0, 1))
        att = torch.empty(n, heads, dh, device="cuda", dtype=F64)
        for h in range(heads):
            sc = (q[:, h] @ ks[:, h].t() / math.sqrt(dh)).masked_fill(seen, -math.inf)
            att[:, h] = torch.softmax(sc, -1) @ vs[:, h]
        x = x + att.reshape(n, d) @ wo
        x = x + _gelu(_rms(x) @ w1) @ w2
    return (_rms(x[-1:]) @ take(d, c["vocab"]))[0], cache.reshape(-1)


def exact(case, seed):
    c = case
    kind = c["kind"]
    if kind == "decode" and c["steps"] > 1:
        return None  # each step follows the greedy token of the one before
    i = _inputs(c, seed)
    if kind == "linear":
        return i["x"].to(F64) @ i["w"].to(F64)
    if kind == "mlp_train":
        x, w1, w2, dy = (i[k].to(F64) for k in ("x", "w1", "w2", "dy"))
        a = (x @ w1).requires_grad_(True)
        g = _gelu(a)
        da, = torch.autograd.grad(g, a, dy @ w2.t())
        a, g = a.detach(), g.detach()
        return dict(y=g @ w2, dx=da @ w1.t(), dw1=x.t() @ da, dw2=g.t() @ dy)
    if kind in ("attention", "attention_train"):
        return _exact_attention(c, i)
    if kind == "decode_attention":
        n, heads, dh = c["pos"] + 1, c["heads"], c["dh"]
        kc, vc = i["kc"].to(F64), i["vc"].to(F64)
        kc[:, c["pos"]], vc[:, c["pos"]] = i["k"][:, 0].to(F64), i["v"][:, 0].to(F64)
        q = i["q"].to(F64).reshape(c["b"], 1, heads, dh)
        kh, vh = (t[:, :n].reshape(c["b"], n, heads, dh) for t in (kc, vc))
        p = torch.softmax((q * kh).sum(-1, keepdim=True) / math.sqrt(dh), 1)
        return dict(o=(p * vh).sum(1).reshape(c["b"], 1, heads * dh), kc=kc, vc=vc)
    if kind == "lm_ends":
        emb, wout = i["emb"].to(F64), i["wout"].to(F64)
        ids, tg = i["ids"].long(), i["targets"].long()
        x = emb[ids].requires_grad_(True)
        xn = _rms(x)
        logits = xn.detach() @ wout
        ok = tg != 0
        grad = torch.softmax(logits, -1)
        grad[torch.arange(len(tg), device="cuda"), tg] -= 1.0
        grad = grad * ok[:, None] / ok.sum()
        loss = (torch.logsumexp(logits, -1) - logits.gather(1, tg[:, None])[:, 0])[ok].mean()
        dx, = torch.autograd.grad(xn, x, grad @ wout.t())
        return dict(loss=loss.reshape(1), logits=logits, dwout=xn.detach().t() @ grad, demb=torch.zeros_like(emb).index_add_(0, ids, dx))
    if kind == "prefill":
        logits, cache = _exact_model(c, i, i["tokens"], 0)
        return dict(logits=logits, cache=cache)
    logits, cache = _exact_model(c, i, i["token"], c["pos"])
    return dict(logits=logits, io=None, cache=cache)


# ---------------------------------------------------------------------------
# work and tolerance
# ---------------------------------------------------------------------------
def _layer_elems(c):
    return 4 * c["d"] * c["d"] + 2 * c["d"] * c["hidden"]


def work(case):
    c = case
    kind = c["kind"]
    if kind == "linear":
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=2.0 * (m * k + k * n + m * n), flops=2.0 * m * n * k)
    if kind == "mlp_train":
        t, d, h = c["t"], c["d"], c["h"]
        return dict(bytes=2.0 * (4 * t * d + 4 * d * h), flops=12.0 * t * d * h)
    if kind in ("attention", "attention_train"):
        b, s, nh, dh = c["b"], c["s"], c["heads"], c["dh"]
        one = 4.0 * b * nh * s * s * dh * (0.5 if c["causal"] else 1.0)
        if kind == "attention":
            return dict(bytes=2.0 * b * s * (2 * nh + 2) * dh + 4.0 * b * nh * s, flops=one)
        return dict(bytes=2.0 * b * s * (4 * nh + 4) * dh + 4.0 * b * nh * s, flops=3.5 * one)
    if kind == "decode_attention":
        b, n, d = c["b"], c["pos"] + 1, c["heads"] * c["dh"]
        return dict(bytes=2.0 * b * d * (2 * n + 6), flops=4.0 * b * n * d)
    if kind == "lm_ends":
        t, d, v = c["t"], c["d"], c["vocab"]
        return dict(bytes=2.0 * (t * d + 3 * d * v + t * v), flops=6.0 * t * d * v)
    n = c["n"] if kind == "prefill" else c["steps"]
    weights = 1.0 * c["layers"] * _layer_elems(c)
    if kind == "prefill":
        return dict(bytes=2.0 * (weights + c["d"] * c["vocab"] + n * c["d"] * (1 + 2 * c["layers"])),
                    flops=2.0 * n * weights + c["layers"] * 2.0 * n * n * c["d"] + 2.0 * c["d"] * c["vocab"])
    rows = sum(c["pos"] + s + 1 for s in range(n)) * 2.0 * c["layers"] * c["d"]
    step = weights + c["d"] * c["vocab"]
    return dict(bytes=2.0 * (n * step + rows), flops=2.0 * (n * step + rows))


# Outputs are fp16: one rounding of a 32-bit sum is 2.1e-4 from the 64-bit
# result (measured), chains of two to five roundings 2.5e-4 to 4e-4, twelve
# layers 1.3e-3.  About four times that; the gradients of the head pass
# through fp16 subnormals (softmax / tokens), hence the wider figure there.
TOLERANCE = {
    "linear": dict(rel=1e-3),
    "mlp_train": dict(rel=2e-3),
    "attention": dict(rel=2e-3),
    "attention_train": dict(rel=4e-3),
    "decode_attention": dict(rel=1e-3),
    "lm_ends": dict(rel=4e-3),
    "prefill": dict(rel=6e-3),
    "decode": dict(rel=6e-3),
}


def tolerance(case):
    return TOLERANCE[case["kind"]]
