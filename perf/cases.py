"""Performance cases: what a program asks of this package, through its public entry points.

A case is one call sequence on one resident model.  Models are the shapes of this repository's benchmark and its quick functional
runs (the Llama family with k-quant or fp32 weights, the layered designs Vudelix and Lezepel with bf16 weights); the call sequences
are the ones that `generate`, `sample`, the benchmark and the trace replay are made of:

  decode   the greedy token loop on a cache that already holds `start` positions
  prompt   a batched prompt pass, logits of the last position
  score    a batched prompt pass, logits of chosen positions
  chat     a prompt pass and the greedy token loop behind it
  sample   the temperature loop: one step, one draw, per token

Weights are random with the spread a trained model's have, N(0, 1 / inputs), and norms of one; large matrices are cut from a pool
of random rows, entered at a row of its own for each matrix.  The classifier prefers one successor for every token, and a router's
experts specialise in kinds of token, as a trained model's do: a greedy token and a choice of experts are then decided by a margin,
not by the last bit of a flat distribution.  Layered models have fewer layers and experts than the benchmark's, so that they load
in seconds; their widths are the benchmark's.

`exact` computes the same in 64 bits with torch alone: k-quant matrices multiply q8_K-quantized inputs token by token and plain
ones in a prompt pass, as the entry points specify."""
import math

import numpy as np
import torch

import __graft_entry__ as entry

DEVICE = "cuda" if torch.cuda.is_available() else "cpu"
F32, Q4, Q5, Q6, BF16 = 0, 12, 13, 14, 30
KINDS = 64  # kinds of token

# shapes of the Llama family that the benchmark runs: (dim, hidden, heads, key/value heads, vocabulary, rope base, neox)
LLAMA = {
    "8b": (4096, 14336, 32, 8, 128256, 500000.0, False),     # the headline model
    "phi3": (3072, 8192, 32, 32, 32064, 10000.0, True),      # no shared key/value heads, rotation in halves
    "2k": (2048, 8192, 16, 4, 32000, 500000.0, False),       # beside the layered models of width 2048
    "tiny": (512, 1024, 8, 2, 2048, 500000.0, False),        # the benchmark's quick functional shape
    "llama2c": (512, 1376, 8, 8, 32000, 10000.0, False),     # a llama2.c checkpoint, fp32
}
# tensor types of a file: (embedding, attention and w1 / w3, w2, classifier)
PLANS = {"q4ks": (Q4, Q4, Q4, Q6), "q5km": (Q4, Q5, Q6, Q6), "q4": (Q4, Q4, Q4, Q4), "f32": (F32, F32, F32, F32)}


def listed():
    def llama(name, shape, plan, layers, op, **kw):
        return dict(name=name, family="llama", shape=shape, plan=plan, layers=layers, op=op, **kw)

    def layered(name, family, width, ff, experts, eff, layers, op, **kw):
        return dict(name=name, family=family, width=width, ff=ff, experts=experts, eff=eff, layers=layers, precision=kw.pop("precision", "bfloat16"),
                    op=op, **kw)
    return [
        # an interactive answer of the headline model, all 32 layers
        llama("decode 8b q4ks", "8b", "q4ks", 32, "decode", start=31, new=24),
        # the same model reading a document
        llama("prompt 8b q4ks", "8b", "q4ks", 32, "prompt", prompt=2048),
        # the better-quantized file drawn from at a temperature, one call per step and draw
        llama("sample 8b q5km", "8b", "q5km", 8, "sample", start=100, new=12),
        # late in a long conversation: the cache outweighs the weights
        llama("decode phi3 long", "phi3", "q4", 16, "decode", start=3840, new=16),
        # a small fp32 checkpoint: latency of the token loop
        llama("decode llama2c", "llama2c", "f32", 8, "decode", start=15, new=48),
        # the smallest model: launches and hand-overs only
        llama("decode tiny", "tiny", "q4ks", 4, "decode", start=7, new=6),
        # a short question to a middle-sized model, and its answer
        llama("chat 2k q4ks", "2k", "q4ks", 8, "chat", prompt=37, new=16),
        # layered models of the benchmark: a long prompt ...
        layered("prompt vudelix 2k", "vudelix", 2048, 8192, 32, 1024, 4, "prompt", prompt=2048),
        layered("prompt lezepel 4k", "lezepel", 4096, 14336, 32, 2048, 3, "prompt", prompt=2048),
        # ... a conversation's turn of ordinary length ...
        layered("chat vudelix 4k", "vudelix", 4096, 14336, 16, 2048, 4, "chat", prompt=333, new=16),
        layered("chat lezepel 2k", "lezepel", 2048, 8192, 16, 1024, 4, "chat", prompt=57, new=32),
        # ... and the log-likelihood of a text in the precision option that checks are run in
        layered("score vudelix 1k f32", "vudelix", 1024, 4096, 16, 512, 4, "score", prompt=509, every=61, precision="float32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: shapes between the smallest and the largest of the benchmark, lengths over the whole range."""
    op = rng.choice(["decode", "prompt", "chat", "sample", "score"])
    lengths = {"prompt": dict(prompt=_log_int(rng, 2, 2048)), "chat": dict(prompt=_log_int(rng, 2, 1024), new=rng.randint(2, 32)),
               "score": dict(prompt=_log_int(rng, 16, 1500)), "sample": dict(start=_log_int(rng, 1, 1500), new=rng.randint(2, 16)),
               "decode": dict(start=_log_int(rng, 1, 4000), new=rng.randint(2, 40))}[op]
    if op == "score":
        lengths["every"] = rng.randint(7, 97)
    if rng.random() < 0.4:
        shape = rng.choice(sorted(LLAMA))
        plan = "f32" if shape == "llama2c" else rng.choice(["q4ks", "q5km", "q4"])
        return dict(family="llama", shape=shape, plan=plan, layers=rng.randint(2, 12), op=op, **lengths)
    if op == "decode":  # (a layered model's sequence starts at position 0: its loop comes behind a prompt)
        op, lengths = "chat", dict(prompt=_log_int(rng, 2, 64), new=lengths["new"])
    if op == "sample":
        lengths = dict(start=0, new=lengths["new"])
    width = 128 * _log_int(rng, 4, 28)
    return dict(family=rng.choice(["vudelix", "lezepel"]), width=width, ff=64 * (width * rng.randint(2, 4) // 64 + rng.choice([0, 0, 1])),
                experts=rng.choice([8, 16, 32] if width < 2048 else [8, 16]), eff=32 * (width // 64 + rng.choice([0, 0, 1])),
                layers=rng.randint(2, 4),
                precision="float32" if rng.random() < 0.15 else "bfloat16", op=op, **lengths)


# ---- model descriptions ------------------------------------------------------------------------------------------------
def _layer_specs(c):
    """One dict per layer of a layered model, the fields of LayerSpec that its design sets."""
    W, H = c["width"], c["width"] // 128
    G = math.gcd(H, max(1, H // 4))
    out = []
    for i in range(c["layers"]):
        dense = i % 2 == 0
        s = dict(ff=1 if dense else 2, ff_dim=c["ff"] if dense else c["eff"], n_experts=0 if dense else c["experts"], top=0 if dense else 4)
        if c["family"] == "lezepel":
            s.update(mixer=2, n_heads=H, n_kv_heads=H, dim=128, vdim=128, q_rank=3 * W // 8, kv_rank=512 if W >= 2048 else W // 4, rot_size=64,
                     rot_dims=64, rot_base=500000.0, rot_half=True, out_gate=True, parallel=True, ff_gated=True, scale=192 ** -0.5,
                     ff_act=3 if dense else 4, route=1, router_bias=not dense)
        elif i % 4 == 3:
            s.update(mixer=0, n_heads=H, n_kv_heads=G, dim=128, vdim=128, window=1024, rot_dims=128, rot_base=500000.0, qk_norm=True, head_gate=True,
                     scale=128 ** -0.5, ff_act=0 if dense else 1)
        else:
            s.update(mixer=1, n_heads=H, n_kv_heads=H, dim=128, vdim=128, taps=4, decay_rank=128, gate_rank=128, ff_act=0 if dense else 1)
        out.append(s)
    return out


def _loop(c):
    """A stretch of layers that runs twice, where the model has one behind its first layers."""
    return (2, 4, 2) if c["family"] == "lezepel" and c["layers"] >= 4 else None


def _runs(c):
    n, loop = list(range(c["layers"])), _loop(c)
    return n[:loop[0]] + n[loop[0]:loop[1]] * loop[2] + n[loop[1]:] if loop else n


def _seq_len(c):
    return max(512, -(-(c.get("start", 0) + c.get("prompt", 0) + c.get("new", 0)) // 512) * 512)


def _matrices(c):
    """[(name, outputs, inputs, type)] of everything that comes from the pools, embedding and classifier apart."""
    if c["family"] == "llama":
        dim, hidden, H, G = LLAMA[c["shape"]][:4]
        kv, (_, t, t2, _) = dim // H * G, PLANS[c["plan"]]
        return [((n, l), o, i, ty) for l in range(c["layers"]) for n, o, i, ty in
                (("wq", dim, dim, t), ("wk", kv, dim, t), ("wv", kv, dim, t), ("wo", dim, dim, t), ("w1", hidden, dim, t), ("w2", dim, hidden, t2),
                 ("w3", hidden, dim, t))]
    W, out = c["width"], []
    for l, s in enumerate(_layer_specs(c)):
        H, G, D, V = s["n_heads"], s["n_kv_heads"], s["dim"], s["vdim"]
        if s["mixer"] == 0:
            m = [("q", H * D, W), ("k", G * D, W), ("v", G * V, W), ("g", H, W), ("o", W, H * V)]
        elif s["mixer"] == 1:
            m = [("q", G * D, W), ("k", G * D, W), ("v", H * V, W), ("b", H, W), ("a1", 128, W), ("a2", H * D, 128), ("g1", 128, W),
                 ("g2", H * V, 128), ("o", W, H * V)]
        else:
            C, R, Q = s["kv_rank"], s["rot_size"], s["q_rank"]
            m = [("dq", Q, W), ("uq", H * (D + R), Q), ("dkv", C + R, W), ("uk", H * D, C), ("uv", H * V, C), ("g", H * V, W), ("o", W, H * V)]
        m = [("mix." + n, o, i) for n, o, i in m]
        experts = [""] if s["ff"] == 1 else ["e%d." % e for e in range(s["n_experts"])]
        for e in experts:
            for n in ("gate", "up") if s.get("ff_gated") else ("up",):
                m.append(("mlp.%s%s" % (e, n), s["ff_dim"], W))
            m.append(("mlp.%sdown" % e, W, s["ff_dim"]))
        if c["family"] == "vudelix":
            m += [("side.gate", 256, W), ("side.proj", W, 256)]
        out += [("l%d.%s" % (l, n), o, i, BF16) for n, o, i in m]
    return out


# ---- numbers -------------------------------------------------------------------------------------------------------------
def _generator(seed, stream):
    return torch.Generator(device=DEVICE).manual_seed((int(seed) * 1000003 + stream) % (1 << 62))


def _normal(seed, stream, *shape):
    return torch.randn(*shape, generator=_generator(seed, stream), device=DEVICE)


def _half(x):
    return x.half().float()


def _pack_scales(sc, mn):
    """eight 6-bit scales and eight 6-bit minima in 12 bytes"""
    lo = sc[:, :4] | (sc[:, 4:] >> 4 << 6)
    hi = mn[:, :4] | (mn[:, 4:] >> 4 << 6)
    return torch.cat([lo, hi, (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4], 1)


def _bytes(h):
    return h.half().view(torch.uint8).reshape(h.shape[0], 2)


def _encode(x, kind):
    """x [rows][inputs] fp32 -> (GGUF bytes [rows][row bytes] uint8, the values they stand for, fp32)"""
    rows, b = x.shape[0], x.reshape(-1, 256)
    if kind == Q6:
        s = b.reshape(-1, 16, 16)
        scale = s.abs().amax(2) / 31
        d = _half(scale.amax(1, keepdim=True) / 127).clamp_min(6e-8)
        sc = (scale / d).round().clamp(1, 127)
        step = (d * sc)[:, :, None]
        q = (s / step).round().clamp(-32, 31)
        y, u = (q * step).reshape(rows, -1), (q + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
        ql = torch.stack([(u[:, :, 0] & 15) | (u[:, :, 2] & 15) << 4, (u[:, :, 1] & 15) | (u[:, :, 3] & 15) << 4], 2)
        qh = (u[:, :, 0] >> 4) | (u[:, :, 1] >> 4 << 2) | (u[:, :, 2] >> 4 << 4) | (u[:, :, 3] >> 4 << 6)
        raw = [ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.int8).view(torch.uint8), _bytes(d)]
    else:
        most, s = (15 if kind == Q4 else 31), b.reshape(-1, 8, 32)
        lo = (-s.amin(2)).clamp_min(0)
        scale = (s.amax(2) + lo) / most
        d, dmin = (_half(v.amax(1, keepdim=True) / 63).clamp_min(6e-8) for v in (scale, lo))
        sc, mn = (scale / d).round().clamp(1, 63), (lo / dmin).round().clamp(0, 63)
        step, off = (d * sc)[:, :, None], (dmin * mn)[:, :, None]
        q = ((s + off) / step).round().clamp(0, most)
        y, u = (q * step - off).reshape(rows, -1), q.to(torch.uint8)
        qs = (u[:, 0::2] & 15) | (u[:, 1::2] & 15) << 4
        raw = [_bytes(d), _bytes(dmin), _pack_scales(sc.to(torch.uint8), mn.to(torch.uint8)), qs.reshape(-1, 128)]
        if kind == Q5:
            raw.insert(3, sum((u[:, k] >> 4) << k for k in range(8)))
    return torch.cat(raw, 1).reshape(rows, -1), y


class _Bank:
    """All matrices of a model: a pool of random rows for each (inputs, type), each matrix a run of rows of it.  `rows` is the form
    the package takes, on the host; `values` the numbers, on the GPU in fp64."""
    SLACK = 1024  # rows that a matrix's place can move by

    def __init__(self, c, seed):
        self.seed, self.places, most = seed, {}, {}
        for name, o, i, t in _matrices(c):
            most[i, t] = max(most.get((i, t), 0), o)
        r = np.random.default_rng([int(seed), 1])
        for name, o, i, t in _matrices(c):
            self.places[name] = (i, t, int(r.integers(0, self.SLACK)), o)
        self.sizes = {k: n + self.SLACK for k, n in most.items()}
        self.made = {}

    def _pool(self, key):
        i, t = key
        return _normal(self.seed, 10 + 32 * i + t, self.sizes[key], i) / math.sqrt(i)

    def rows(self, name):
        i, t, at, n = self.places[name]
        if (i, t) not in self.made:
            x = self._pool((i, t))
            self.made[i, t] = _host(x, t)
        return self.made[i, t][at:at + n]

    def values(self, name):
        i, t, at, n = self.places[name]
        if (i, t) not in self.made:
            self.made[i, t] = _stored(self._pool((i, t)), t)
        return self.made[i, t][at:at + n].double()


def _host(x, t):
    """the host form of a matrix: block bytes, bf16 bit patterns or fp32"""
    if t == F32:
        return x.cpu().numpy()
    return x.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16) if t == BF16 else _encode(x, t)[0].cpu().numpy()


def _stored(x, t):
    """the values a matrix holds once it is stored"""
    return x if t == F32 else x.bfloat16().float() if t == BF16 else torch.cat([_encode(p, t)[1] for p in x.split(8192)])


def _embedding(c, seed):
    """(embedding [vocab][dim], classifier: the row of a token's successor is the token's embedding) before rounding"""
    V, dim = (LLAMA[c["shape"]][4], LLAMA[c["shape"]][0]) if c["family"] == "llama" else (32000, c["width"])
    e = _normal(seed, 1, V, dim)
    if c["family"] != "llama":
        e = 0.75 * e + 0.66 * _kinds(c, seed)[torch.arange(V, device=DEVICE) % KINDS]
    return (e / 16.0 if c["family"] == "lezepel" else e), torch.roll(e, 7919 % V, 0) / math.sqrt(dim)


def _kinds(c, seed):
    """what tokens of a kind have in common"""
    return _normal(seed, 4, KINDS, c["width"])


def _router(c, seed, n):
    """rows of a router: token kind j is the business of the experts j, j + n / 4, j + n / 2, j + 3 n / 4 (mod n)"""
    rows, kinds = torch.zeros(n, c["width"], device=DEVICE), _kinds(c, seed)
    for k in range(4):
        rows.index_add_(0, (torch.arange(KINDS, device=DEVICE) + k * (n // 4)) % n, kinds)
    return rows * (13.0 / c["width"])


def _vectors(c, seed):
    """name -> fp32 vector or small matrix of a layered model that is not a product's matrix"""
    out, W = {}, c["width"]

    def put(name, a, rounded=True):
        out[name] = a.bfloat16().float() if rounded else a
    put("final.norm", torch.ones(W, device=DEVICE))
    if c["family"] == "vudelix":
        put("side.embed", _normal(seed, 2, 32000, 256 * c["layers"]) / 16)
    elif _loop(c):
        put("loop.step", 0.8 * _normal(seed, 2, _loop(c)[2], W))
    for l, s in enumerate(_layer_specs(c)):
        g, p, H, D = _generator(seed, 100 + l), "l%d." % l, s["n_heads"], s["dim"]

        def uniform(lo, hi, n):
            return torch.rand(n, generator=g, device=DEVICE) * (hi - lo) + lo
        put(p + "norm1", uniform(0.8, 1.2, W))
        if s["mixer"] == 1:
            put(p + "mix.A_log", uniform(-2.5, 0.5, H))
            put(p + "mix.dt_bias", uniform(-5.0, 0.5, H * D))
            put(p + "mix.norm", uniform(0.8, 1.2, s["vdim"]))
            for n in "qkv":
                put(p + "mix.%s.conv" % n, 0.6 * torch.randn(H * D, s["taps"], generator=g, device=DEVICE))
        if s["mixer"] == 2:
            put(p + "mix.dq.norm", uniform(0.8, 1.2, s["q_rank"]))
            put(p + "mix.dkv.norm", uniform(0.8, 1.2, s["kv_rank"]))
        if c["family"] == "vudelix":
            put(p + "norm2", uniform(0.8, 1.2, W))
            put(p + "side.norm", uniform(0.8, 1.2, W))
        if s["ff"] == 2:
            put(p + "mlp.router", _router(c, seed, s["n_experts"]))
        if s.get("router_bias"):
            put(p + "mlp.router.b", uniform(-0.5, 0.5, s["n_experts"]))
    return out


def _inputs(c, seed):
    """tokens of the prompt, the first token of a loop, uniform numbers of the draws"""
    r = np.random.default_rng([int(seed), 2])
    V = LLAMA[c["shape"]][4] if c["family"] == "llama" else 32000
    return r.integers(0, V, c.get("prompt", 0)).astype(np.int32), int(r.integers(0, V)), r.random(64) * 0.98 + 0.01


def _cache_rows(c, seed, l):
    """keys and values [start][kv_dim] that the loop finds in layer l's cache"""
    dim, _, H, G = LLAMA[c["shape"]][:4]
    kv, n = dim // H * G, c["start"]
    x = _normal(seed, 3, 2 * n + 64, kv)
    return x[l:l + n], x[n + l:2 * n + l]


# ---- the package's side --------------------------------------------------------------------------------------------------
def prepare(case, seed):
    c, pkg = case, entry.load_package()
    bank, (e, o) = _Bank(c, seed), _embedding(c, seed)
    if c["family"] == "llama":
        dim, hidden, H, G, V, base, neox = LLAMA[c["shape"]]
        te, _, _, to = PLANS[c["plan"]]

        def matrix(raw, t, i):
            return raw if t == F32 else pkg.QuantMatrix(t, raw.reshape(-1), i, raw.shape[0])

        def whole(x, t):
            return matrix(np.concatenate([_host(p, t) for p in x.split(32768)]), t, dim)
        ones = np.ones(dim, np.float32)
        layers = [pkg.TransformerLayerWeights(ones, ones, **{n: matrix(bank.rows((n, l)), bank.places[n, l][1], bank.places[n, l][0])
                                                             for n in ("wq", "wk", "wv", "wo", "w1", "w2", "w3")}) for l in range(c["layers"])]
        cfg = pkg.ModelConfig(dim, hidden, c["layers"], H, G, V, _seq_len(c), base, neox)
        weights = pkg.TransformerWeights(whole(e, te), layers, ones, whole(o, to))
    else:
        v = _vectors(c, seed)
        specs = [pkg.LayerSpec(**s) for s in _layer_specs(c)]
        kind = c["family"].capitalize()
        cfg = pkg.LayeredConfig(width=c["width"], vocab_size=32000, layers=specs, norm_eps=1e-5, residual_mult=0.4 if kind == "Vudelix" else 1.0,
                                embed_scale=1.0 if kind == "Vudelix" else 16.0, side_dim=256 if kind == "Vudelix" else 0, loop=_loop(c),
                                seq_len=_seq_len(c), precision=c["precision"], architecture=kind)

        def tensor(name):
            if name in ("embed", "head"):
                return _host(e if name == "embed" else o, BF16)
            return _host(v[name], F32 if v[name].dim() == 1 else BF16) if name in v else bank.rows(name)
        from llama2_jl_amd import layered
        weights = layered.DESIGNS[kind][1](cfg, tensor)
    model = pkg.LanguageModel(cfg, None, weights)
    dev = model.device()
    tokens, first, draws = _inputs(c, seed)
    if c["family"] == "llama" and c.get("start"):
        for l in range(c["layers"]):
            k, val = _cache_rows(c, seed, l)
            dev.kv_write(l, 0, k.cpu().numpy(), val.cpu().numpy())
    dev.ctx.sync()
    model.weights = None  # (a program lets go of the host's copy once the model is resident)
    return dict(dev=dev, case=c, tokens=tokens, first=first, draws=draws, want=np.arange(0, len(tokens), c.get("every", 1), dtype=np.int32))


def run(state):
    dev, c = state["dev"], state["case"]
    op, start = c["op"], c.get("start", 0)
    if op == "decode":
        return dict(zip(("ids", "logits"), dev.generate_greedy([state["first"]], c["new"], pos0=start, want_logits=True)))
    if op == "prompt":
        return dict(zip(("logits", "next"), dev.prefill(state["tokens"])))
    if op == "score":
        return dict(logits=dev.prefill_logits(state["tokens"], state["want"]))
    if op == "chat":
        logits, nxt = dev.prefill(state["tokens"])
        ids, last = dev.generate_greedy([nxt], c["new"], pos0=len(state["tokens"]), want_logits=True)
        return dict(logits=logits, next=nxt, ids=ids, last=last)
    token, ids, probs = state["first"], [], None
    for i in range(c["new"]):
        dev.forward(token, start + i, want_logits=False)
        if i + 1 < c["new"]:
            token = dev.sample_token(0.9, state["draws"][i])
        else:
            token, probs = dev.sample_token(0.9, state["draws"][i], want_probs=True)
        ids.append(token)
    return dict(ids=np.array(ids, np.int32), probs=probs, logits=dev.state("logits"))


# ---- what a pass cannot do without -----------------------------------------------------------------------------------------
def work(case):
    c = case
    steps = c.get("new", 0)
    n = c.get("prompt", 0)
    size = {F32: 4.0, BF16: 2.0, Q4: 144 / 256, Q5: 176 / 256, Q6: 210 / 256}
    if c["family"] == "llama":
        dim, _, H, G, V, _, _ = LLAMA[c["shape"]]
        width, classifier, specs, runs = dim, size[PLANS[c["plan"]][3]], None, list(range(c["layers"]))
    else:
        width, V, classifier, specs, runs = c["width"], 32000, 2.0, _layer_specs(c), _runs(c)
    at = c.get("start", 0) + n  # position of the loop's first step
    prompt_bytes = step_bytes = flops = 0.0
    for name, o, i, t in _matrices(c):
        layer = name[1] if specs is None else int(name.split(".")[0][1:])
        times, share = runs.count(layer), 1.0
        b = o * i * size[t]
        used = b
        if specs and ".mlp.e" in name:
            share = specs[layer]["top"] / specs[layer]["n_experts"]
            used = b * (1 - (1 - share) ** n)  # (an expert that no position chooses is not read)
        prompt_bytes += used if n else 0
        step_bytes += b * share * times  # (a step's weights do not stay on the chip until the next)
        flops += 2.0 * o * i * share * times * (n + steps)
    for l in runs:
        if specs is None:
            row, per_key, window = 2 * dim // H * G * 4, 4 * dim, 1 << 30
        else:
            s = specs[l]
            H, G, D, Vd = s["n_heads"], s["n_kv_heads"], s["dim"], s["vdim"]
            if s["mixer"] == 1:
                flops += 7.0 * H * D * Vd * (n + steps)
                step_bytes += 8.0 * H * D * Vd
                prompt_bytes += 4.0 * H * D * Vd
                continue
            row, per_key, window = (4 * G * (D + Vd), 2 * H * (D + Vd), s["window"]) if s["mixer"] == 0 else \
                (4 * (s["kv_rank"] + s["rot_size"]), 2 * H * (D + s["rot_size"] + Vd), 1 << 30)
        seen = [min(p + 1, window) for p in range(n)]
        flops += per_key * float(sum(seen)) + per_key * float(sum(min(at + k + 1, window) for k in range(steps)))
        prompt_bytes += row * n
        step_bytes += row * min(at + steps / 2.0, window)
    wanted = -(-n // c["every"]) if c["op"] == "score" else 1
    flops += 2.0 * width * V * ((wanted if n else 0) + steps)
    prompt_bytes += (width * V * classifier + 4.0 * V * wanted) if n else 0
    step_bytes += width * V * classifier
    return dict(bytes=prompt_bytes + steps * step_bytes + 4.0 * V, flops=flops)


def tolerance(case):
    c = case
    if c["op"] in ("decode", "sample"):
        if c["family"] == "llama" and c["plan"] != "f32":
            return dict(rel=3e-2, max=0.5, differ=0.0)  # q8_K quants that fall the other way: 0.03 to 0.06 off the same in 64 bits
        return dict(rel=1e-5, max=1e-3, differ=0.0)     # 32-bit sums in another order: 3e-7 to 2e-6
    if c.get("precision") == "float32":
        return dict(rel=1e-5, max=1e-3, differ=0.0)
    return dict(rel=3e-2, max=0.5, differ=0.0)          # bf16 activations between the products of a prompt pass: 0.002 to 0.014


# ---- the same in 64 bits -----------------------------------------------------------------------------------------------------
def _rms(x, eps=1e-5):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _turn(x, pos, base, dims, half):
    """the first `dims` of the last axis of x [n][heads][size] turned by pos * base^(-2 i / dims), pairs (2i, 2i+1) or (i, i + dims / 2)"""
    k = dims // 2
    f = pos[:, None].double() * base ** (-2.0 * torch.arange(k, device=x.device).double() / dims)
    co, si = torch.cos(f)[:, None], torch.sin(f)[:, None]
    y = x.clone()
    a, b = (x[..., :k], x[..., k:dims]) if half else (x[..., 0:dims:2], x[..., 1:dims:2])
    pa, pb = (y[..., :k], y[..., k:dims]) if half else (y[..., 0:dims:2], y[..., 1:dims:2])
    pa.copy_(a * co - b * si)
    pb.copy_(b * co + a * si)
    return y


def _attend(q, k, v, first, scale, window=1 << 30):
    """q [n][H][d] at positions first.., k [m][G][d], v [m][G][e] from position 0 -> [n][H][e]"""
    n, m, r = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    pos, key = torch.arange(first, first + n, device=q.device)[:, None], torch.arange(m, device=q.device)[None]
    hidden = (key > pos) | (key <= pos - window)
    out = q.new_empty(n, q.shape[1], v.shape[2])
    for h in range(q.shape[1]):
        s = (q[:, h] @ k[:, h // r].T * scale).masked_fill(hidden, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // r]
    return out


def _q8(x):
    """q8_K of x [n][inputs]: blocks of 256 in steps of their largest element / -127"""
    b = x.reshape(-1, 256)
    top = b.gather(1, b.abs().argmax(1, keepdim=True))
    inv = torch.where(top == 0, torch.ones_like(top), -127.0 / top)
    return ((b * inv).round().clamp_max(127) / inv).reshape(x.shape)


class _Exact:
    """A sequence of one model in fp64: step(tokens) runs the next positions and returns the residual stream behind the last layer."""

    def __init__(self, c, seed):
        self.c, self.bank, self.at, self.mem = c, _Bank(c, seed), 0, {}
        e, o = _embedding(c, seed)
        te, to = (PLANS[c["plan"]][0], PLANS[c["plan"]][3]) if c["family"] == "llama" else (BF16, BF16)
        self.e, self.o = _stored(e, te), _stored(o, to)
        self.quantized = False
        if c["family"] == "llama":
            self.layers = range(c["layers"])
            if c.get("start"):
                self.at = c["start"]
                for l in self.layers:
                    self.mem[l] = tuple(a.double().reshape(self.at, LLAMA[c["shape"]][3], -1) for a in _cache_rows(c, seed, l))
        else:
            self.v = {k: x.double() for k, x in _vectors(c, seed).items()}
            self.specs = _layer_specs(c)

    def mul(self, name, x):
        return x @ self.bank.values(name).T

    def logits(self, x):
        x = _rms(x)
        if self.c["family"] == "llama":
            return torch.cat([(_q8(x) if self.quantized else x) @ p.double().T for p in self.o.split(16384)], 1)
        return torch.cat([(x * self.v["final.norm"]) @ p.double().T for p in self.o.split(16384)], 1)

    def step(self, tokens):
        tokens = torch.as_tensor(np.atleast_1d(tokens), device=DEVICE, dtype=torch.long)
        x = (self._llama if self.c["family"] == "llama" else self._layered)(tokens, torch.arange(self.at, self.at + len(tokens), device=DEVICE))
        self.at += len(tokens)
        return x

    def _keep(self, run, *new):
        """the run's cache with the rows of these positions behind it"""
        old = self.mem.get(run)
        self.mem[run] = new if old is None else tuple(torch.cat([a, b]) for a, b in zip(old, new))
        return self.mem[run]

    def _llama(self, tokens, pos):
        dim, _, H, G, _, base, neox = LLAMA[self.c["shape"]]
        hs, n, cast = dim // H, len(tokens), (_q8 if self.quantized else lambda z: z)
        x = self.e[tokens].double()
        for l in self.layers:
            h = cast(_rms(x))
            q, k, v = (self.mul((w, l), h).reshape(n, -1, hs) for w in ("wq", "wk", "wv"))
            k, v = self._keep(l, _turn(k, pos, base, hs, neox), v)
            a = _attend(_turn(q, pos, base, hs, neox), k, v, self.at, hs ** -0.5)
            x = x + self.mul(("wo", l), cast(a.reshape(n, -1)))
            h = cast(_rms(x))
            x = x + self.mul(("w2", l), cast(torch.nn.functional.silu(self.mul(("w1", l), h)) * self.mul(("w3", l), h)))
        return x

    def _layered(self, tokens, pos):
        vud, v = self.c["family"] == "vudelix", self.v
        x0 = self.e[tokens].double() * (1.0 if vud else 16.0)
        x, loop, turn = x0, _loop(self.c), 0
        for r, l in enumerate(_runs(self.c)):
            s, p = self.specs[l], "l%d." % l
            if loop and l == loop[0] and turn < loop[2]:
                x = x + (x0 if turn else 0) + v["loop.step"][turn]
                turn += 1
            h = _rms(x) * v[p + "norm1"]
            mixed = (self._window, self._delta, self._latent)[s["mixer"]](r, s, p + "mix.", h, pos)
            if not vud:
                x = x + mixed + self._feed(s, p + "mlp.", h)
                continue
            x = x + 0.4 * mixed
            x = x + 0.4 * self._feed(s, p + "mlp.", _rms(x) * v[p + "norm2"])
            e = v["side.embed"][tokens, l * 256:(l + 1) * 256]
            y = self.mul(p + "side.proj", torch.nn.functional.gelu(self.mul(p + "side.gate", x), approximate="tanh") * e)
            x = x + 0.4 * _rms(y) * v[p + "side.norm"]
        return x

    def _window(self, r, s, p, h, pos):
        n = len(h)
        q, k, val = (self.mul(p + w, h).reshape(n, -1, 128) for w in "qkv")
        q, k = (_rms(_turn(a, pos, s["rot_base"], s["rot_dims"], False)) for a in (q, k))
        k, val = self._keep(r, k, val)
        a = _attend(q, k, val, self.at, s["scale"], s["window"]) * torch.sigmoid(self.mul(p + "g", h))[:, :, None]
        return self.mul(p + "o", a.reshape(n, -1))

    def _delta(self, r, s, p, h, pos):
        n, H, D, v = len(h), s["n_heads"], s["dim"], self.v
        past, S = self.mem.get(r, (None, None))
        S = h.new_zeros(H, D, s["vdim"]) if S is None else S
        raw = torch.cat([self.mul(p + w, h) for w in "qkv"], 1)
        taps = torch.cat([v[p + w + ".conv"] for w in "qkv"])
        full = torch.cat([raw.new_zeros(s["taps"] - 1, raw.shape[1]) if past is None else past, raw])
        y = torch.nn.functional.silu(sum(full[j:j + n] * taps[:, j] for j in range(s["taps"])))
        q, k, val = (a.reshape(n, H, D) for a in y.split(H * D, 1))
        q, k = (a / torch.sqrt((a * a).sum(-1, keepdim=True) + 1e-6) for a in (q, k))
        q = q / math.sqrt(D)
        beta = torch.sigmoid(self.mul(p + "b", h))
        rate = torch.nn.functional.softplus(self.mul(p + "a2", self.mul(p + "a1", h)) + v[p + "dt_bias"]).reshape(n, H, D)
        g = torch.exp(-torch.exp(v[p + "A_log"])[:, None] * rate)
        o = h.new_empty(n, H, s["vdim"])
        for t in range(n):
            S = S * g[t][:, :, None]
            u = beta[t][:, None] * (val[t] - torch.bmm(k[t][:, None], S)[:, 0])
            S = torch.baddbmm(S, k[t][:, :, None], u[:, None])
            o[t] = torch.bmm(q[t][:, None], S)[:, 0]
        self.mem[r] = (full[n:], S)
        gate = torch.sigmoid(self.mul(p + "g2", self.mul(p + "g1", h))).reshape(n, H, -1)
        return self.mul(p + "o", (_rms(o) * v[p + "norm"] * gate).reshape(n, -1))

    def _latent(self, r, s, p, h, pos):
        n, H, D, R, v = len(h), s["n_heads"], s["dim"], s["rot_size"], self.v
        q = self.mul(p + "uq", _rms(self.mul(p + "dq", h)) * v[p + "dq.norm"]).reshape(n, H, D + R)
        d = self.mul(p + "dkv", h)
        c = _rms(d[:, :s["kv_rank"]]) * v[p + "dkv.norm"]
        q = torch.cat([q[..., :D], _turn(q[..., D:], pos, s["rot_base"], s["rot_dims"], True)], 2)
        shared = _turn(d[:, None, s["kv_rank"]:], pos, s["rot_base"], s["rot_dims"], True).expand(n, H, R)
        k = torch.cat([self.mul(p + "uk", c).reshape(n, H, D), shared], 2)
        k, val = self._keep(r, k, self.mul(p + "uv", c).reshape(n, H, -1))
        a = _attend(q, k, val, self.at, s["scale"]).reshape(n, -1)
        return self.mul(p + "o", a * torch.sigmoid(self.mul(p + "g", h)))

    def _feed(self, s, p, h):
        act = (torch.nn.functional.gelu, lambda z: torch.relu(z) ** 2, None, torch.relu, torch.nn.functional.silu)[s["ff_act"]]

        def one(e, z):
            if s.get("ff_gated"):
                return self.mul(p + e + "down", act(self.mul(p + e + "gate", z)) * self.mul(p + e + "up", z))
            return self.mul(p + e + "down", act(self.mul(p + e + "up", z)))
        if s["ff"] == 1:
            return one("", h)
        z = h @ self.v[p + "router"].T
        if s.get("router_bias"):
            z = z + self.v[p + "router.b"]
        top, who = z.topk(s["top"], 1)
        w, y = (torch.softmax(top, 1) if s.get("route") else torch.sigmoid(top)), torch.zeros_like(h)
        for e in range(s["n_experts"]):
            rows, slot = (who == e).nonzero(as_tuple=True)
            if len(rows):
                we = w[rows, slot][:, None]
                y.index_add_(0, rows, we * one("e%d." % e, h[rows]) if s.get("route") else one("e%d." % e, we * h[rows]))
        return y


def exact(case, seed):
    c, m = case, _Exact(case, seed)
    tokens, first, draws = _inputs(c, seed)
    quantized = c["family"] == "llama" and c["plan"] != "f32"  # (the token loop's products take q8_K inputs, the prompt pass's do not)

    def loop(token):
        m.quantized = quantized
        ids = []
        for _ in range(c["new"]):
            logits = m.logits(m.step(token))[0]
            token = int(logits.argmax())
            ids.append(token)
        return np.array(ids, np.int32), logits
    if c["op"] == "decode":
        ids, logits = loop(first)
        return dict(ids=ids, logits=logits)
    if c["op"] == "sample":
        m.quantized, token, ids = quantized, first, []
        for i in range(c["new"]):
            logits = m.logits(m.step(token))[0]
            probs = torch.softmax(logits / 0.9, 0)
            token = int((probs.cumsum(0) < draws[i] * probs.sum()).sum())
            ids.append(token)
        return dict(ids=np.array(ids, np.int32), probs=probs, logits=logits)
    x = m.step(tokens)
    if c["op"] == "score":
        return dict(logits=m.logits(x[::c["every"]]))
    logits = m.logits(x[-1:])[0]
    out = dict(logits=logits, next=int(logits.argmax()))
    if c["op"] == "chat":
        out["ids"], out["last"] = loop(out["next"])
    return out
