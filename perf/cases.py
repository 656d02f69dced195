"""The work that this framework's users have it do, as cases that can be timed and compared.

A case is one call of a serving program through the public binding (``rstr.hip``): a decode step
over paged lanes (primed tokens in, logits and greedy tokens out), one bulk-prefill tile, the
isolated routed attention, or a durable K/V chunk moved in and out of the page pool.  Whole models
are used where the logits are small enough to be read back by a serving program; the other decode
cases are the first layers of the benchmark's models at full width with a 4096-entry vocabulary,
so that the layers are what is timed.  Weights and K/V prefixes are the library's seeded synthetic
ones, contexts follow the benchmark's distributions (the same multiset of lengths for every seed,
dealt to the lanes by the seed), and pages are a random permutation of the pool.
"""
import math
import os
import statistics
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "pretrained-rstr_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from rstr import configs, hip  # noqa: E402

PAGE = 16
LAYER_VOCAB = 4096


def listed():
    return [
        # one interactive user of a small Q8 model: a whole decode step, logits read back
        dict(name="gemma_whole_1lane_q8", kind="step", model="gemma3_270m", layers=18, vocab=262144, bits=8,
             lanes=1, dist="uniform", lo=64, hi=64, shared=0, split=128),
        # a handful of users of a small Q4 model: a whole decode step, long and short contexts
        dict(name="qwen_whole_5lane", kind="step", model="qwen3_06b", layers=28, vocab=151936, bits=4,
             lanes=5, dist="log", lo=256, hi=8192, shared=0, split=256),
        # one user of an 8B model, 2k of context
        dict(name="llama_1lane", kind="step", model="llama3_8b", layers=4, vocab=LAYER_VOCAB, bits=4,
             lanes=1, dist="uniform", lo=2113, hi=2113, shared=0, split=64),
        # a few users of an 8B model in Q8, an odd number of lanes
        dict(name="llama_7lane_q8", kind="step", model="llama3_8b", layers=4, vocab=LAYER_VOCAB, bits=8,
             lanes=7, dist="uniform", lo=128, hi=3000, shared=0, split=256),
        # a small model with sliding windows over 16 lanes, ragged contexts
        dict(name="gemma_16lane", kind="step", model="gemma3_270m", layers=18, vocab=LAYER_VOCAB, bits=4,
             lanes=16, dist="uniform", lo=64, hi=2048, shared=0, split=32),
        # 64 lanes over a forked prompt prefix (half the lanes share 1024 tokens)
        dict(name="qwen_64lane_shared", kind="step", model="qwen3_06b", layers=4, vocab=LAYER_VOCAB, bits=4,
             lanes=64, dist="log", lo=256, hi=8192, shared=1024, split=640),
        # a half-full server of an 8B model
        dict(name="llama_45lane", kind="step", model="llama3_8b", layers=4, vocab=LAYER_VOCAB, bits=4,
             lanes=45, dist="uniform", lo=128, hi=4608, shared=0, split=256),
        # a full server of an 8B model: 128 lanes of continuous decode
        dict(name="llama_128lane", kind="step", model="llama3_8b", layers=4, vocab=LAYER_VOCAB, bits=4,
             lanes=128, dist="uniform", lo=128, hi=4608, shared=0, split=256),
        # the last tile of a 4096-token prompt
        dict(name="prefill_llama_512", kind="prefill", model="llama3_8b", layers=4, vocab=LAYER_VOCAB, bits=4,
             rows=512, start=3584, split=256),
        # a short ragged prompt suffix after a cached prefix
        dict(name="prefill_qwen_77", kind="prefill", model="qwen3_06b", layers=4, vocab=LAYER_VOCAB, bits=4,
             rows=77, start=1003, split=256),
        # attention alone over very ragged routes, a quarter of the pages shared between lanes
        dict(name="attention_128lane", kind="attention", model="llama3_8b", lanes=128, dist="lognormal", lo=16,
             hi=32768, split=256),
        # a conversation's K/V restored from and exported to its durable form (128 KiB a token)
        dict(name="chunk_roundtrip_500", kind="chunk", model="llama3_8b", tokens=500, start=37),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choices(("step", "prefill", "attention", "chunk"), (6, 3, 1, 1))[0]
    model = rng.choice(("llama3_8b", "qwen3_06b", "gemma3_270m"))
    bits = rng.choice((4, 4, 4, 8))
    layers = 6 if model == "gemma3_270m" else 4
    if kind == "step":
        hi = log_int(64, 4608)
        return dict(kind=kind, model=model, layers=layers, vocab=LAYER_VOCAB, bits=bits, lanes=log_int(1, 128),
                    dist=rng.choice(("uniform", "log")), lo=max(1, hi // rng.choice((1, 8, 30))), hi=hi,
                    shared=rng.choice((0, 0, hi // 4)), split=rng.choice((64, 128, 256, 256, 512)))
    if kind == "prefill":
        rows = log_int(12, 512)
        return dict(kind=kind, model=model, layers=layers, vocab=LAYER_VOCAB, bits=bits, rows=rows,
                    start=rng.choice((0, rng.randrange(4096 - rows))), split=rng.choice((128, 256, 256, 512)))
    if kind == "attention":
        return dict(kind=kind, model=rng.choice(("llama3_8b", "qwen3_06b")), lanes=log_int(2, 128), dist="log", lo=16,
                    hi=log_int(500, 9000), split=rng.choice((128, 256, 512)))
    return dict(kind=kind, model=model, tokens=log_int(50, 500), start=rng.randrange(200))


# ---- the cases' sizes -------------------------------------------------------------------------


def _config(case):
    cfg = dict(configs.MODELS[case["model"]])
    if case["kind"] == "attention":
        cfg.update(n_layers=1, vocab=LAYER_VOCAB)
    elif case["kind"] == "chunk":
        cfg.update(vocab=LAYER_VOCAB)
    else:
        cfg.update(n_layers=case["layers"], vocab=case["vocab"], weight_bits=case["bits"])
    return cfg


def _lengths(case):
    """The lanes' visible lengths: the distribution's quantiles, shortest first."""
    n, lo, hi = case["lanes"], case["lo"], case["hi"]
    p = [(i + 0.5) / n for i in range(n)]
    if case["dist"] == "uniform":
        v = [lo + x * (hi - lo) for x in p]
    elif case["dist"] == "log":
        v = [math.exp(math.log(lo) + x * (math.log(hi) - math.log(lo))) for x in p]
    else:
        v = [math.exp(7.0 + 1.2 * statistics.NormalDist().inv_cdf(x)) for x in p]
    return [int(min(hi, max(lo, round(x)))) for x in v]


def _pages(tokens):
    return -(-tokens // PAGE)


def _routes(case, seed):
    """(lengths by lane, page lists, pages of the pool): a permuted pool, a prefix of whole pages that the
    first half of the lanes share (``shared`` tokens), or half of each odd lane's pages shared with the
    lane before it (isolated attention)."""
    rng = np.random.default_rng(seed)
    lengths = [int(x) for x in rng.permutation(_lengths(case))]
    total = sum(_pages(n) for n in lengths) + _pages(case.get("shared", 0)) + 4
    free = [int(x) for x in rng.permutation(total)]
    prefix = [free.pop() for _ in range(case.get("shared", 0) // PAGE)]
    pages = []
    for b, n in enumerate(lengths):
        own = []
        if b < len(lengths) // 2:
            own = prefix[:(n - 1) // PAGE]
        if case["kind"] == "attention" and b % 2:
            own = pages[b - 1][:min(lengths[b - 1], n) // PAGE // 2]
        pages.append(own + [free.pop() for _ in range(_pages(n) - len(own))])
    return lengths, pages, total


def _table(pages, width):
    table = np.full((len(pages), width), -1, np.int32)
    for b, own in enumerate(pages):
        table[b, :len(own)] = own
    return table


# ---- state ------------------------------------------------------------------------------------


class State:
    """A session with what a serving program keeps open; closed with the object."""

    def __init__(self):
        self.session = hip.Session(0)

    def __del__(self):
        session, self.session = getattr(self, "session", None), None
        if session is not None:
            session.close()


def prepare(case, seed):
    cfg, s = _config(case), State()
    s.kind = case["kind"]
    rng = np.random.default_rng(seed + 1)
    model = hip.Model(s.session, cfg, seed=seed)
    if s.kind == "chunk":
        end = case["start"] + case["tokens"]
        s.pool = hip.Pool(model, PAGE, _pages(end) + 4)
        s.pages = rng.permutation(s.pool.physical_pages).astype(np.int32)[:_pages(end)]
        s.start, s.tokens = case["start"], case["tokens"]
        payload = torch.randn(s.pool.chunk_elements(s.tokens), dtype=torch.float16, device="cuda",
                              generator=torch.Generator("cuda").manual_seed(seed))
        s.payload = payload.cpu().numpy().view(np.uint16)
        return s
    if s.kind == "prefill":
        rows, start = case["rows"], case["start"]
        n = start + rows
        s.pool = hip.Pool(model, PAGE, _pages(n) + 4)
        s.pages = np.random.default_rng(seed).permutation(s.pool.physical_pages).astype(np.int32)[:_pages(n)]
        if start:
            s.pool.fill_synthetic(s.pages[:_pages(start)], seed)
        s.tile = hip.Prefill(model, s.pool, rows, _pages(n), _pages(n) * PAGE, case["split"])
        s.positions = np.arange(start, n, dtype=np.int32)
        s.slots = s.pages[s.positions // PAGE] * PAGE + s.positions % PAGE
        s.tokens = rng.integers(0, cfg["vocab"], rows).astype(np.int32)
        s.length = n
        return s
    lengths, pages, total = _routes(case, seed)
    width = _pages(max(lengths)) + 2
    s.pool = hip.Pool(model, PAGE, total)
    s.pool.fill_synthetic(sorted({p for own in pages for p in own}), seed)
    s.table, s.lengths = _table(pages, width), np.array(lengths, np.int32)
    if s.kind == "attention":
        s.split = case["split"]
        s.query = rng.standard_normal((case["lanes"], cfg["n_q"], cfg["head_dim"]), np.float32)
        return s
    lanes = case["lanes"]
    s.decoder = hip.Decoder(model, s.pool, lanes, width, width * PAGE, case["split"])
    s.lanes = np.arange(lanes, dtype=np.int32)
    s.tokens = rng.integers(0, cfg["vocab"], lanes).astype(np.int32)
    last = s.lengths - 1
    s.slots = s.table[s.lanes, last // PAGE] * PAGE + last % PAGE
    s.rows = np.arange(lanes + 1, dtype=np.int32)
    s.starts = np.zeros(lanes, np.int32)
    s.positions = last.astype(np.int32)
    return s


def run(s):
    if s.kind == "step":
        s.decoder.prime_lanes(s.lanes, s.tokens)
        tokens = s.decoder.step_lanes(s.slots, s.rows, s.positions, s.table, s.lengths, s.starts)
        return {"logits": s.decoder.logits(), "tokens": tokens}
    if s.kind == "prefill":
        s.tile.prefill_range(s.tokens, s.slots, s.positions, s.pages, s.length, 0)
        return s.tile.rows_out()
    if s.kind == "attention":
        return s.pool.attention(0, s.query, s.table, s.lengths, split=s.split)
    s.pool.restore_submit(s.pages, s.start, s.tokens, s.payload).complete()
    return s.pool.export_submit(s.pages, s.start, s.tokens).complete()["payload"].view(np.int16)


# ---- what a pass cannot do without ------------------------------------------------------------


def work(case):
    cfg = _config(case)
    hd, n_q, n_kv, d, ff, L = (cfg[k] for k in ("head_dim", "n_q", "n_kv", "d_model", "d_ff", "n_layers"))
    row = 2 * n_kv * hd * 2  # bytes of one token's K and V in one layer
    if case["kind"] == "chunk":
        moved = case["tokens"] * row * L
        return {"bytes": 4 * moved, "flops": 0}  # payload read, pages written, pages read, payload written
    if case["kind"] == "attention":
        lengths, pages, _ = _routes(case, 0)
        unique = len({p for own in pages for p in own}) * PAGE
        return {"bytes": unique * row + 2 * 4 * case["lanes"] * n_q * hd, "flops": 4 * n_q * hd * sum(lengths)}
    layer_weights = d * hd * (n_q + 2 * n_kv) + d * n_q * hd + 3 * d * ff
    per_weight = (18 if cfg["weight_bits"] == 4 else 34) / 32
    flops, size = 0, L * layer_weights * per_weight
    if case["kind"] == "prefill":
        rows, n = case["rows"], case["start"] + case["rows"]
        visible = [list(range(case["start"] + 1, n + 1))] * L
        unique = [n] * L
        out = rows * d * 4
    else:
        rows = case["lanes"]
        lengths, pages, _ = _routes(case, 0)
        visible, unique = [], []
        for layer in range(L):
            w = _window(cfg, layer)
            visible.append([min(n, w) if w else n for n in lengths])
            shared = 0 if w else sum(map(len, pages)) - len({p for own in pages for p in own})
            unique.append(sum(visible[-1]) - shared * PAGE)
        out = rows * cfg["vocab"] * 4
        size += d * cfg["vocab"] * per_weight
        flops += 2 * rows * d * cfg["vocab"]
    if case["kind"] == "prefill":
        visible = [[min(n, w) if w else n for n in v] for v, w in zip(visible, (_window(cfg, i) for i in range(L)))]
        unique = [min(n, w + rows) if w else n for n, w in zip(unique, (_window(cfg, i) for i in range(L)))]
    size += sum(unique) * row + rows * row * L + out
    flops += 2 * rows * L * layer_weights + 4 * n_q * hd * sum(sum(v) for v in visible)
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # chunks are bytes; every computed case is a chain of fp32 sums whose 8-bit activation
    # quantisation turns a last-bit change into a rounding step: measured by comparing with the
    # same case at another attention split and with exact() below, stated at about four times that
    if case["kind"] == "chunk":
        return "exact"
    if case["kind"] == "attention":
        return {"rel": 1e-6, "max": 2e-5}
    return {"rel": 0.03, "max": 0.3, "differ": 0.01}


# ---- the same in 64 bits ----------------------------------------------------------------------

_ROLES = dict(embed=0, final_norm=1, attn_norm=2, q=3, k=4, v=5, o=6, q_norm=7, k_norm=8, post_attn_norm=9,
              ffn_pre_norm=10, ffn_post_norm=11, gate=12, up=13, down=14)
_MASK = (1 << 64) - 1
_GOLDEN, _C1, _C2 = 0x9E3779B97F4A7C15, 0xBF58476D1CE4E5B9, 0x94D049BB133111EB


def _signed(v):
    return v - (1 << 64) if v >> 63 else v


def _mix(z):
    """splitmix64 of a Python integer or of an int64 tensor (products wrap)."""
    if isinstance(z, int):
        z = (z + _GOLDEN) & _MASK
        z = ((z ^ (z >> 30)) * _C1) & _MASK
        z = ((z ^ (z >> 27)) * _C2) & _MASK
        return z ^ (z >> 31)

    def shifted(x, n):
        return (x >> n) & ((1 << (64 - n)) - 1)

    z = z + _signed(_GOLDEN)
    z = (z ^ shifted(z, 30)) * _signed(_C1)
    z = (z ^ shifted(z, 27)) * _signed(_C2)
    return z ^ shifted(z, 31)


def _key(seed, layer, role):
    return _mix(_mix(seed) ^ (((layer + 1) << 16) | role))


def _normal(key, index, mean, std):
    """The seeded synthetic values (float32) at the int64 positions ``index``."""
    total = torch.zeros_like(index)
    for j in range(3):
        r = _mix((3 * index + j) * _signed(_GOLDEN) + _signed(key))
        for shift in (0, 16, 32, 48):
            total += (r >> shift) & 0xFFFF
    v = (total.double() + 6.0) / 65536.0 - 6.0
    return (mean + std * v).float()


class _Weights:
    def __init__(self, cfg, seed):
        self.cfg, self.seed = cfg, seed

    def linear(self, layer, role, n, k):
        """One linear's weights as they are stored (blocks of 32, fp16 scale), in 64 bits [n][k]."""
        out = torch.empty(n, k, dtype=torch.float64, device="cuda")
        key, step = _key(self.seed, layer, _ROLES[role]), max(1, (1 << 25) // k)
        for r in range(0, n, step):
            m = min(step, n - r)
            index = torch.arange(r * k, (r + m) * k, dtype=torch.int64, device="cuda")
            w = _normal(key, index, 0.0, 0.02).view(m, k // 32, 32)
            if self.cfg["weight_bits"] == 4:
                top = w.gather(2, w.abs().argmax(2, keepdim=True))
                scale = top / -8.0
                inverse = torch.where(scale != 0, 1.0 / scale, torch.zeros_like(scale))
                q = (w * inverse + 8.5).int().clamp(max=15) - 8
            else:
                scale = w.abs().amax(2, keepdim=True) / 127.0
                inverse = torch.where(scale != 0, 1.0 / scale, torch.zeros_like(scale))
                q = torch.round(w * inverse).clamp(-127, 127)
            out[r:r + m] = (q.double() * scale.half().double()).view(m, k)
        return out

    def gain(self, layer, role, n):
        index = torch.arange(n, dtype=torch.int64, device="cuda")
        g = _normal(_key(self.seed, layer, _ROLES[role]), index, 0.0 if self.cfg["gain_offset"] else 1.0, 0.02)
        return g.double() + (1.0 if self.cfg["gain_offset"] else 0.0)

    def embedding(self, tokens):
        d = self.cfg["d_model"]
        index = torch.tensor(tokens, dtype=torch.int64, device="cuda")[:, None] * d + torch.arange(d, device="cuda")
        e = _normal(_key(self.seed, -1, _ROLES["embed"]), index, 0.0, 0.02).double()
        return (e * (math.sqrt(d) if self.cfg["embed_scale_sqrt_d"] else 1.0)).float().double()

    def prefix(self, layer, slab, pages, n):
        """K (slab 0) or V (1) of the first ``n`` tokens of a route over synthetic pages."""
        width = self.cfg["n_kv"] * self.cfg["head_dim"]
        pick = torch.tensor([(_mix(self.seed ^ int(p)) >> 32) % 64 for p in pages], dtype=torch.int64, device="cuda")
        index = pick[:, None] * (PAGE * width) + torch.arange(PAGE * width, device="cuda")
        v = _normal(_key(self.seed, layer, 64 + slab), index, 0.0, 1.0).half().double()
        return v.view(-1, self.cfg["n_kv"], self.cfg["head_dim"])[:n]


def _window(cfg, layer):
    local = cfg["global_pattern"] > 0 and (layer + 1) % cfg["global_pattern"]
    return cfg["sliding_window"] if local else 0


def _rms(x, gain, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * gain


def _quantised(x):
    """Activations as the linears take them: 8-bit blocks of 32, the scale rounded up to 4 significant bits."""
    b = x.reshape(*x.shape[:-1], -1, 32)
    m, e = torch.frexp(b.abs().amax(-1, keepdim=True) / 127.0)
    d = torch.ldexp(torch.ceil(m * 16) / 16, e).clamp(2.0 ** -21, 480.0)
    return (torch.round(b / d).clamp(-127, 127) * d).reshape(x.shape)


def _rotated(x, positions, theta):
    half = x.shape[-1] // 2
    inverse = theta ** (-2.0 * torch.arange(half, dtype=torch.float64, device="cuda") / x.shape[-1])
    angle = positions.double()[:, None, None] * inverse
    c, s, a, b = angle.cos(), angle.sin(), x[..., :half], x[..., half:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _attend(q, k, v, visible, window, scale):
    """q [rows][n_q][hd] over one route's k, v [n][n_kv][hd]; row i sees its last ``window`` of visible[i] tokens."""
    rows, n_q, hd = q.shape
    n_kv = k.shape[1]
    first = max(0, int(visible.min()) - window) if window else 0
    k, v = k[first:], v[first:]
    at = torch.arange(first, first + k.shape[0], device="cuda")
    hidden = at[None, :] >= visible[:, None]
    if window:
        hidden |= at[None, :] < visible[:, None] - window
    out = torch.empty_like(q)
    for h in range(n_kv):
        g = slice(h * n_q // n_kv, (h + 1) * n_q // n_kv)
        s = torch.matmul(q[:, g].reshape(-1, hd), k[:, h].T.contiguous()).view(rows, -1, k.shape[0]) * scale
        p = s.masked_fill(hidden[:, None, :], -math.inf).softmax(-1)
        out[:, g] = torch.matmul(p.reshape(-1, k.shape[0]), v[:, h].contiguous()).view(rows, -1, hd)
    return out


def _forward(cfg, seed, tokens, routes, head):
    """The layers' rows in 64 bits.  ``routes``: (pages, first row, visible lengths of its rows); every row's K/V
    is appended at its last visible position.  Logits with ``head``, else the last layer's rows."""
    w, eps = _Weights(cfg, seed), cfg["eps"]
    hd, n_q, n_kv, d, ff = (cfg[k] for k in ("head_dim", "n_q", "n_kv", "d_model", "d_ff"))
    x = w.embedding(tokens)
    rows = x.shape[0]
    positions = torch.tensor([n - 1 for _, _, v in routes for n in v], device="cuda")

    def project(a, layer, role, n):
        return torch.matmul(a, w.linear(layer, role, n, a.shape[-1]).T)

    for layer in range(cfg["n_layers"]):
        window = _window(cfg, layer)
        theta = cfg["rope_local"] if cfg["rope_dual"] and (layer + 1) % max(1, cfg["global_pattern"]) else cfg["rope_global"]
        a = _quantised(_rms(x, w.gain(layer, "attn_norm", d), eps))
        q = project(a, layer, "q", n_q * hd).view(rows, n_q, hd)
        k = project(a, layer, "k", n_kv * hd).view(rows, n_kv, hd)
        v = project(a, layer, "v", n_kv * hd).view(rows, n_kv, hd).half().double()
        if cfg["qk_norm"]:
            q = _rms(q, w.gain(layer, "q_norm", hd), eps)
            k = _rms(k, w.gain(layer, "k_norm", hd), eps)
        q = _rotated(q, positions, theta)
        k = _rotated(k, positions, theta).half().double()
        o = torch.empty_like(q)
        for pages, r, visible in routes:
            n = len(visible)
            seen = torch.tensor(visible, device="cuda")
            kk, vv = (w.prefix(layer, slab, pages, max(visible)) for slab in (0, 1))
            kk[seen - 1], vv[seen - 1] = k[r:r + n], v[r:r + n]
            o[r:r + n] = _attend(q[r:r + n], kk, vv, seen, window, cfg["attn_scale"])
        o = project(_quantised(o.reshape(rows, -1)), layer, "o", d)
        if cfg["sandwich"]:
            o = _rms(o, w.gain(layer, "post_attn_norm", d), eps)
        x = x + o
        a = _quantised(_rms(x, w.gain(layer, "ffn_pre_norm", d), eps))
        gate, up = project(a, layer, "gate", ff), project(a, layer, "up", ff)
        act = torch.nn.functional.gelu(gate, approximate="tanh") if cfg["ffn_geglu"] else torch.nn.functional.silu(gate)
        y = project(_quantised(act * up), layer, "down", d)
        if cfg["sandwich"]:
            y = _rms(y, w.gain(layer, "ffn_post_norm", d), eps)
        x = x + y
    if not head:
        return x
    return project(_quantised(_rms(x, w.gain(-1, "final_norm", d), eps)), -1, "embed", cfg["vocab"])


def exact(case, seed):
    cfg = _config(case)
    if case["kind"] == "chunk":
        return None
    rng = np.random.default_rng(seed + 1)
    if case["kind"] == "prefill":
        n = case["start"] + case["rows"]
        pages = np.random.default_rng(seed).permutation(_pages(n) + 4)[:_pages(n)]
        tokens = rng.integers(0, cfg["vocab"], case["rows"])
        return _forward(cfg, seed, tokens, [(pages, 0, list(range(case["start"] + 1, n + 1)))], False)
    lengths, pages, _ = _routes(case, seed)
    if case["kind"] == "attention":
        q = torch.from_numpy(rng.standard_normal((case["lanes"], cfg["n_q"], cfg["head_dim"]), np.float32))
        q, w = q.double().cuda(), _Weights(cfg, seed)
        return torch.cat([_attend(q[b:b + 1], w.prefix(0, 0, own, n), w.prefix(0, 1, own, n),
                                  torch.tensor([n], device="cuda"), 0, cfg["attn_scale"])
                          for b, (n, own) in enumerate(zip(lengths, pages))])
    tokens = rng.integers(0, cfg["vocab"], case["lanes"])
    routes = [(own, b, [n]) for b, (n, own) in enumerate(zip(lengths, pages))]
    return {"logits": _forward(cfg, seed, tokens, routes, True), "tokens": None}
