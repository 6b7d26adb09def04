"""The work this framework is measured on: calls that a program serving a Q8 model makes.

A case names a model shape, a weight storage, a number of layers and a call:

  forward   Model.forward: one token over a filled cache, logits back
  turn      Model.prefill of a prompt, Model.generate_greedy, and the forward that follows
  prefill   Model.prefill of a prompt, logits of its last token
  multi     Model.prefill_multi / prefill_shared: ragged sequences in one batch, one hidden row each
  batch     Model.decode_batch: one token for each of several sequences, their logits
  ops       a stack of layers driven through the backend's single operations, as a driver
            above the backend seam issues them (llama.rs:786-862), ended by logits

Shapes, contexts and lengths are those of the benchmark and of the configurations in the tests;
where a model is cut in depth its layers, embedding and classifier keep their full size.

Every output is defined bit for bit: the reference fixes the order of each f32 sum and the
rounding of each step, so any correct implementation returns the same bits.
"""

import math
import random

import numpy as np
import torch

import kernrt_amd as K

# dim, hidden, heads, kv heads, head_dim, vocab, depth, eps, theta, q/k norms
SHAPES = {
    "135m": dict(dim=576, hidden_dim=1536, n_heads=9, n_kv_heads=3, head_dim=64, vocab_size=49152, depth=30,
                 rms_eps=1e-5, rope_theta=100_000.0, qk_norm=False),
    "360m": dict(dim=960, hidden_dim=2560, n_heads=15, n_kv_heads=5, head_dim=64, vocab_size=49152, depth=32,
                 rms_eps=1e-5, rope_theta=100_000.0, qk_norm=False),
    "1.7b": dict(dim=2048, hidden_dim=8192, n_heads=32, n_kv_heads=32, head_dim=64, vocab_size=49152, depth=24,
                 rms_eps=1e-5, rope_theta=130_000.0, qk_norm=False),
    "lfm2-700m": dict(dim=1536, hidden_dim=4608, n_heads=24, n_kv_heads=8, head_dim=64, vocab_size=65536, depth=16,
                      rms_eps=1e-5, rope_theta=1_000_000.0, qk_norm=True),
    "qwen3-0.6b": dict(dim=1024, hidden_dim=3072, n_heads=16, n_kv_heads=8, head_dim=128, vocab_size=151936, depth=28,
                       rms_eps=1e-6, rope_theta=1_000_000.0, qk_norm=True),
}
LFM2_ATTENTION = (2, 5, 8, 10, 12, 14)  # the other layers are short convolutions
CONV_K = 3


def listed():
    return [
        # The smallest call: a driver above the seam decoding one token through the single
        # operations (a quarter of the 360M shape's depth). Launches and latency.
        dict(name="ops-decode-360m-x4", kind="ops", model="360m", storage="q8_0x4", layers=8, rows=1, start=300,
             context=1024),
        # The same driver reading a prompt of an odd length; two full-width 1.7B layers.
        dict(name="ops-prompt200-1.7b", kind="ops", model="1.7b", storage="q8_0", layers=2, rows=200, start=0,
             context=512),
        # One chat token on the smallest model, the whole of it, logits back for sampling.
        dict(name="forward-135m", kind="forward", model="135m", storage="q8_0", layers=30, pos=130, context=1024),
        # The headline workload: the whole 360M shape at 512 positions; a short user turn, then
        # greedy tokens on the device.
        dict(name="greedy-360m-x4", kind="turn", model="360m", storage="q8_0x4", layers=32, start=512, prompt=9,
             steps=64, context=1024),
        # A token at the end of a long document, where the cache and the attention weigh most.
        dict(name="forward-long-qwen3", kind="forward", model="qwen3-0.6b", storage="q8_0", layers=28, pos=3100,
             context=4096),
        # The hybrid model: a 128-token prompt, then greedy decoding.
        dict(name="turn-lfm2-x4", kind="turn", model="lfm2-700m", storage="q8_0x4", layers=16, start=0, prompt=128,
             steps=32, context=2048),
        # An ordinary chat prompt of an odd length on the packed storage.
        dict(name="prompt77-360m-x4", kind="prefill", model="360m", storage="q8_0x4", layers=32, start=0, prompt=77,
             context=1024),
        # The benchmark's 128-token prompt at the 1.7B shape, a third of its depth.
        dict(name="prompt128-1.7b", kind="prefill", model="1.7b", storage="q8_0", layers=8, start=0, prompt=128,
             context=256),
        # A document: 2048 tokens through the whole Qwen3-0.6B shape.
        dict(name="prompt2048-qwen3", kind="prefill", model="qwen3-0.6b", storage="q8_0", layers=28, start=0,
             prompt=2048, context=2048),
        # Many short ragged texts in one call, one hidden row each (embedding and ranking).
        dict(name="multi24-360m-x4", kind="multi", model="360m", storage="q8_0x4", layers=16, n_seq=24, tokens=700,
             shared=0, context=1024),
        # A small server: a handful of sequences, one token each.
        dict(name="batch6-360m-x4", kind="batch", model="360m", storage="q8_0x4", layers=32, n_seq=6, context=400),
        # A loaded server: 64 sequences of up to 1024 positions, at half the model's depth.
        dict(name="batch64-qwen3", kind="batch", model="qwen3-0.6b", storage="q8_0", layers=14, n_seq=64,
             context=1024),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("ops", "forward", "turn", "prefill", "prefill", "multi", "batch"))
    model = rng.choice(tuple(SHAPES))
    if model == "lfm2-700m" and kind not in ("turn", "prefill"):  # the calls a hybrid model has
        kind = rng.choice(("turn", "prefill"))
    storage = "q8_0x4" if model == "lfm2-700m" else rng.choice(("q8_0", "q8_0x4"))
    layers = rng.randint(3, 6)
    case = dict(kind=kind, model=model, storage=storage, layers=layers)
    if kind == "ops":
        rows = _log(rng, 1, 300)
        start = rng.choice((0, rng.randint(1, 500)))
        case.update(rows=rows, start=start, context=start + rows + rng.randint(0, 300))
    elif kind == "forward":
        pos = _log(rng, 1, 3500)
        case.update(pos=pos, context=pos + rng.randint(1, 1000))
    elif kind in ("turn", "prefill"):
        prompt = _log(rng, 1, 1500) if kind == "prefill" else _log(rng, 1, 300)
        start = 0 if model == "lfm2-700m" else rng.choice((0, 0, rng.randint(1, 700)))
        steps = rng.randint(2, 24) if kind == "turn" else 0
        case.update(start=start, prompt=prompt, context=start + prompt + steps + rng.randint(2, 500))
        if kind == "turn":
            case["steps"] = steps
    elif kind == "multi":
        n_seq = rng.randint(2, 40)
        shared = rng.choice((0, rng.randint(3, 200)))
        tokens = n_seq * rng.randint(2, 30)
        case.update(n_seq=n_seq, tokens=tokens, shared=shared, context=shared + tokens + rng.randint(0, 200))
    else:
        n_seq = _log(rng, 2, 64)
        case.update(n_seq=n_seq, context=rng.randint(40, max(60, min(1000, 20000 // n_seq))))
    return case


# ---- what follows from a case alone ------------------------------------------


def _is_attention(case, layer):
    return case["model"] != "lfm2-700m" or layer in LFM2_ATTENTION


def _projections(case, layer):
    s = SHAPES[case["model"]]
    d, h, q, kv = s["dim"], s["hidden_dim"], s["n_heads"] * s["head_dim"], s["n_kv_heads"] * s["head_dim"]
    if _is_attention(case, layer):
        p = {"q": (q, d), "k": (kv, d), "v": (kv, d), "o": (d, q)}
    else:
        p = {"conv_in": (3 * d, d), "conv_out": (d, d)}
    return {**p, "gate": (h, d), "up": (h, d), "down": (d, h)}


def _lens(case):
    """The ragged lengths of a `multi` case: positive, `tokens` in all."""
    r = random.Random(case["n_seq"] * 100_003 + case["tokens"])
    cuts = sorted(r.sample(range(1, case["tokens"]), case["n_seq"] - 1))
    return [b - a for a, b in zip([0] + cuts, cuts + [case["tokens"]])]


def _positions(case):
    """How far each sequence of a `batch` case is: a server's sequences differ."""
    r = random.Random(case["n_seq"] * 100_003 + case["context"])
    return [r.randint(case["context"] // 2, case["context"] - 1) for _ in range(case["n_seq"])]


def _slots_total(case):
    """The cache's slots: the sequences of a batch keep ranges of their own in it."""
    return case["context"] * (case["n_seq"] if case["kind"] == "batch" else 1)


def _filled(case):
    """Slots that hold keys and values before the call."""
    if case["kind"] == "batch":
        return _slots_total(case)
    return case["pos"] if case["kind"] == "forward" else case.get("start", 0)


def _rows(case, tokens):
    """The rows of the call's (first) pass, (token, position, slot, first slot, shared end), and
    those that the answer is taken from."""
    kind = case["kind"]
    if kind == "batch":
        c = case["context"]
        rows = [(t, p, i * c + p, i * c, 0) for i, (t, p) in enumerate(zip(tokens, _positions(case)))]
        return rows, list(range(len(rows)))
    if kind == "multi":
        pre, rows, last = case["shared"], [], []
        rows += [(tokens[i], i, i, 0, 0) for i in range(pre)]
        base = pre
        for n in _lens(case):
            rows += [(tokens[base + i], pre + i, base + i, base, pre) for i in range(n)]
            base += n
            last.append(len(rows) - 1)
        return rows, last
    start = case["pos"] if kind == "forward" else case["start"]
    rows = [(t, start + i, start + i, 0, 0) for i, t in enumerate(tokens)]
    return rows, [len(rows) - 1]


def _n_tokens(case):
    return {"ops": case.get("rows"), "forward": 1, "turn": case.get("prompt"), "prefill": case.get("prompt"),
            "multi": case.get("shared", 0) + case.get("tokens", 0), "batch": case.get("n_seq")}[case["kind"]]


def work(case):
    s = SHAPES[case["model"]]
    q, kv = s["n_heads"] * s["head_dim"], s["n_kv_heads"] * s["head_dim"]
    per_weight = 1 + (4 if case["storage"] == "q8_0" else 2) / 32
    rows, answers = _rows(case, [0] * _n_tokens(case))
    weights = sum(n * k for l in range(case["layers"]) for n, k in _projections(case, l).values())
    n_att = sum(_is_attention(case, l) for l in range(case["layers"]))
    head = 0 if case["kind"] == "multi" else s["vocab_size"]

    def one_pass(rows, answers):
        scored = sum(slot - first + 1 + shared for _, _, slot, first, shared in rows)  # (row, position) pairs
        # keys and values that are in the cache before the pass are read once each, its own rows' written once
        read = sum(p for _, p, _, _, _ in rows) if case["kind"] == "batch" else _filled(case)
        out = answers * (head if head else s["dim"])
        nbytes = (weights + head * s["dim"]) * per_weight + len(rows) * s["dim"] * per_weight
        nbytes += n_att * (read + len(rows)) * 2 * kv * 4 + out * 4
        flops = 2 * len(rows) * weights + 2 * answers * head * s["dim"] + n_att * scored * 4 * q
        return nbytes, flops

    nbytes, flops = one_pass(rows, len(answers))
    if case["kind"] == "turn":
        at = case["start"] + case["prompt"]
        for i in range(case["steps"] + 1):
            b, f = one_pass([(0, at + i, at + i, 0, 0)], 1)
            nbytes += b + n_att * (at + i - _filled(case)) * 2 * kv * 4
            flops += f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # the path is specified to the bit (see the head of this file)
    return "exact"


# ---- inputs --------------------------------------------------------------------


class _Inputs:
    """The weights, cache and tokens of (case, seed), drawn on the GPU in a fixed order."""

    def __init__(self, case, seed):
        self.case, self.shape = case, SHAPES[case["model"]]
        self.gen = torch.Generator(device="cuda").manual_seed(seed)
        g = np.random.default_rng(seed)
        self.tokens = [int(t) for t in g.integers(0, self.shape["vocab_size"], _n_tokens(case))]
        d = self.shape["dim"]
        self.norm_final = self.normal(d).mul_(0.1).add_(1)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.gen, device="cuda")

    def matrix(self, n, k):
        """N(0, 0.02) weights as Q8: int8 [n, k] and f32 block scales [n, k / 32] (representable
        in f16 for the packed storage)."""
        w = self.normal(n, k // 32, 32).mul_(0.02)
        d = w.abs().amax(2) / 127
        q = (w / d[..., None]).round_().clamp_(-127, 127).to(torch.int8)
        return q.view(n, k), d.half().float() if self.case["storage"] == "q8_0x4" else d

    def layer(self, l):
        s, hs = self.shape, self.shape["head_dim"]
        out = {"att": self.normal(s["dim"]).mul_(0.1).add_(1), "ffn": self.normal(s["dim"]).mul_(0.1).add_(1)}
        if _is_attention(self.case, l):
            if s["qk_norm"]:
                out["qn"], out["kn"] = (self.normal(hs).mul_(0.1).add_(1) for _ in range(2))
        else:
            out["conv"] = self.normal(s["dim"], CONV_K).mul_(0.5)
        out["proj"] = {name: self.matrix(n, k) for name, (n, k) in _projections(self.case, l).items()}
        return out

    def cache(self, l):
        """The layer's filled keys and values, f32 [slots, kv_dim] each."""
        kv = self.shape["n_kv_heads"] * self.shape["head_dim"]
        return self.normal(_filled(self.case), kv), self.normal(_filled(self.case), kv)


def _np(t):
    return t.cpu().numpy()


def _q8(storage, m):
    q, s = m
    n, k = q.shape
    if storage == "q8_0":
        return K.Q8Matrix("q8_0", n, k, quants=_np(q), scales=_np(s))
    # 136-byte records of 4 rows: f16 scales [4], then quants [8 segments][4 rows][4]
    g, nb = n // 4, k // 32
    rec = torch.empty(g, nb, 136, dtype=torch.uint8, device=q.device)
    rec[:, :, :8] = s.half().view(g, 4, nb).transpose(1, 2).contiguous().view(torch.uint8).view(g, nb, 8)
    rec[:, :, 8:] = q.view(g, 4, nb, 8, 4).permute(0, 2, 3, 1, 4).reshape(g, nb, 128).view(torch.uint8)
    return K.Q8Matrix("q8_0x4", n, k, blocks=_np(rec).ravel())


class _State:
    def __init__(self, case, seed):
        self.case = case
        x = _Inputs(case, seed)
        s, storage = x.shape, case["storage"]
        self.tokens = x.tokens
        self.config = K.Config(s["dim"], s["hidden_dim"], case["layers"], s["n_heads"], s["n_kv_heads"],
                               s["vocab_size"], _slots_total(case), s["rms_eps"], s["rope_theta"], False,
                               s["head_dim"])
        self.hip = hip = K.open("hip")
        handles, layers, caches = [], [], []
        for l in range(case["layers"]):
            w = x.layer(l)
            handles.append({name: hip.upload_matrix(_q8(storage, m)) for name, m in w["proj"].items()})
            layers.append(K.LayerWeights(*(None if w.get(k) is None else _np(w[k]) for k in ("att", "ffn")),
                                         rms_q=None if "qn" not in w else _np(w["qn"]),
                                         rms_k=None if "kn" not in w else _np(w["kn"]),
                                         conv_kernel=None if "conv" not in w else _np(w["conv"]),
                                         is_attention=_is_attention(case, l)))
            if _filled(case):
                caches.append(x.cache(l))
        embedding = hip.upload_matrix(_q8(storage, x.matrix(s["vocab_size"], s["dim"])))
        hip.bind_handles(embedding, 0xFFFFFFFF, handles)
        self.model = None
        if case["kind"] == "ops":
            self._prepare_ops(x, layers)
        else:
            self.model = K.Model(self.config, hip, None, lfm2=case["model"] == "lfm2-700m", layers=layers,
                                 rms_final=_np(x.norm_final))
        for l, (k, v) in enumerate(caches):
            at = l * self.config.seq_len * self.config.kv_dim
            hip.kv_upload(0, at, _np(k))
            hip.kv_upload(1, at, _np(v))
        hip.synchronize()

    def _prepare_ops(self, x, layers):
        """A driver's own buffers: the embedded rows, the norms and the activations."""
        c, hip, rows = self.config, self.hip, self.case["rows"]
        hip.prepare(None, K.KvSpec(c.n_layers, c.kv_dim, c.seq_len))
        self.norms = [(hip.upload(lw.rms_att), hip.upload(lw.rms_ffn)) for lw in layers]
        self.qk = [None if lw.rms_q is None else (hip.upload(lw.rms_q), hip.upload(lw.rms_k)) for lw in layers]
        self.norm_final = hip.upload(_np(x.norm_final))
        self.buf = {n: hip.alloc(rows * w) for n, w in dict(
            x0=c.dim, x=c.dim, xb=c.dim, q=c.q_dim, k=c.kv_dim, v=c.kv_dim, attn=c.q_dim, o=c.dim,
            gate=c.hidden_dim, up=c.hidden_dim, att=c.n_heads * c.seq_len).items()}
        self.logits = hip.alloc(c.vocab_size)
        for r, t in enumerate(self.tokens):
            hip.embed(t, self.buf["x0"], r * c.dim)
        at = range(self.case["start"], self.case["start"] + rows)
        self.positions = np.array(at, np.uint64)
        self.windows = [K.Window(0, p) for p in at]
        self.rope = K.RopeSpec(c.head_dim, c.rope_theta, False)
        self.attn = K.AttnSpec(c.n_heads, c.kv_mul, c.head_dim, c.kv_dim, c.seq_len)

    def run_ops(self):
        c, h, b, n = self.config, self.hip, self.buf, self.case["rows"]
        h.copy(b["x0"], 0, b["x"], 0, n * c.dim)
        for l in range(c.n_layers):
            h.rms_norm(b["xb"], b["x"], self.norms[l][0], n, c.dim, c.rms_eps)
            h.project_qkv(l, b["xb"], b["q"], b["k"], b["v"], n)
            if self.qk[l]:
                h.qk_norm(b["q"], n, c.q_dim, c.head_dim, self.qk[l][0], c.rms_eps)
                h.qk_norm(b["k"], n, c.kv_dim, c.head_dim, self.qk[l][1], c.rms_eps)
            h.rope(b["q"], b["k"], c.q_dim, c.kv_dim, n, self.positions, self.rope)
            h.kv_write(l, self.positions, b["k"], b["v"], n)
            h.attention(b["q"], b["attn"], b["att"], l, self.windows, self.attn)
            h.project(l, "o", b["attn"], b["o"], n)
            h.add_in_place(b["x"], b["o"], n * c.dim)
            h.rms_norm(b["xb"], b["x"], self.norms[l][1], n, c.dim, c.rms_eps)
            h.project_gate_up(l, b["xb"], b["gate"], b["up"], n)
            h.silu_mul(b["gate"], b["up"], n * c.hidden_dim)
            h.project(l, "down", b["gate"], b["o"], n)
            h.add_in_place(b["x"], b["o"], n * c.dim)
        h.copy(b["x"], (n - 1) * c.dim, b["xb"], 0, c.dim)
        h.rms_norm(b["o"], b["xb"], self.norm_final, 1, c.dim, c.rms_eps)
        h.logits(b["o"], self.logits)
        return h.read(self.logits, c.vocab_size)


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    case, model, kind = state.case, state.model, state.case["kind"]
    if kind == "ops":
        return state.run_ops()
    if kind == "forward":
        return model.forward(state.tokens[0], case["pos"])
    if kind == "prefill":
        return model.prefill(state.tokens, case["start"])
    if kind == "multi":
        ends = np.cumsum([case["shared"]] + _lens(case))
        seqs = [state.tokens[a:b] for a, b in zip(ends, ends[1:])]
        if case["shared"]:
            return model.prefill_shared(state.tokens[:case["shared"]], seqs)
        return model.prefill_multi(seqs)
    if kind == "batch":
        at, c = np.array(_positions(case)), case["context"]
        first = np.arange(case["n_seq"]) * c
        return model.decode_batch(state.tokens, at, first + at, first)
    logits = model.prefill(state.tokens, case["start"])
    at = case["start"] + case["prompt"]
    tokens = model.generate_greedy(int(np.argmax(logits)), at, case["steps"])
    return logits, tokens.astype(np.int64), model.forward(int(tokens[-1]), at + case["steps"])


# ---- the same in 64 bits -------------------------------------------------------


def _quantized(x, half_scales):
    """Rows of x as their Q8 values: the quantization is part of the path's definition."""
    x = x.float().view(x.shape[0], -1, 32)
    d = x.abs().amax(2, keepdim=True) / 127
    v = x * torch.where(d > 0, 1 / d, torch.zeros_like(d))
    q = (v.abs() + 0.5).floor().clamp(max=127) * v.sign()
    return (q.double() * (d.half() if half_scales else d).double()).flatten(1)


def _times(x, m, half_scales):
    q, s = m
    w = (q.view(q.shape[0], -1, 32).double() * s.double()[..., None]).flatten(1)
    return _quantized(x, half_scales) @ w.t()


def _rms(x, w, eps):
    return x / (x.square().mean(-1, keepdim=True) + eps).sqrt() * w.double()


def _rotate(x, pos, heads, hs, theta):
    """The half-split RoPE; the angles are f32 by definition."""
    power = np.float64(theta) ** (np.arange(0, hs, 2, dtype=np.float32) / np.float32(hs)).astype(np.float64)
    freq = torch.from_numpy(np.float32(1) / power.astype(np.float32)).cuda()
    a = (pos.float()[:, None] * freq).double()
    c, s = a.cos()[:, None], a.sin()[:, None]
    x = x.view(-1, heads, hs)
    p, r = x[..., :hs // 2], x[..., hs // 2:]
    return torch.cat([p * c - r * s, p * s + r * c], -1).flatten(1)


def _attend(q, k, v, mask, s):
    hs, mul = s["head_dim"], s["n_heads"] // s["n_kv_heads"]
    out = []
    for h in range(s["n_heads"]):
        at = slice(h // mul * hs, (h // mul + 1) * hs)
        p = (q[:, h * hs:(h + 1) * hs] @ k[:, at].t()) / math.sqrt(hs)
        out.append(p.masked_fill(~mask, -math.inf).softmax(1) @ v[:, at])
    return torch.cat(out, 1)


def exact(case, seed):
    """The call in 64 bits, with the activations' quantization as the path defines it. A value that
    falls on the other side of a rounding step moves by a whole one and moves others after it: over
    many layers the two part by a few hundredths, the size of the quantization itself."""
    x_in = _Inputs(case, seed)
    s, half = x_in.shape, case["storage"] == "q8_0x4"
    rows, answers = _rows(case, x_in.tokens)
    pos, slot, first, shared = (torch.tensor([r[i] for r in rows], device="cuda") for i in (1, 2, 3, 4))
    slots = torch.arange(int(slot.max()) + 1, device="cuda")[None]
    mask = ((slots >= first[:, None]) & (slots <= slot[:, None])) | (slots < shared[:, None])
    layers = []
    for l in range(case["layers"]):
        w = x_in.layer(l)
        layers.append((w, x_in.cache(l) if _filled(case) else None))
    embedding = x_in.matrix(s["vocab_size"], s["dim"])
    ids = torch.tensor([r[0] for r in rows], device="cuda")
    x = (embedding[0][ids].view(len(rows), -1, 32).double() * embedding[1][ids].double()[..., None]).flatten(1)
    for w, cache in layers:
        p = w["proj"]
        b = _rms(x, w["att"], s["rms_eps"])
        if "q" in p:
            q, k, v = (_times(b, p[n], half) for n in ("q", "k", "v"))
            if "qn" in w:
                q, k = (_rms(t.view(len(rows), -1, s["head_dim"]), n, s["rms_eps"]).flatten(1)
                        for t, n in ((q, w["qn"]), (k, w["kn"])))
            q = _rotate(q, pos, s["n_heads"], s["head_dim"], s["rope_theta"])
            k = _rotate(k, pos, s["n_kv_heads"], s["head_dim"], s["rope_theta"])
            kc, vc = (torch.zeros(slots.shape[1], k.shape[1], dtype=torch.float64, device="cuda") for _ in range(2))
            if cache is not None:
                n = min(len(kc), len(cache[0]))
                kc[:n], vc[:n] = cache[0][:n].double(), cache[1][:n].double()
            kc[slot], vc[slot] = k, v
            x = x + _times(_attend(q, kc, vc, mask, s), p["o"], half)
        else:
            d = s["dim"]
            t = _times(b, p["conv_in"], half)
            h = torch.cat([torch.zeros(CONV_K - 1, d, dtype=torch.float64, device="cuda"), t[:, :d] * t[:, 2 * d:]])
            conv = sum(h[j:j + len(rows)] * w["conv"][:, j].double() for j in range(CONV_K))
            x = x + _times(t[:, d:2 * d] * conv, p["conv_out"], half)
        b = _rms(x, w["ffn"], s["rms_eps"])
        g = _times(b, p["gate"], half)
        x = x + _times(g * g.sigmoid() * _times(b, p["up"], half), p["down"], half)
    x = _rms(x[torch.tensor(answers, device="cuda")], x_in.norm_final, s["rms_eps"])
    if case["kind"] == "multi":
        return _np(x)
    logits = _np(_times(x, embedding, False))
    if case["kind"] == "turn":  # the tokens that follow hang on near ties of the logits
        return logits[0], None, None
    return logits if case["kind"] == "batch" else logits[0]
