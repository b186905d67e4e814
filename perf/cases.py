"""The calls that the encoder backend is timed on.

A case is one call as a serving or indexing program makes it: token rows in
through a session's public methods (embed, a range write, rerank, QA span
logits), vectors or scores out on the host. The model and the session are
what such a program keeps from call to call; the rows are the call's own.

The widths are those of the workloads in turboembed_amd/workloads.py. Three
things are cut so that a case can be made quickly: the vocabulary to 30522
rows, the depth to the `layers` a case names (the two calls over a whole
encoder at BERT-base width and both MiniLM ones keep it), and the weights
are random: N(0, 0.55 / sqrt(hidden)), so 0.02 at width 768, with norms about 1.

A row's lengths are spread evenly over [lo, hi], and dealt to the rows by the
seed where the results' shapes do not follow them, so every seed has the
same work. `cap_rows` x `cap_seq` is the size
the session was opened at, as a server opens one for its largest batch.
"""
import math

import numpy as np
import torch

import turboembed_amd as T
from turboembed_amd import seam as S
from turboembed_amd.model import ModelDesc
from turboembed_amd.rerank import RerankHead

VOCAB = 30522

# family, hidden, heads, FFN width, positions, [CLS], [SEP], padding, eps
MODELS = {
    "minilm": ("bert", 384, 12, 1536, 512, 101, 102, 0, 1e-12),
    "bert-base": ("bert", 768, 12, 3072, 512, 101, 102, 0, 1e-12),
    "xlmr-large": ("roberta", 1024, 16, 4096, 8194, 0, 2, 1, 1e-5),
    "modernbert": ("modernbert", 768, 12, 1152, 8192, 101, 102, 0, 1e-5),
    "deberta-v3-base": ("deberta", 768, 12, 3072, 512, 1, 2, 0, 1e-7),
}
BUCKETS, FARTHEST = 256, 512             # DeBERTa's relative rows
THETA, WINDOW, EVERY = (160000.0, 10000.0), 128, 3   # ModernBERT's rotary bases, window, global layers

TIERS = {"f32": S.TURBO_PRECISION_EXACT, "f16": S.TURBO_PRECISION_FASTEST, "bf16": S.TURBO_PRECISION_MODEL,
         "int8": S.TURBO_PRECISION_FASTEST}


def _case(name, model, tier, layers, op, rows, lo, hi, cap_rows, cap_seq, ranges=0):
    c = dict(model=model, tier=tier, layers=layers, op=op, rows=rows, lo=lo, hi=hi, cap_rows=cap_rows,
             cap_seq=cap_seq, ranges=ranges)
    return dict(c, name=name) if name else c


def listed():
    return [
        # A search box's query in the exact tier: one short row, where launches and copies count.
        _case("minilm-f32-query", "minilm", "f32", 6, "mean", 1, 16, 16, 32, 128),
        # The repository's exact-tier batch of sentences.
        _case("minilm-f32-batch", "minilm", "f32", 6, "mean", 32, 16, 128, 32, 128),
        # Passages indexed with a small 16-bit model (heads of 32).
        _case("minilm-f16-batch", "minilm", "f16", 6, "mean", 128, 32, 256, 128, 256),
        # One query through a whole BERT-base in the fastest tier, on a session opened for batches.
        _case("bert-base-f16-query", "bert-base", "f16", 12, "cls", 1, 24, 24, 64, 512),
        # A server's small dynamic batch of queries and sentences.
        _case("bert-base-f16-online", "bert-base", "f16", 4, "mean", 12, 9, 96, 64, 512),
        # The headline batch: a whole BERT-base over full rows.
        _case("bert-base-f16-bulk", "bert-base", "f16", 12, "cls", 64, 512, 512, 64, 512),
        # Exact-tier embeddings at BERT-base width.
        _case("bert-base-f32-batch", "bert-base", "f32", 2, "mean", 24, 33, 300, 32, 512),
        # Extractive QA over a document's windows: start and end logits of every token.
        _case("bert-base-f16-qa", "bert-base", "f16", 4, "qa", 16, 300, 384, 16, 384),
        # Late chunking of long documents: 64 range vectors a row.
        _case("xlmr-large-bf16-chunks", "xlmr-large", "bf16", 2, "ranges", 8, 1024, 4096, 8, 4096, ranges=64),
        # Long documents with sliding windows: two global layers of four.
        _case("modernbert-f16-long", "modernbert", "f16", 4, "mean", 16, 2048, 8192, 16, 8192),
        # Reranking a first stage's hits in the int8 tier: passages of 64 to 480 tokens behind short queries.
        _case("rerank-int8-pairs", "bert-base", "int8", 3, "rerank", 128, 64, 480, 128, 512),
        # Relative attention over passages.
        _case("deberta-f16-bulk", "deberta-v3-base", "f16", 3, "mean", 64, 128, 512, 64, 512),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


# (model, tier, layers, op, most rows, longest row, most tokens)
_KINDS = [
    ("minilm", "f32", 6, "mean", 64, 256, 8192),
    ("minilm", "f16", 6, "mean", 256, 512, 65536),
    ("bert-base", "f16", 4, "mean", 128, 512, 65536),
    ("bert-base", "f16", 12, "cls", 64, 512, 32768),
    ("bert-base", "f32", 2, "mean", 64, 512, 8192),
    ("bert-base", "f16", 4, "qa", 32, 512, 12288),
    ("xlmr-large", "bf16", 2, "ranges", 16, 8192, 32768),
    ("modernbert", "f16", 4, "mean", 64, 8192, 49152),
    ("bert-base", "int8", 3, "rerank", 128, 480, 65536),
    ("deberta-v3-base", "f16", 3, "mean", 64, 512, 32768),
]


def draw(rng):
    """One more case: any of the kinds above, rows and lengths log-uniform
    over what its model takes, from one short row up."""
    model, tier, layers, op, most, longest, tokens = rng.choice(_KINDS)
    hi = _log(rng, 8, longest)
    lo = max(1 if op != "rerank" else 4, int(hi * rng.choice([0.12, 0.5, 1.0])))
    rows = _log(rng, 1, min(most, max(1, tokens // hi)))
    ranges = rng.randint(1, min(64, lo)) if op == "ranges" else 0
    # A session opened for the batch itself, or for a larger one.
    cap_rows = min(most, rows * rng.choice([1, 2, 4]))
    room = 36 if op == "rerank" else 0
    cap_seq = min(MODELS[model][4] if model != "xlmr-large" else 8192, (hi + room) * rng.choice([1, 2]))
    return _case("", model, tier, layers, op, rows, lo, hi, cap_rows, cap_seq, ranges)


# ---- what a program has in hand before the call -------------------------------------

def _weights(case, seed):
    """The model's tensors on the GPU in the stored type, in the order the
    model description takes them."""
    fam, H, _, I, positions, _, _, _, _ = MODELS[case["model"]]
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 + seed)
    kind = torch.bfloat16 if case["tier"] == "bf16" else torch.float32
    std = 0.55 / math.sqrt(H)

    def w(*shape):
        return (torch.randn(*shape, generator=g, device="cuda") * std).to(kind)

    def norm():
        return (1 + 0.1 * torch.randn(H, generator=g, device="cuda")).to(kind)

    if fam == "modernbert":
        t = [w(VOCAB, H), norm(), norm()]
        for layer in range(case["layers"]):
            t += [None if layer == 0 else norm(), w(3 * H, H), w(H, H), norm(), w(2 * I, H), w(H, I)]
        return t
    if fam == "deberta":
        t = [w(VOCAB, H), norm(), w(H), w(2 * BUCKETS, H), norm(), w(H)]
    else:
        t = [w(VOCAB, H), w(positions, H), w(2 if fam == "bert" else 1, H), norm(), w(H)]
    for _ in range(case["layers"]):
        t += [w(H, H), w(H), w(H, H), w(H), w(H, H), w(H), w(H, H), w(H), norm(), w(H),
              w(I, H), w(I), w(H, I), w(H), norm(), w(H)]
    return t


def _heads(case, seed):
    """QA's span head, or the cross-encoder's pooler and classifier."""
    H = MODELS[case["model"]][1]
    g = np.random.Generator(np.random.PCG64([7, seed]))
    f = lambda *s: (g.standard_normal(s, dtype=np.float32) * np.float32(0.02))  # noqa: E731
    if case["op"] == "qa":
        return f(2, H), f(2)
    if case["op"] == "rerank":
        return f(H, H), f(H), f(H), 0.125
    return None


def _lengths(case, seed):
    n = np.rint(np.linspace(case["lo"], case["hi"], case["rows"])).astype(int)
    if case["op"] in ("qa", "rerank"):
        return n
    return np.random.Generator(np.random.PCG64([11, seed])).permutation(n)


def _tokens(case, seed):
    """The rows' token ids, one array a row; a pair for a rerank."""
    _, _, _, _, _, cls, sep, _, _ = MODELS[case["model"]]
    g = np.random.Generator(np.random.PCG64([13, seed]))
    out = []
    for i, n in enumerate(_lengths(case, seed)):
        body = g.integers(1000, VOCAB, size=n).astype(np.int32)
        if case["op"] == "rerank":
            out.append((g.integers(1000, VOCAB, size=4 + i * 7 % 29).astype(np.int32), body))
            continue
        body[0] = cls
        if n > 1:
            body[-1] = sep
        out.append(body)
    return out


def _ranges(case, seed):
    """Each row cut into case["ranges"] pieces."""
    g = np.random.Generator(np.random.PCG64([17, seed]))
    out = []
    for r, n in enumerate(_lengths(case, seed)):
        cuts = np.sort(g.choice(np.arange(1, n), size=case["ranges"] - 1, replace=False)) if n > 1 else []
        edges = [0] + [int(c) for c in cuts] + [int(n)]
        out += [(r, a, b) for a, b in zip(edges, edges[1:])]
    return out


_context = None


class State:
    """A loaded model, its open session and one call's rows."""

    def __init__(self, case, seed):
        global _context
        fam, H, heads, I, positions, _, _, pad, eps = MODELS[case["model"]]
        if _context is None:
            _context = T.Runtime().context(0)

        def host(t):
            if t is None:
                return None
            if t.dtype == torch.bfloat16:
                return t.view(torch.int16).cpu().numpy().view(np.uint16)
            return t.cpu().numpy()

        head = _heads(case, seed)
        family = {"bert": S.TURBO_FAMILY_BERT, "roberta": S.TURBO_FAMILY_ROBERTA,
                  "modernbert": S.TURBO_FAMILY_MODERNBERT, "deberta": S.TURBO_FAMILY_DEBERTA_V2}[fam]
        more = {}
        if fam == "modernbert":
            more = dict(rope=THETA, attention_window=WINDOW, global_every=EVERY, mlp=S.TURBO_MLP_GATED,
                        activation=S.TURBO_ACTIVATION_GELU_ERF, norm=S.TURBO_NORM_LAYER_NO_BIAS)
        if fam == "deberta":
            more = dict(relative=(BUCKETS, FARTHEST))
        if fam == "roberta":
            more = dict(position_offset=2)
        if case["tier"] == "int8":
            more["compute_dtype"] = S.TURBO_DTYPE_I8
        if case["op"] == "qa":
            more["span_head"] = head
        desc = ModelDesc(family, case["layers"], H, heads, I, VOCAB, positions, 2 if fam == "bert" else 1, eps,
                         [host(t) for t in _weights(case, seed)], **more)
        self.op = case["op"]
        self.model = _context.load(desc)
        task = {"qa": S.TURBO_TASK_EXTRACTIVE_QA, "rerank": S.TURBO_TASK_RERANK}.get(self.op, S.TURBO_TASK_EMBED)
        self.session = self.model.session(case["cap_rows"], case["cap_seq"], TIERS[case["tier"]], task=task,
                                          max_ranges=case["cap_rows"] * case["ranges"])
        rows = _tokens(case, seed)
        self.cls, self.sep = MODELS[case["model"]][5:7]
        if self.op == "rerank":
            self.pairs = rows
            self.head = RerankHead(head[2], head[3], head[0], head[1])
            return
        if self.op == "qa":
            self.windows = [(r, (np.arange(len(r)) > len(r) // 8).astype(np.int32)) for r in rows]
            return
        seq = max(len(r) for r in rows)
        self.ids = np.full((len(rows), seq), pad, np.int32)
        self.mask = np.zeros_like(self.ids)
        self.types = np.zeros_like(self.ids)
        for i, r in enumerate(rows):
            self.ids[i, :len(r)] = r
            self.mask[i, :len(r)] = 1
        self.ranges = _ranges(case, seed) if self.op == "ranges" else None

    def __del__(self):
        for what in ("session", "model"):
            if hasattr(self, what):
                getattr(self, what).close()


def prepare(case, seed):
    return State(case, seed)


def run(state):
    s = state.session
    if state.op == "rerank":
        return s.rerank(state.pairs, state.head, state.cls, state.sep, query_tokens=32)
    if state.op == "qa":
        return s.span_logits(state.windows)
    if state.op == "ranges":
        s.write_ranges(state.ids, state.mask, state.ranges, state.types)
        s.run()
        return s.read()
    return s.embed(state.ids, state.mask, state.types,
                   pooling=S.TURBO_POOLING_CLS if state.op == "cls" else S.TURBO_POOLING_MEAN)


def _token_counts(case):
    n = [int(v) for v in np.rint(np.linspace(case["lo"], case["hi"], case["rows"]))]
    return [v + 3 + 4 + i * 7 % 29 for i, v in enumerate(n)] if case["op"] == "rerank" else n


def work(case):
    """The encoder's products and attention over live tokens; the weights of
    the layers, the live tokens' embedding rows, ids, mask and types read
    once and the output written once."""
    fam, H, _, I, _, _, _, _, _ = MODELS[case["model"]]
    lens, L = _token_counts(case), case["layers"]
    tokens = sum(lens)
    per_layer = H * (3 * H + H + (3 if fam == "modernbert" else 2) * I)
    flops = 2.0 * tokens * L * per_layer
    for n in lens:
        if fam == "modernbert":
            near = sum(min(n, i + WINDOW // 2 + 1) - max(0, i - WINDOW // 2) for i in range(n))
            glob = len(range(0, L, EVERY))
            flops += 4.0 * H * (glob * n * n + (L - glob) * near)
        else:
            flops += (8.0 if fam == "deberta" else 4.0) * H * L * n * n
    el = {"f32": 4, "f16": 2, "bf16": 2, "int8": 1}[case["tier"]]
    out = {"qa": 2 * tokens, "rerank": len(lens), "ranges": case["rows"] * case["ranges"] * H}.get(case["op"],
                                                                                                  case["rows"] * H)
    if case["op"] == "rerank":
        flops += 2.0 * len(lens) * H * (H + 1)
    emb = 4 if case["tier"] != "bf16" else 2
    return {"bytes": float(L * per_layer * el + tokens * (H * emb + 12) + 4 * out), "flops": flops}


def tolerance(case):
    """About four times the distance from the results in 64 bits (f32 tier
    2e-7 to 4e-7 on means, more on single tokens; f16 3e-4 on means, 1.1e-3
    on CLS rows after 12 layers; bf16 6e-4 on ranges of many tokens, 8 times
    f16's on single ones; int8 1.1e-2 on scores, a changed rounding moving
    single codes)."""
    return {"f32": {"rel": 1e-5}, "f16": {"rel": 4e-3}, "bf16": {"rel": 1e-2}, "int8": {"rel": 2e-2}}[case["tier"]]


# ---- the same in 64 bits ------------------------------------------------------------

def _norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    x = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w
    return x if b is None else x + b


def _rotate(x, theta):
    """x [heads, n, d], rotated by its columns' halves."""
    d, n = x.shape[-1], x.shape[1]
    inv = theta ** (-torch.arange(0, d, 2, device="cuda", dtype=torch.float64) / d)
    a = torch.arange(n, device="cuda", dtype=torch.float64)[:, None] * inv
    cos, sin = torch.cat([a.cos()] * 2, -1), torch.cat([a.sin()] * 2, -1)
    return x * cos + torch.cat([-x[..., d // 2:], x[..., :d // 2]], -1) * sin


def _bucket_index(n):
    """Relative row of i - j, [n, n]."""
    mid = BUCKETS // 2
    r = np.arange(n)[:, None] - np.arange(n)[None, :]
    a = np.maximum(np.abs(r), mid).astype(np.float32) / np.float32(mid)
    far = np.ceil(np.log(a) / np.log(np.float32(FARTHEST - 1) / np.float32(mid)) * np.float32(mid - 1)) + mid
    r = np.where(np.abs(r) <= mid, r, np.sign(r) * far).astype(np.int64)
    return torch.from_numpy(np.clip(r + BUCKETS, 0, 2 * BUCKETS - 1)).cuda()


def _split(x, heads):
    return x.reshape(x.shape[0], heads, -1).transpose(0, 1).contiguous()


def _attend(q, k, v, rel=None, window=None):
    """One row's heads [heads, n, d], a few at a time."""
    heads, n, d = q.shape
    out = []
    few = max(1, min(heads, int(2e8) // (n * n)))
    for h in range(0, heads, few):
        s = torch.bmm(q[h:h + few], k[h:h + few].transpose(1, 2).contiguous())
        if rel is not None:
            index, pk, pq = rel
            ix = index.expand(s.shape[0], -1, -1)
            s += torch.gather(torch.bmm(q[h:h + few], pk[h:h + few].transpose(1, 2).contiguous()), 2, ix)
            s += torch.gather(torch.bmm(k[h:h + few], pq[h:h + few].transpose(1, 2).contiguous()), 2,
                              ix.transpose(1, 2).contiguous()).transpose(1, 2)
        s /= math.sqrt((1 if rel is None else 3) * d)
        if window is not None:
            i = torch.arange(n, device="cuda")
            s.masked_fill_((i[:, None] - i[None, :]).abs() > window, -math.inf)
        out.append(torch.bmm(torch.softmax(s, -1), v[h:h + few]))
        del s
    return torch.cat(out).transpose(0, 1).reshape(n, heads * d)


def _states(case, t, ids, types):
    """Final states of one row of live tokens."""
    fam, H, heads, I, _, _, _, _, eps = MODELS[case["model"]]
    n = len(ids)
    ids = torch.from_numpy(ids.astype(np.int64)).cuda()
    gelu = torch.nn.functional.gelu
    if fam == "modernbert":
        x = _norm(t[0][ids], t[1], None, eps)
        for layer in range(case["layers"]):
            n1, wqkv, wo, n2, wi, wd = t[3 + 6 * layer:9 + 6 * layer]
            whole = layer % EVERY == 0
            y = (x if n1 is None else _norm(x, n1, None, eps)) @ wqkv.T
            q, k, v = (_split(y[:, i * H:(i + 1) * H], heads) for i in range(3))
            theta = THETA[0 if whole else 1]
            x = x + _attend(_rotate(q, theta), _rotate(k, theta), v, None, None if whole else WINDOW // 2) @ wo.T
            y = _norm(x, n2, None, eps) @ wi.T
            x = x + (gelu(y[:, :I]) * y[:, I:]) @ wd.T
        return _norm(x, t[2], None, eps)
    rel = None
    if fam == "deberta":
        x = _norm(t[0][ids], t[1], t[2], eps)
        rows, index, at = _norm(t[3], t[4], t[5], eps), _bucket_index(n), 6
    else:
        first = 2 if fam == "roberta" else 0
        x = t[0][ids] + t[1][first:first + n] + t[2][torch.from_numpy(types.astype(np.int64)).cuda()]
        x, at = _norm(x, t[3], t[4], eps), 5
    for layer in range(case["layers"]):
        wq, bq, wk, bk, wv, bv, wo, bo, n1, c1, wi, bi, wd, bd, n2, c2 = t[at + 16 * layer:at + 16 + 16 * layer]
        q, k, v = (_split(x @ w.T + b, heads) for w, b in ((wq, bq), (wk, bk), (wv, bv)))
        if fam == "deberta":
            rel = (index, _split(rows @ wk.T + bk, heads), _split(rows @ wq.T + bq, heads))
        x = _norm(x + _attend(q, k, v, rel) @ wo.T + bo, n1, c1, eps)
        x = _norm(x + gelu(x @ wi.T + bi) @ wd.T + bd, n2, c2, eps)
    return x


def exact(case, seed):
    t = [None if w is None else w.double() for w in _weights(case, seed)]
    head = _heads(case, seed)
    _, _, _, _, _, cls, sep, _, _ = MODELS[case["model"]]
    cut = _ranges(case, seed) if case["op"] == "ranges" else None
    out = []
    for r, row in enumerate(_tokens(case, seed)):
        types = np.zeros(len(row), np.int32)
        if case["op"] == "rerank":
            q, p = row
            row = np.concatenate([[cls], q, [sep], p, [sep]])
            types = (np.arange(len(row)) >= len(q) + 2).astype(np.int32)
        if case["op"] == "qa":
            types = (np.arange(len(row)) > len(row) // 8).astype(np.int32)
        x = _states(case, t, row, types)
        if case["op"] == "rerank":
            pw, pb, cw, cb = (torch.as_tensor(h, dtype=torch.float64, device="cuda") for h in head)
            out.append(torch.tanh(pw @ x[0] + pb) @ cw + cb)
            continue
        if case["op"] == "qa":
            w, b = (torch.as_tensor(h, dtype=torch.float64, device="cuda") for h in head)
            y = (x @ w.T + b).cpu().numpy()
            out.append((y[:, 0], y[:, 1]))
            continue
        vs = [x[a:b].mean(0) for at, a, b in cut if at == r] if cut else [x[0] if case["op"] == "cls" else x.mean(0)]
        out += [v / v.norm() for v in vs]
    return out if case["op"] == "qa" else torch.stack(out).cpu().numpy()
