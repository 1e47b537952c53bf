"""Work that programs give this framework, as cases that can be timed.

``listed()`` holds fixed cases and ``draw(rng)`` gives further ones of the same
ranges; ``prepare`` makes what a program has in hand before the call, ``run``
is one pass through the public entry points, ``exact`` the same results in 64
bits from plain torch.  Two directions are covered: verification and token by
token decoding (few rows over long caches: attention, linear layers,
normalisation, the captured decoder step) and the prompt (hundreds to
thousands of rows: causal attention chunks, linear layers, the element-wise
kernels of a prefill, the decoder's prefill).  All of it runs in bf16, the
only data type the framework builds; vocabulary scores and squares are fp32.

Kinds of a case:
  attn    fused_attn_hyb over a trie: prompt K/V, ``committed`` open node slots,
          then ``nodes`` trie nodes that see their ancestors
  chunk   fused_attn_hyb over ``rows`` prompt tokens, causal among themselves,
          after ``prompt`` earlier ones (a prefill chunk)
  linear  linear(x, w): ``rows`` x ``k`` by ``n`` x ``k``
  norm    one layer's RMSNorm + q/k norm + RoPE, and its SwiGLU product
  rows    one layer's element-wise work of a prefill, and a vision RoPE
  trie    verify_trie(graph=True): one captured decoder step over a trie
  token   forward_token(graph=True): one captured decoder step over one token
  prompt  Decoder.prefill of ``rows`` tokens
"""
import math
import random

import torch

from respect_amd.candidates.trie import build_trie
from respect_amd.decoding.engine import Decoder, DecoderConfig
from respect_amd.decoding.kv_buffer import KVCache
from respect_amd.decoding.sequential import forward_token
from respect_amd.decoding.verify import node_slots, verify_trie
from respect_amd.kernels.attention import fused_attn_hyb
from respect_amd.kernels.gemm import linear, tile_weight
from respect_amd.system.fused import (add_sq, norm_from, rmsnorm_qk_norm_rope, rope, rope_tables, rope_vision,
                                      silu_mul)

BF = torch.bfloat16
DEV = "cuda"
DEPTH = 24            # tokens of one candidate sequence
EPS = 1e-6
THETA = 1.0e6
VISION = (16, 80)     # heads and head_dim of the vision RoPE
HEADS_8B = {"heads": 32, "kv_heads": 8, "head_dim": 128}
WIDTHS_8B = {"hidden": 4096, "heads": 32, "kv_heads": 8, "ffn": 12288, "vocab": 151936}


def listed():
    return [
        # One layer's small element-wise kernels while a 64-node trie is verified: the
        # smallest calls, where the launch is most of the time.
        {"name": "norm_trie", "kind": "norm", "tokens": 64, "hidden": 4096, "ffn": 12288, **HEADS_8B},
        # The verification attention of a 64-node trie after a 3072-token prompt: the
        # headline call.
        {"name": "attn_trie", "kind": "attn", "prompt": 3072, "nodes": 64, "committed": 0, **HEADS_8B},
        # The same call some hundred committed tokens into an answer, with sizes that
        # end inside a tile.
        {"name": "attn_committed", "kind": "attn", "prompt": 3086, "nodes": 61, "committed": 437, **HEADS_8B},
        # The widest trie over the longest prompt.
        {"name": "attn_long", "kind": "attn", "prompt": 16384, "nodes": 128, "committed": 24, **HEADS_8B},
        # Attention of one 512-token prefill chunk late in a 3072-token prompt.
        {"name": "attn_chunk", "kind": "chunk", "prompt": 2560, "rows": 512, **HEADS_8B},
        # The gate projection of a model patched in place (row-major weights), 64 nodes.
        {"name": "linear_trie", "kind": "linear", "rows": 64, "n": 12288, "k": 4096, "weights": "rows", "out": "bf16"},
        # The down projection of one prefill chunk, weights laid out by tile_weight.
        {"name": "linear_chunk", "kind": "linear", "rows": 512, "n": 4096, "k": 12288, "weights": "tiled",
         "out": "bf16"},
        # A small decoder's up projection: 896 is no multiple of 256, the rows of no tile.
        {"name": "linear_odd", "kind": "linear", "rows": 77, "n": 4864, "k": 896, "weights": "rows", "out": "bf16"},
        # One layer's element-wise work over a 3072-token prompt.
        {"name": "rows_prompt", "kind": "rows", "rows": 3072, "hidden": 4096, "ffn": 12288, **HEADS_8B},
        # Plain decoding: one token through a captured decoder step.
        {"name": "step_token", "kind": "token", "layers": 24, "prompt": 3072, "committed": 37, **WIDTHS_8B},
        # Verification: a 64-node trie through a captured decoder step.
        {"name": "step_trie", "kind": "trie", "layers": 24, "prompt": 3072, "committed": 24, "nodes": 64,
         **WIDTHS_8B},
        # The prompt itself: 3072 tokens through the decoder.
        {"name": "prompt", "kind": "prompt", "layers": 4, "rows": 3072, **WIDTHS_8B},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn"] * 4 + ["linear"] * 4 + ["chunk", "norm", "rows", "token", "trie", "prompt"])
    if kind in ("attn", "chunk"):
        h, hk, d = rng.choice([(32, 8, 128)] * 3 + [(16, 8, 128), (32, 4, 128), (8, 2, 64), (16, 2, 64)])
        shape = {"heads": h, "kv_heads": hk, "head_dim": d}
        if kind == "attn":
            return {"kind": kind, "prompt": _log(rng, 64, 16384), "nodes": _log(rng, 1, 128),
                    "committed": rng.choice([0, _log(rng, 1, 600)]), **shape}
        return {"kind": kind, "prompt": rng.choice([0, _log(rng, 64, 8192)]), "rows": _log(rng, 65, 1024), **shape}
    if kind == "linear":
        step = rng.choice([256, 256, 64, 8, 1])
        n, k = (max(1, round(_log(rng, lo, 16384) / step)) * step for lo in (512, 256))
        tiled = k % 256 == 0 and n % 16 == 0 and rng.random() < 0.5
        return {"kind": kind, "rows": _log(rng, 1, 1024), "n": n, "k": k, "weights": "tiled" if tiled else "rows",
                "out": rng.choice(["bf16", "bf16", "fp32"])}
    hidden = rng.choice([1024, 2048, 4096])
    widths = {"hidden": hidden, "heads": hidden // 128, "kv_heads": max(2, hidden // 512), "ffn": 3 * hidden}
    if kind == "norm":
        return {"kind": kind, "tokens": _log(rng, 1, 512), "head_dim": 128, **widths}
    if kind == "rows":
        return {"kind": kind, "rows": _log(rng, 65, 3072), "head_dim": 128, **widths}
    widths["vocab"] = 151936
    if kind == "prompt":
        return {"kind": kind, "layers": rng.randint(1, 4), "rows": _log(rng, 65, 3072), **widths}
    case = {"kind": kind, "layers": _log(rng, 1, 24), "prompt": _log(rng, 64, 3072),
            "committed": rng.choice([0, _log(rng, 1, 300)]), **widths}
    if kind == "trie":
        case["nodes"] = _log(rng, 2, 64)
    return case


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * scale).to(BF)


def _candidates(seed, nodes):
    """Token sequences whose merged trie has ``nodes`` nodes, each sharing a prefix of at
    most 16 tokens with an earlier one, and the trie's parents and depths (nodes in the
    order of insertion)."""
    rng = random.Random(seed)
    tokens = rng.sample(range(30000), nodes)
    seqs, paths, parents, depths = [], [], [], []
    while len(parents) < nodes:
        path = []
        if paths:
            src = rng.choice(paths)
            path = src[:rng.randint(0, min(16, len(src) - 1))]
        while len(path) < DEPTH and len(parents) < nodes:
            parents.append(path[-1] if path else -1)
            depths.append(len(path))
            path = path + [len(parents) - 1]
        paths.append(path)
        seqs.append([tokens[i] for i in path])
    return seqs, tokens, parents, depths


def _trie_mask(parents, base, slots):
    """[nodes, slots] bool: ``base`` committed slots, then each node and its ancestors."""
    m = torch.zeros(len(parents), slots, dtype=torch.bool)
    m[:, :base] = True
    for i, p in enumerate(parents):
        if p >= 0:
            m[i, base:] = m[p, base:]
        m[i, base + i] = True
    return m


def _attn_inputs(case, seed):
    g = _gen(seed)
    H, HK, D, P = case["heads"], case["kv_heads"], case["head_dim"], case["prompt"]
    if case["kind"] == "attn":
        M, base = case["nodes"], case["committed"]
        NN = node_slots(base, M)
        msk = _trie_mask(_candidates(seed, M)[2], base, NN).to(DEV)
    else:
        M = case["rows"]
        NN = -(-M // 32) * 32
        msk = torch.ones(M, NN, dtype=torch.bool, device=DEV).tril()
    # Normalised q and k (unit elements; a score's scale is D ** -0.5) and v of unit scale.
    q = _randn(g, H, M, D)
    kp, vp, kn, vn = (_randn(g, HK, n, D) for n in (P, P, NN, NN))
    return [q, kp, vp, kn, vn, msk]


def _linear_inputs(case, seed):
    g = _gen(seed)
    return [_randn(g, case["rows"], case["k"]), _randn(g, case["n"], case["k"], scale=0.02)]


def _norm_inputs(case, seed):
    g = _gen(seed)
    T, n, D = case["tokens"], case["hidden"], case["head_dim"]
    x = _randn(g, T, n)
    q, k = (_randn(g, T, case[h], D) for h in ("heads", "kv_heads"))
    w, wq, wk = (1 + _randn(g, m, scale=0.02) for m in (n, D, D))
    cos, sin = rope_tables(torch.arange(T, device=DEV) + 3072, D, THETA, device=DEV)
    gu = _randn(g, T, 2 * case["ffn"])
    return [x, w, q, k, wq, wk, cos, sin, gu]


def _rows_inputs(case, seed):
    g = _gen(seed)
    L, n, D = case["rows"], case["hidden"], case["head_dim"]
    r, h = _randn(g, L, n), _randn(g, L, n)
    w = 1 + _randn(g, n, scale=0.02)
    # The projections leave heads inside a row: [1, L, heads, D], seen as [1, heads, L, D].
    q, k = (_randn(g, 1, L, case[m], D).transpose(1, 2) for m in ("heads", "kv_heads"))
    cos, sin = (t[None] for t in rope_tables(torch.arange(L, device=DEV), D, THETA, device=DEV))
    gate, up = _randn(g, L, case["ffn"]), _randn(g, L, case["ffn"])
    xv = _randn(g, L, *VISION)
    ang = torch.rand(L, VISION[1] // 2, generator=g, device=DEV) * 64
    ang = torch.cat((ang, ang), -1)
    return [r, h, w, q, k, cos, sin, gate, up, xv, ang.cos(), ang.sin()]


def _config(case):
    return DecoderConfig(layers=case["layers"], hidden=case["hidden"], heads=case["heads"],
                         kv_heads=case["kv_heads"], head_dim=128, ffn=case["ffn"], vocab=case["vocab"])


def _tokens(case, seed, n):
    return torch.randint(0, case["vocab"], (n,), generator=_gen(seed + 77), device=DEV)


def _cached(case, seed):
    """K and V rows, per layer, of the prompt and the committed tokens: normalised keys,
    values of the scale the projection gives."""
    g = _gen(seed + 99)
    n = case["prompt"] + case["committed"]
    for _ in range(case["layers"]):
        yield _randn(g, case["kv_heads"], n, 128), _randn(g, case["kv_heads"], n, 128)


class _Model:
    """A decoder, its cache and what one call of it is given."""

    def __init__(self, case, seed):
        self.model = Decoder(_config(case), device=DEV, seed=seed)
        self.kind = case["kind"]
        if self.kind == "prompt":
            self.cache = KVCache(case["layers"], case["kv_heads"], 128, case["rows"] + 64, device=DEV)
            self.ids = _tokens(case, seed, case["rows"])
            self.lo, self.hi = 0, case["rows"]
            return
        self.P, self.base = case["prompt"], case["committed"]
        nodes = case.get("nodes", 1)
        rows = 1 if self.kind == "token" else -(-nodes // 64) * 64
        width = node_slots(self.base, nodes, 64)
        self.cache = KVCache(case["layers"], case["kv_heads"], 128, self.P + width + rows + 64, device=DEV)
        n = self.P + self.base
        for i, (k, v) in enumerate(_cached(case, seed)):
            self.cache.k[i][:, :n] = k
            self.cache.v[i][:, :n] = v
        if self.kind == "token":
            self.token = int(_tokens(case, seed, 1))
        else:
            self.tree = build_trie(_candidates(seed, nodes)[0])
        self.lo, self.hi = n, n + nodes
        self.model.graphed(self.cache, self.P, rows, width)   # captured once, as a serving loop does

    def run(self):
        if self.kind == "prompt":
            logits = self.model.prefill(self.ids, self.cache)
        elif self.kind == "token":
            logits = forward_token(self.model, self.cache, self.token, self.P, self.base, graph=True)
        else:
            logits = verify_trie(self.model, self.cache, self.tree, self.P, self.base, graph=True)
        new = [t[:, self.lo:self.hi] for kv in (self.cache.k, self.cache.v) for t in kv]
        return [logits] + new


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("attn", "chunk"):
        return case, _attn_inputs(case, seed)
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        return case, [x, tile_weight(w) if case["weights"] == "tiled" else w]
    if kind == "norm":
        return case, _norm_inputs(case, seed)
    if kind == "rows":
        return case, _rows_inputs(case, seed)
    return case, _Model(case, seed)


# ------------------------------------------------------------------ one pass

def run(state):
    case, a = state
    kind = case["kind"]
    if kind in ("attn", "chunk"):
        return fused_attn_hyb(*a)
    if kind == "linear":
        return linear(*a, out_dtype=torch.float32 if case["out"] == "fp32" else None)
    if kind == "norm":
        x, w, q, k, wq, wk, cos, sin, gu = a
        y, qo, ko = rmsnorm_qk_norm_rope(x, w, EPS, q, k, wq, wk, EPS, cos, sin)
        F = case["ffn"]
        return [y, qo, ko, silu_mul(gu[:, :F], gu[:, F:])]
    if kind == "rows":
        r, h, w, q, k, cos, sin, gate, up, xv, cosv, sinv = a
        x, sq = add_sq(r, h)
        y = norm_from(x, sq, w, EPS)
        return [x, sq, y, rope(q, cos, sin), rope(k, cos, sin), silu_mul(gate, up), rope_vision(xv, cosv, sinv)]
    return a.run()


def work(case):
    kind = case["kind"]
    if kind in ("attn", "chunk"):
        H, HK, D, P = case["heads"], case["kv_heads"], case["head_dim"], case["prompt"]
        if kind == "attn":
            M, seen = case["nodes"], case["committed"] + case["nodes"]
            pairs = M * (P + case["committed"] + 12)     # about 12 ancestors a node
        else:
            M = seen = case["rows"]
            pairs = M * (P + (M + 1) / 2)
        return {"bytes": 4 * HK * D * (P + seen) + 4 * H * M * D + M * seen, "flops": 4 * H * D * pairs}
    if kind == "linear":
        M, N, K = case["rows"], case["n"], case["k"]
        return {"bytes": 2 * (M * K + N * K) + M * N * (4 if case["out"] == "fp32" else 2), "flops": 2 * M * N * K}
    if kind == "norm":
        T, n = case["tokens"], case["hidden"]
        heads = (case["heads"] + case["kv_heads"]) * case["head_dim"]
        return {"bytes": T * (4 * n + 4 * heads + 4 * case["head_dim"] + 6 * case["ffn"]),
                "flops": T * (4 * n + 7 * heads + 6 * case["ffn"])}
    if kind == "rows":
        L, n, V = case["rows"], case["hidden"], VISION[0] * VISION[1]
        heads = (case["heads"] + case["kv_heads"]) * case["head_dim"]
        # add_sq reads two and writes 2 + 4 bytes; norm_from reads x and the squares, writes y.
        return {"bytes": L * (18 * n + 4 * heads + 4 * case["head_dim"] + 6 * case["ffn"] + 4 * V + 8 * VISION[1]),
                "flops": L * (6 * n + 3 * heads + 6 * case["ffn"] + 3 * V)}
    H, F, layers = case["hidden"], case["ffn"], case["layers"]
    params = layers * (H * (2 * case["heads"] + 2 * case["kv_heads"]) * 128 + 3 * H * F)
    head = case["vocab"] * H
    kv = layers * case["kv_heads"] * 128 * 4      # bytes a cached token holds
    if kind == "prompt":
        n = case["rows"]
        return {"bytes": 2 * (params + head) + kv * n,
                "flops": 2 * params * n + 2 * head + layers * 4 * case["heads"] * 128 * n * (n + 1) / 2}
    n, seen = case.get("nodes", 1), case["prompt"] + case["committed"]
    return {"bytes": 2 * (params + head) + kv * (seen + n) + 4 * n * case["vocab"],
            "flops": 2 * n * (params + head) + layers * 4 * case["heads"] * 128 * n * (seen + 12)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("attn", "chunk"):
        return {"rel": 1e-2}          # probabilities and results in bf16
    if kind == "linear":
        return {"rel": 1e-2} if case["out"] == "bf16" else {"rel": 1e-5}
    if kind in ("norm", "rows"):
        return {"rel": 1e-2}          # element-wise, roundings to bf16 in between
    return {"rel": 1e-1}              # bf16 roundings of one layer travel through the rest


# ------------------------------------------------------------------ 64-bit results

def _attention(q, k, v, open_):
    """q [H, M, D], k/v [HK, N, D], open_ [M, N] bool -> [H, M, D], all fp64."""
    gqa = q.shape[0] // k.shape[0]
    out = torch.empty_like(q)
    closed = ~open_
    for h in range(q.shape[0]):
        s = (q[h] @ k[h // gqa].t().contiguous()) * q.shape[-1] ** -0.5
        out[h] = torch.softmax(s.masked_fill_(closed, -math.inf), -1) @ v[h // gqa]
    return out


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w


def _rope(x, cos, sin):
    a, b = x.chunk(2, -1)
    return x * cos + torch.cat((-b, a), -1) * sin


def _silu_mul(g, u):
    return g / (1 + torch.exp(-g)) * u


def _tables(pos):
    """RoPE rows in bf16, as a model keeps them, for use in fp64."""
    f = THETA ** (-torch.arange(0, 128, 2, device=DEV, dtype=torch.float64) / 128)
    a = (pos.double()[:, None] * f).repeat(1, 2)
    return a.cos().to(BF).double()[:, None], a.sin().to(BF).double()[:, None]


def _exact_model(case, seed):
    H, HQ, HK, F, V = case["hidden"], case["heads"], case["kv_heads"], case["ffn"], case["vocab"]
    g = _gen(seed)

    def w(*shape):
        return _randn(g, *shape, scale=0.02)

    def norm_w():
        return (1.0 + torch.randn(H, generator=g, device=DEV) * 0.02).to(BF).double()

    def head_w():
        return (1.0 + torch.randn(128, generator=g, device=DEV) * 0.02).to(BF).double()

    prompt = case["kind"] == "prompt"
    if prompt:
        n, start = case["rows"], 0
        ids, pos = _tokens(case, seed, n), torch.arange(n, device=DEV)
        open_ = torch.ones(n, n, dtype=torch.bool, device=DEV).tril()
    else:
        start = case["prompt"] + case["committed"]
        if case["kind"] == "token":
            n, ids, parents, depths = 1, _tokens(case, seed, 1), [-1], [0]
        else:
            n = case["nodes"]
            _, toks, parents, depths = _candidates(seed, n)
            ids = torch.tensor(toks, device=DEV)
        pos = start + torch.tensor(depths, device=DEV)
        open_ = _trie_mask(parents, start, start + n).to(DEV)
    x = w(V, H)[ids].double()
    cos, sin = _tables(pos)
    past = None if prompt else _cached(case, seed)
    ks, vs = [], []
    for _ in range(case["layers"]):
        in_norm, wqkv, qn, kn, wo, post, wgu, wd = (norm_w(), w((HQ + 2 * HK) * 128, H), head_w(), head_w(),
                                                    w(H, HQ * 128), norm_w(), w(2 * F, H), w(H, F))
        p = (_norm(x, in_norm) @ wqkv.double().t()).view(n, HQ + 2 * HK, 128)
        q = _rope(_norm(p[:, :HQ], qn), cos, sin).transpose(0, 1).contiguous()
        k = _rope(_norm(p[:, HQ:HQ + HK], kn), cos, sin).transpose(0, 1).contiguous()
        v = p[:, HQ + HK:].transpose(0, 1).contiguous()
        ks.append(k)
        vs.append(v)
        if past is not None:
            ck, cv = next(past)
            k, v = torch.cat((ck.double(), k), 1), torch.cat((cv.double(), v), 1)
        o = _attention(q, k, v, open_).transpose(0, 1).reshape(n, HQ * 128)
        x = x + o @ wo.double().t()
        gu = _norm(x, post) @ wgu.double().t()
        x = x + _silu_mul(gu[:, :F], gu[:, F:]) @ wd.double().t()
    y = _norm(x[-1:] if prompt else x, norm_w())
    return [y @ w(V, H).double().t()] + ks + vs


def exact(case, seed):
    kind = case["kind"]
    if kind in ("attn", "chunk"):
        q, kp, vp, kn, vn, msk = _attn_inputs(case, seed)
        open_ = torch.cat((torch.ones(msk.shape[0], kp.shape[1], dtype=torch.bool, device=DEV), msk), 1)
        k, v = torch.cat((kp, kn), 1).double(), torch.cat((vp, vn), 1).double()
        return _attention(q.double(), k, v, open_)
    if kind == "linear":
        x, w = _linear_inputs(case, seed)
        return x.double() @ w.double().t()
    if kind == "norm":
        x, w, q, k, wq, wk, cos, sin, gu = (t.double() for t in _norm_inputs(case, seed))
        cos, sin, F = cos[:, None], sin[:, None], case["ffn"]
        return [_norm(x, w), _rope(_norm(q, wq), cos, sin), _rope(_norm(k, wk), cos, sin),
                _silu_mul(gu[:, :F], gu[:, F:])]
    if kind == "rows":
        r, h, w, q, k, cos, sin, gate, up, xv, cosv, sinv = (t.double() for t in _rows_inputs(case, seed))
        x = r + h
        cos, sin = cos[:, None], sin[:, None]
        return [x, x.square(), _norm(x, w), _rope(q, cos, sin), _rope(k, cos, sin), _silu_mul(gate, up),
                _rope(xv, cosv[:, None], sinv[:, None])]
    return _exact_model(case, seed)
