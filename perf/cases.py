"""The work that is timed: what a trainer on this framework has it do, each
case one pass through the public entry points.

Kinds of case:
  attn     one batch of trie attention, forward (and backward), on a held plan
  batches  a trie processed as partition-sized row ranges over streams
  varlen   the packed drop-in calls, one query per node or one per edge token
  loss     the per-query loss and its gradient
  rows     the row kernels around one transformer block (projection epilogue,
           norm forward and backward, ReLU backward)
  model    forward and backward of the 4-layer model over one batch

Sizes are the repository's own: heads and head dims of its configurations and
tests, corpora of its Markov generator at 65 and 256 symbols, depths 16 to
128, batches from one small subtree to a few million node-tokens. A case is
one corpus (its trie is what a trainer plans once and keeps); the tensors over
it are made from the seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from agpt_amd import attention as A
from agpt_amd import block, loss as L, trie
from agpt_amd.model import ModelConfig, TrieBatch, TrieGPT

DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
DEV = "cuda"


def listed() -> list[dict]:
    return [
        # A single small subtree of a shallow trie: the trainer's per-subtree
        # call, where launches and latency count.
        dict(name="attn_subtree", kind="attn", n=181, order=3, vocab=65, depth=16, H=4, hd=16,
             dtype="f32", grad=True, rope=True, acc=False),
        # The headline shape: character corpus at depth 32, d_model 128 as
        # 8 heads x 16, a few million node-tokens in one plan.
        dict(name="attn_chars", kind="attn", n=110_000, order=5, vocab=65, depth=32, H=8, hd=16,
             dtype="f32", grad=True, rope=True, acc=False),
        # The same width as 4 heads x 32, one training batch, with descendant
        # sums handed in (a trie that continues in another batch).
        dict(name="attn_wide_heads", kind="attn", n=26_003, order=3, vocab=65, depth=32, H=4, hd=32,
             dtype="f32", grad=True, rope=True, acc=True),
        # bf16 activations at the headline head shape.
        dict(name="attn_bf16", kind="attn", n=30_011, order=5, vocab=65, depth=32, H=8, hd=16,
             dtype="bf16", grad=True, rope=True, acc=False),
        # Deep and wide: byte vocabulary, depth 128, 8 heads x 64 in bf16.
        dict(name="attn_deep", kind="attn", n=6_007, order=8, vocab=256, depth=128, H=8, hd=64,
             dtype="bf16", grad=True, rope=False, acc=False),
        # Plain causal sequences: 512 unshared paths of 256 tokens.
        dict(name="attn_chains", kind="attn", chains=512, chain_len=256, n=512 * 256, order=0, vocab=65,
             depth=256, H=4, hd=64, dtype="bf16", grad=True, rope=False, acc=False),
        # A trie cut into batches of whole bigram partitions, one plan each,
        # dealt over streams.
        dict(name="attn_batches", kind="batches", n=60_013, order=5, vocab=65, depth=32, H=8, hd=16,
             dtype="f32", rows=131_072),
        # The packed drop-in call with one query per node (each node's path
        # gathered by the caller).
        dict(name="varlen_nodes", kind="varlen", n=9_001, order=5, vocab=65, depth=32, H=8, hd=16, radix=False),
        # The packed drop-in call of the radix trainer: every token of an
        # edge a query over the edge's shared rows.
        dict(name="varlen_edges", kind="varlen", n=60_013, order=5, vocab=65, depth=32, H=8, hd=16, radix=True),
        # The loss over a character vocabulary with corpus-mass weights.
        dict(name="loss_chars", kind="loss", n=60_013, order=5, vocab=65, depth=32, V=65, entropy=0.0,
             mass=True, ce_only=False),
        # The row kernels of one block over one training batch: d_model 128,
        # FFN 512, RMS norm, residual gradient added in the norm's backward.
        dict(name="rows_block", kind="rows", T=819_203, H=8, hd=16, ff=512, layer=False, dres=True),
        # Forward and backward of the whole 4-layer model over one batch.
        dict(name="model_batch", kind="model", n=28_001, order=3, vocab=65, depth=32, d_model=128, H=8,
             layers=4, ff=512, layer=False),
    ]


def _log(rng, lo: int, hi: int) -> int:
    """A whole number, odd as often as even, spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    kind = rng.choice(["attn", "attn", "attn", "attn", "deep", "chains", "batches", "varlen", "loss", "rows",
                       "model"])
    order = rng.choice([3, 5])
    if kind == "attn":
        # fp32 and bf16, head shapes of 64 to 256 columns, depths 16 to 64
        H, hd = rng.choice([(4, 16), (8, 16), (4, 32), (2, 64), (4, 64)])
        depth = rng.choice([16, 32, 32, 48, 64])
        return dict(kind="attn", n=_log(rng, 100, 60_000 * 32 // depth), order=order, vocab=65, depth=depth, H=H,
                    hd=hd, dtype=rng.choice(["f32", "f32", "bf16"]), grad=rng.random() < 0.75,
                    rope=rng.random() < 0.75, acc=rng.random() < 0.25)
    if kind == "deep":
        H = rng.choice([4, 8])
        return dict(kind="attn", n=_log(rng, 200, 6_000), order=8, vocab=256, depth=rng.choice([96, 128, 160]), H=H,
                    hd=64, dtype="bf16", grad=rng.random() < 0.75, rope=rng.random() < 0.5, acc=False)
    if kind == "chains":
        c, ln = _log(rng, 8, 512), _log(rng, 33, 256)
        return dict(kind="attn", chains=c, chain_len=ln, n=c * ln, order=0, vocab=65, depth=ln,
                    H=rng.choice([2, 4, 8]), hd=64, dtype="bf16", grad=rng.random() < 0.75, rope=rng.random() < 0.5,
                    acc=False)
    if kind == "batches":
        return dict(kind="batches", n=_log(rng, 6_000, 60_000), order=order, vocab=65, depth=32,
                    H=rng.choice([4, 8]), hd=16, dtype="f32", rows=_log(rng, 32_768, 262_144))
    if kind == "varlen":
        radix = rng.random() < 0.5
        H, hd = rng.choice([(4, 16), (8, 16), (4, 32), (4, 64)])
        return dict(kind="varlen", n=_log(rng, 150, 30_000 if radix else 6_000), order=order, vocab=65,
                    depth=rng.choice([16, 32]), H=H, hd=hd, radix=radix)
    if kind == "loss":
        big = rng.random() < 0.4
        return dict(kind="loss", n=_log(rng, 150, 12_000 if big else 60_000), order=8 if big else order,
                    vocab=256 if big else 65, depth=32, V=256 if big else 65, entropy=rng.choice([0.0, 0.5]),
                    mass=rng.random() < 0.75, ce_only=rng.random() < 0.25)
    if kind == "rows":
        H, hd = rng.choice([(4, 16), (8, 16), (4, 32), (4, 64), (8, 64)])
        return dict(kind="rows", T=_log(rng, 900, 400_000), H=H, hd=hd, ff=rng.choice([256, 512]),
                    layer=rng.random() < 0.5, dres=rng.random() < 0.5)
    return dict(kind="model", n=_log(rng, 400, 20_000), order=order, vocab=65, depth=rng.choice([16, 32]),
                d_model=rng.choice([64, 128]), H=rng.choice([4, 8]), layers=rng.choice([2, 4]),
                ff=rng.choice([256, 512]), layer=rng.random() < 0.5)


# -- inputs -------------------------------------------------------------------

def _trie(case, counts=False):
    if case.get("chains"):
        tok = trie.uniform_tokens(case["chains"] * case["chain_len"], case["vocab"], case["n"])
        return trie.build_chains(tok, case["chains"], case["chain_len"])
    zipf = 1.2 if case["vocab"] == 256 else 1.1
    tok = trie.markov_corpus(case["n"], case["order"], case["vocab"], zipf, case["n"])
    return trie.build_radix_trie(tok, case["depth"], counts=counts)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape, dtype=torch.float32, std=1.0):
    x = torch.randn(*shape, generator=g, device=DEV)
    if std != 1.0:
        x *= std
    return x.to(dtype)


def _attn_inputs(case, seed, tr):
    """Post-norm projections have unit variance, so scores spread over a few
    units as in a trained model."""
    g = _gen(seed)
    T, D, dt = tr.n_nodes, case["H"] * case["hd"], DTYPES[case["dtype"]]
    q, k, v = (_randn(g, T, D, dtype=dt) for _ in range(3))
    d_o = _randn(g, T, D, dtype=dt) if case.get("grad", True) else None
    acc = tuple(_randn(g, T, D) for _ in range(2)) if case.get("acc") else (None, None)
    return q, k, v, d_o, acc


def _batch_ranges(case, tr):
    return A.range_batches(tr.n_nodes, case["rows"], A.partition_starts(tr.radix_head, tr.depth))


def _paths(parent, depth, nodes):
    """Packed rows of the nodes' root-to-node paths: offsets, lengths, row ids."""
    lens = depth[nodes].astype(np.int64)
    offs = np.zeros(nodes.shape[0], np.int64)
    np.cumsum(lens[:-1], out=offs[1:])
    rows = np.empty(int(lens.sum()), np.int64)
    cur, at, live = nodes.astype(np.int64), offs + lens - 1, np.arange(nodes.shape[0])
    while live.size:
        rows[at[live]] = cur[live]
        cur[live] = parent[cur[live]]
        at[live] -= 1
        live = live[cur[live] >= 0]
    return offs.astype(np.int32), lens.astype(np.int32), rows


def _varlen_layout(case, tr):
    """Device tables of the packed layout, and per query its first packed
    row and visible rows."""
    T = tr.n_nodes
    if case["radix"]:
        heads = np.flatnonzero(tr.radix_head)
        qoff = np.append(heads, T).astype(np.int32)
        elen = np.diff(qoff)
        q2n = np.repeat(np.arange(heads.shape[0], dtype=np.int32), elen)
        offs, lens, rows = _paths(tr.parent, tr.depth, qoff[1:] - 1)
        first = offs[q2n].astype(np.int64)
        vis = (lens[q2n] - elen[q2n] + np.arange(T) - qoff[q2n] + 1).astype(np.int64)
        tabs = (q2n, qoff, offs, lens)
    else:
        offs, lens, rows = _paths(tr.parent, tr.depth, np.arange(T))
        first, vis = offs.astype(np.int64), lens.astype(np.int64)
        tabs = (offs, lens)
    return tabs, rows, first, vis, int(lens.max())


def _varlen_inputs(case, seed, tr, rows):
    g = _gen(seed)
    T, D = tr.n_nodes, case["H"] * case["hd"]
    q, k, v, d_o = (_randn(g, T, D) for _ in range(4))
    idx = torch.from_numpy(rows).to(DEV)
    return q, k.index_select(0, idx), v.index_select(0, idx), d_o


def _loss_inputs(case, seed, tr):
    cfg = ModelConfig(vocab=case["V"])
    batch = TrieBatch(tr, cfg, DEV, L.MASS_LINEAR if case["mass"] else L.MASS_OFF)
    return _randn(_gen(seed), batch.T, case["V"], std=2.0), batch


def _rows_inputs(case, seed):
    g = _gen(seed)
    T, D, Fd = case["T"], case["H"] * case["hd"], case["ff"]
    pos = torch.randint(0, 32, (T,), generator=g, device=DEV, dtype=torch.int32)
    cos, sin = A.rope_tables(32, case["hd"], device=DEV)
    return dict(qkv=_randn(g, T, 3 * D), bias=_randn(g, 3 * D, std=0.1), pos=pos, cos=cos, sin=sin,
                x=_randn(g, T, D), w=1.0 + _randn(g, D, std=0.1),
                b=_randn(g, D, std=0.1) if case["layer"] else None, dy=_randn(g, T, D),
                dres=_randn(g, T, D) if case["dres"] else None,
                # the ReLU's output: half of it zero
                h=_randn(g, T, Fd).clamp_(min=0.0), dh=_randn(g, T, Fd))


def _model_cfg(case) -> ModelConfig:
    return ModelConfig(vocab=case["vocab"], d_model=case["d_model"], n_heads=case["H"], n_layers=case["layers"],
                       d_ff=case["ff"], max_depth=case["depth"], norm="layer" if case["layer"] else "rms")


def prepare(case, seed) -> dict:
    kind = case["kind"]
    s = dict(case=case)
    if kind == "rows":
        return s | _rows_inputs(case, seed)
    tr = _trie(case, counts=kind in ("loss", "model"))
    if kind == "attn":
        att = A.TrieAttention(case["H"], case["hd"], max_depth=case["depth"], dtype=DTYPES[case["dtype"]])
        att.plan(tr.parent)
        rope = A.rope_tables(case["depth"], case["hd"], device=DEV) if case["rope"] else None
        return s | dict(att=att, rope=rope, x=_attn_inputs(case, seed, tr))
    if kind == "batches":
        att = A.RangedTrieAttention(case["H"], case["hd"], tr.parent, _batch_ranges(case, tr),
                                    max_depth=case["depth"], dtype=DTYPES[case["dtype"]])
        return s | dict(att=att, x=_attn_inputs(case, seed, tr),
                        rope=A.rope_tables(case["depth"], case["hd"], device=DEV))
    if kind == "varlen":
        tabs, rows, _, _, max_len = _varlen_layout(case, tr)
        q, kp, vp, d_o = _varlen_inputs(case, seed, tr, rows)
        # a row of the weights table is written up to its query's length, so
        # the trainer's table starts as zeros
        w = torch.zeros(tr.n_nodes * case["H"] * max_len, device=DEV)
        return s | dict(x=(q, kp, vp, d_o), tabs=[torch.from_numpy(t).to(DEV) for t in tabs], w=w, max_len=max_len)
    if kind == "loss":
        logits, batch = _loss_inputs(case, seed, tr)
        return s | dict(logits=logits, batch=batch)
    m = TrieGPT(_model_cfg(case), device=DEV, seed=seed)
    m.plan(tr)
    return s | dict(model=m)


# -- one pass -----------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attn":
        att = s["att"]
        q, k, v, d_o, (acc_dk, acc_dv) = s["x"]
        o, lse = att.forward(q, k, v)
        if d_o is None:
            return dict(o=o, lse=lse)
        dq, dk, dv = att.backward(q, k, v, o, lse, d_o, acc_dk=acc_dk, acc_dv=acc_dv, rope=s["rope"])
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    if kind == "batches":
        q, k, v, d_o, _ = s["x"]
        o, lse, (dq, dk, dv) = s["att"].fwd_bwd(q, k, v, d_o, rope=s["rope"])
        return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)
    if kind == "varlen":
        q, kp, vp, d_o = s["x"]
        T, H, hd = q.shape[0], case["H"], case["hd"]
        w, scale = s["w"], A.default_scale(hd)
        out, dq = torch.empty_like(q), torch.empty_like(q)
        args = (T, H, hd, s["max_len"], scale)
        if case["radix"]:
            dk, dv = torch.zeros_like(kp), torch.zeros_like(vp)  # the call adds into them
            A.batched_varlen_attention_L_queries(q, kp, vp, *s["tabs"], out, w, *args)
            A.batched_varlen_attention_L_queries_backward(q, kp, vp, w, d_o, *s["tabs"], dq, dk, dv, *args)
        else:
            dk, dv = torch.empty_like(kp), torch.empty_like(vp)
            A.batched_varlen_attention(q, kp, vp, *s["tabs"], out, w, *args)
            A.batched_varlen_attention_backward(q, kp, vp, w, d_o, *s["tabs"], dq, dk, dv, *args)
        return dict(o=out, w=w, dq=dq, dk=dk, dv=dv)
    if kind == "loss":
        d, loss = L.loss_per_query(s["logits"], *s["batch"].loss_args, mass_weights=s["batch"].mass,
                                   entropy_lambda=case["entropy"], ce_only=case["ce_only"])
        return dict(d_logits=d, loss=loss)
    if kind == "rows":
        q, k, v = block.bias_rope_split(s["qkv"], s["bias"], s["pos"], s["cos"], s["sin"], case["H"])
        y, mean, rstd = block.norm_fwd(s["x"], s["w"], s["b"])
        dx, dw, db = block.norm_bwd(s["dy"], s["x"], s["w"], mean, rstd, case["layer"], s["dres"])
        dh, dbh = block.relu_bwd(s["dh"], s["h"])
        return dict(q=q, k=k, v=v, y=y, dx=dx, dw=dw, db=db, dh=dh, dbh=dbh)
    m = s["model"]
    m.flat.grad = None
    losses = []
    for grp in m.groups:
        lv = m.loss(grp)
        lv.backward()
        losses.append(lv.detach())
    return dict(loss=torch.stack(losses), grad=m.flat.grad)


# -- what a pass cannot do without ----------------------------------------------

@functools.lru_cache(maxsize=64)
def _shape(n, order, vocab, depth, chains, chain_len):
    tr = _trie(dict(n=n, order=order, vocab=vocab, depth=depth, chains=chains, chain_len=chain_len))
    return tr.n_nodes, tr.sum_depth, tr


def work(case) -> dict:
    kind = case["kind"]
    if kind == "rows":
        T, D, Fd = case["T"], case["H"] * case["hd"], case["ff"]
        norm = 4 * T * D * (2 + 3 + bool(case["dres"])) + 4 * T * (4 if case["layer"] else 2)
        return {"bytes": 4 * T * 6 * D + 4 * T + norm + 4 * T * 3 * Fd, "flops": T * (15 * D + 2 * Fd)}
    T, sd, tr = _shape(case["n"], case["order"], case["vocab"], case["depth"], case.get("chains", 0),
                       case.get("chain_len", 0))
    if kind in ("attn", "batches"):
        D, H = case["H"] * case["hd"], case["H"]
        e = 2 if case["dtype"] == "bf16" else 4
        grad = case.get("grad", True)
        b = T * (4 * D * e + 4 * H) + grad * T * (5 * D * e + 4 * H + 12 * D + 8 * D * bool(case.get("acc")))
        return {"bytes": b, "flops": sd * D * (12 if grad else 4)}
    if kind == "varlen":
        _, rows, _, vis, _ = _varlen_layout(case, tr)
        D, H, R, S = case["H"] * case["hd"], case["H"], rows.shape[0], int(vis.sum())
        # forward: q, packed k, v, out, weights; backward: q, k, v, weights,
        # dO in, dq, dk, dv out
        return {"bytes": 4 * (T * D * 5 + R * D * 6 + S * H * 2), "flops": S * D * 12}
    if kind == "loss":
        return {"bytes": T * (8 * case["V"] + 16), "flops": T * case["V"] * 8}
    D, Fd, V, nl = case["d_model"], case["ff"], case["vocab"], case["layers"]
    mm = 2 * T * (nl * (4 * D * D + 2 * D * Fd) + V * D)
    # each layer's activations written once and read once in the backward
    # (n1, q, k, v, o, x, n2, h), the stream read and written per layer in
    # both directions
    b = 4 * T * nl * (2 * (7 * D + Fd) + 4 * D) + 4 * T * 2 * V
    return {"bytes": b, "flops": 3 * mm + nl * 12 * sd * D}


def tolerance(case) -> dict:
    """About four times what a pass shows against 64 bits: 32-bit paths 5e-8
    to 5e-7, bf16 ones 2e-3 (the rounding of O and of the weights), the
    model's gradient 4e-6 to 3e-5 (32-bit sums over a batch through its
    layers; the most where the batch is small)."""
    if case["kind"] == "model":
        return {"rel": 1e-4}
    if case.get("dtype") == "bf16":
        return {"rel": 8e-3}
    return {"rel": 2e-6}


# -- the same in 64 bits --------------------------------------------------------

def _anc(depth, j):
    """Row of each row's ancestor at depth j (any row above where it has
    none): the last earlier row of that depth in depth-first order."""
    idx = torch.arange(depth.shape[0], device=depth.device)
    return torch.where(depth == j, idx, 0).cummax(0).values


def _seg_sum(x, first, end):
    """Sums of x [T, D] over the row ranges [first, end), by a running sum."""
    c = x.t().contiguous().cumsum(1)
    lo = torch.where((first > 0)[None, :], c[:, (first - 1).clamp(min=0)], 0.0)
    return (c[:, end - 1] - lo).t()


def _trie_fwd64(q, k, v, depth, H, scale):
    T, D = q.shape
    P = int(depth.max())
    S = torch.full((P, T, H), -math.inf, dtype=torch.float64, device=q.device)
    for j in range(1, P + 1):
        s = (q * k[_anc(depth, j)]).view(T, H, -1).sum(-1) * scale
        S[j - 1] = torch.where((depth >= j)[:, None], s, -math.inf)
    lse = torch.logsumexp(S, 0)
    o = torch.zeros_like(q)
    for j in range(1, P + 1):
        S[j - 1] = torch.exp(S[j - 1] - lse)
        o += (S[j - 1][:, :, None] * v[_anc(depth, j)].view(T, H, -1)).view(T, D)
    return o, lse, S


def _trie_bwd64(q, k, v, W, g, depth, end, H, scale):
    T, D = q.shape
    P = W.shape[0]
    dW = torch.zeros_like(W)
    for j in range(1, P + 1):
        dW[j - 1] = (g * v[_anc(depth, j)]).view(T, H, -1).sum(-1)
    delta = (W * dW).sum(0)
    dq, dk, dv = (torch.zeros_like(q) for _ in range(3))
    for j in range(1, P + 1):
        ds = W[j - 1] * (dW[j - 1] - delta) * scale
        dq += (ds[:, :, None] * k[_anc(depth, j)].view(T, H, -1)).view(T, D)
        keys = (depth == j).nonzero()[:, 0]
        dk[keys] = _seg_sum((ds[:, :, None] * q.view(T, H, -1)).view(T, D), keys, end[keys])
        dv[keys] = _seg_sum((W[j - 1][:, :, None] * g.view(T, H, -1)).view(T, D), keys, end[keys])
    return dq, dk, dv


def _rotate(x, cos, sin, pos, H, sign):
    """Rotates the pairs (2i, 2i+1) of every head by sign times the angle at pos."""
    T, D = x.shape
    c = cos.double()[pos][:, None, 0::2]
    s = sign * sin.double()[pos][:, None, 0::2]
    p = x.view(T, H, -1, 2)
    a, b = p[..., 0], p[..., 1]
    return torch.stack([a * c - b * s, a * s + b * c], -1).reshape(T, D)


def _depth_end(tr):
    return (torch.from_numpy(tr.depth.astype(np.int64)).to(DEV),
            torch.from_numpy(tr.subtree_end.astype(np.int64)).to(DEV))


def _exact_attn(case, seed):
    tr = _trie(case)
    q, k, v, d_o, (ak, av) = _attn_inputs(case, seed, tr)
    depth, end = _depth_end(tr)
    H, scale = case["H"], 1.0 / math.sqrt(case["hd"])
    q, k, v = q.double(), k.double(), v.double()
    o, lse, W = _trie_fwd64(q, k, v, depth, H, scale)
    if d_o is None:
        return dict(o=o, lse=lse)
    dq, dk, dv = _trie_bwd64(q, k, v, W, d_o.double(), depth, end, H, scale)
    if ak is not None:
        dk += ak.double()
        dv += av.double()
    if case.get("rope", True):
        cos, sin = _own_rope(case["depth"], case["hd"])
        dq = _rotate(dq, cos, sin, depth - 1, H, -1.0)
        dk = _rotate(dk, cos, sin, depth - 1, H, -1.0)
    return dict(o=o, lse=lse, dq=dq, dk=dk, dv=dv)


def _own_rope(seq, hd):
    """The caller's own cos / sin tables, [seq, hd] in 32 bits, each angle twice."""
    pos = np.arange(seq, dtype=np.float32)[:, None]
    i = np.arange(hd // 2, dtype=np.float32)[None, :]
    theta = (pos / np.power(np.float32(10000.0), np.float32(2.0) * i / np.float32(hd))).astype(np.float32)
    return tuple(torch.from_numpy(np.repeat(f(theta), 2, axis=1).astype(np.float32)).to(DEV)
                 for f in (np.cos, np.sin))


def _exact_varlen(case, seed):
    tr = _trie(case)
    _, rows, first, vis, max_len = _varlen_layout(case, tr)
    q, kp, vp, g = (x.double() for x in _varlen_inputs(case, seed, tr, rows))
    T, D = q.shape
    H, scale = case["H"], 1.0 / math.sqrt(case["hd"])
    first, vis = torch.from_numpy(first).to(DEV), torch.from_numpy(vis).to(DEV)

    def at(p):
        return (first + p).clamp(max=rows.shape[0] - 1)
    W = torch.full((T, H, max_len), -math.inf, dtype=torch.float64, device=DEV)
    for p in range(max_len):
        s = (q * kp[at(p)]).view(T, H, -1).sum(-1) * scale
        W[:, :, p] = torch.where((vis > p)[:, None], s, -math.inf)
    W = torch.softmax(W, -1)
    o, dq, dk, dv = (torch.zeros_like(x) for x in (q, q, kp, vp))
    dW = torch.zeros_like(W)
    for p in range(max_len):
        vr = vp[at(p)].view(T, H, -1)
        o += (W[:, :, p, None] * vr).view(T, D)
        dW[:, :, p] = (g.view(T, H, -1) * vr).sum(-1)
    dS = W * (dW - (W * dW).sum(-1, keepdim=True)) * scale
    for p in range(max_len):
        see = (vis > p).nonzero()[:, 0]
        r = at(p)[see]
        dq[see] += (dS[see, :, p, None] * kp[r].view(-1, H, case["hd"])).view(-1, D)
        dk.index_add_(0, r, (dS[see, :, p, None] * q[see].view(-1, H, case["hd"])).view(-1, D))
        dv.index_add_(0, r, (W[see, :, p, None] * g[see].view(-1, H, case["hd"])).view(-1, D))
    return dict(o=o, w=W.reshape(-1), dq=dq, dk=dk, dv=dv)


def _loss64(logits, loss_args, mass, entropy, ce_only):
    """(d_logits, loss per query) of 64-bit logits."""
    q2n, qoff, rid, tok, coff, ctok, cval = (t.long() for t in loss_args)
    T, V = logits.shape
    idx = torch.arange(T, device=logits.device)
    p = torch.softmax(logits, -1)
    endp = qoff[q2n + 1] == idx + 1
    if ce_only:
        endp &= idx + 1 == T
    mass = torch.ones(T, dtype=torch.float64, device=logits.device) if mass is None else mass.double()
    # targets: the next token of the edge, or the endpoint's count shares
    tgt = torch.zeros_like(p)
    inner = (~endp).nonzero()[:, 0]
    tgt[inner, tok[inner + 1]] = 1.0
    ends = endp.nonzero()[:, 0]
    node = rid[q2n[ends]]
    n_ent = coff[node + 1] - coff[node]
    owner = torch.repeat_interleave(ends, n_ent)
    ent = torch.repeat_interleave(coff[node] - (n_ent.cumsum(0) - n_ent), n_ent) + torch.arange(
        owner.shape[0], device=owner.device)
    tot = torch.zeros(T, dtype=torch.float64, device=p.device).index_add_(0, owner, cval[ent].double())
    share = cval[ent].double() / tot[owner]
    tgt.index_put_((owner, ctok[ent]), share, accumulate=True)
    w = mass.clone()
    if entropy > 0:
        Hq = torch.zeros_like(tot).index_add_(0, owner, -share * torch.log(share))
        w = w * (1.0 + entropy * Hq / math.log(V))
    empty = ends[n_ent == 0]
    loss = -(tgt * torch.log(p + 1e-10)).sum(-1) * w
    w[empty] = 1.0  # an endpoint without counts keeps the plain softmax
    return (p - tgt) * w[:, None], loss


def _exact_loss(case, seed):
    logits, batch = _loss_inputs(case, seed, _trie(case, counts=True))
    d, loss = _loss64(logits.double(), batch.loss_args, batch.mass, case["entropy"], case["ce_only"])
    return dict(d_logits=d, loss=loss)


def _exact_rows(case, seed):
    s = _rows_inputs(case, seed)
    H, D = case["H"], case["H"] * case["hd"]
    qkv = s["qkv"].double() + s["bias"].double()
    q, k, v = qkv[:, :D].contiguous(), qkv[:, D:2 * D].contiguous(), qkv[:, 2 * D:].contiguous()
    pos = s["pos"].long()
    x, w, dy = s["x"].double(), s["w"].double(), s["dy"].double()
    xc = x - x.mean(-1, keepdim=True) if case["layer"] else x
    r = (xc.square().mean(-1, keepdim=True) + 1e-5).rsqrt()
    xh, gy = xc * r, dy * w
    dx = r * (gy - xh * (gy * xh).mean(-1, keepdim=True) - (gy.mean(-1, keepdim=True) if case["layer"] else 0.0))
    if s["dres"] is not None:
        dx = dx + s["dres"].double()
    dh = torch.where(s["h"] > 0, s["dh"], 0.0)
    return dict(q=_rotate(q, s["cos"], s["sin"], pos, H, 1.0), k=_rotate(k, s["cos"], s["sin"], pos, H, 1.0), v=v,
                y=xh * w + (s["b"].double() if case["layer"] else 0.0), dx=dx, dw=(dy * xh).sum(0),
                db=dy.sum(0) if case["layer"] else None, dh=dh.double(), dbh=dh.double().sum(0))


class _Attn64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, depth, end, H, scale):
        o, _, W = _trie_fwd64(q, k, v, depth, H, scale)
        ctx.save_for_backward(q, k, v, W, depth, end)
        ctx.meta = H, scale
        return o

    @staticmethod
    def backward(ctx, g):
        q, k, v, W, depth, end = ctx.saved_tensors
        H, scale = ctx.meta
        return *_trie_bwd64(q, k, v, W, g.contiguous(), depth, end, H, scale), None, None, None, None


def _exact_model(case, seed):
    from torch.utils.checkpoint import checkpoint
    cfg = _model_cfg(case)
    tr = _trie(case, counts=True)
    m = TrieGPT(cfg, device=DEV, seed=seed)  # its initial weights only
    flat = m.flat.detach().double().requires_grad_(True)
    hd = cfg.d_model // cfg.n_heads
    cos, sin = _own_rope(cfg.max_depth, hd)
    m.flat = flat
    P = m.params()

    def norm(x, w, b):
        if case["layer"]:
            x = x - x.mean(-1, keepdim=True)
        y = x * (x.square().mean(-1, keepdim=True) + cfg.eps).rsqrt() * w
        return y + b if case["layer"] else y

    def layer(x, l, depth, end):
        n1 = norm(x, P[f"n1_w{l}"], P[f"n1_b{l}"])
        q, k, v = (n1 @ P[f"w{c}{l}"].t() + P[f"b{c}{l}"] for c in "qkv")
        pos = depth - 1
        q, k = (_rotate(t, cos, sin, pos, cfg.n_heads, 1.0) for t in (q, k))
        x = x + _Attn64.apply(q, k, v, depth, end, cfg.n_heads, 1.0 / math.sqrt(hd)) @ P[f"wo{l}"].t() + P[f"bo{l}"]
        n2 = norm(x, P[f"n2_w{l}"], P[f"n2_b{l}"])
        return x + torch.relu(n2 @ P[f"w1{l}"].t() + P[f"b1{l}"]) @ P[f"w2{l}"].t() + P[f"b2{l}"]

    losses = []
    from agpt_amd.model import subtree_groups
    depth_all, end_all = _depth_end(tr)
    for a, b in subtree_groups(tr, 1 << 20):
        batch = TrieBatch(tr, cfg, DEV, L.MASS_LINEAR, rows=(a, b))
        depth, end = depth_all[a:b], end_all[a:b] - a
        x = P["tok_emb"][batch.tokens]
        for l in range(cfg.n_layers):
            x = checkpoint(layer, x, l, depth, end, use_reentrant=False)
        logits = norm(x, P["nf_w"], P["nf_b"]) @ P["w_out"].t() + P["b_out"]
        d, loss_q = _loss64(logits.detach(), batch.loss_args, batch.mass, 0.0, False)
        logits.backward(d, retain_graph=True)
        losses.append(loss_q.sum())
    return dict(loss=torch.stack(losses), grad=flat.grad)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("attn", "batches"):
        return _exact_attn(case, seed)
    return dict(varlen=_exact_varlen, loss=_exact_loss, rows=_exact_rows, model=_exact_model)[kind](case, seed)
