"""The packed varlen drop-ins (agpt_varlen_attention{,_backward,_L_queries,
_L_queries_backward}) against the oracle's packed restatement and the trie
oracle, through the C ABI, over head counts (odd ones leave lanes idle) and
head dims (32 and 64 split a head slice over lanes).

Bar: fp32 within 1e-4 relative / 1e-5 absolute.
"""
from __future__ import annotations

import numpy as np
import pytest

from helpers import assert_close, scale_of, small_trie, tensors
from oracle import oracle as ORC

pytestmark = pytest.mark.gpu


def _pack_nodes(parent, Q, K, V, H, hd):
    """Reference packing (batched_depth_forward.cr:668-742): node i's packed
    prefix = its ancestors' rows then its own, duplicated per node."""
    depth = ORC.depths(parent)
    T = parent.shape[0]
    offs = np.zeros(T, np.int32)
    lens = depth.astype(np.int32)
    offs[1:] = np.cumsum(lens)[:-1]
    rows = []
    for n in range(T):
        path = []
        a = n
        while a >= 0:
            path.append(a)
            a = parent[a]
        rows.extend(path[::-1])
    rows = np.array(rows, np.int64)
    return offs, lens, rows, K[rows], V[rows]


@pytest.mark.parametrize("H,hd", [(4, 8), (1, 4), (3, 16), (8, 16), (2, 32), (5, 32), (16, 64)])
def test_varlen_matches_trie(gpu, H, hd):
    import torch

    from agpt_amd import attention as A
    tr = small_trie(n_tokens=300, depth=9, seed=31)
    T = tr.n_nodes
    D = H * hd
    Q, K, V, G = tensors(T, D, 13)
    scale = scale_of(hd)
    offs, lens, rows, Kp, Vp = _pack_nodes(tr.parent, Q, K, V, H, hd)
    max_len = int(lens.max())
    cu = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    out = torch.zeros(T * D, device="cuda")
    w = torch.zeros(T * H * max_len, device="cuda")
    A.batched_varlen_attention(cu(Q), cu(Kp), cu(Vp), cu(offs), cu(lens), out, w, T, H, hd,
                               max_len, scale)
    o_ref, w_ref = ORC.varlen_fwd(Q, Kp, Vp, offs, lens, T, H, hd, max_len, scale)
    torch.cuda.synchronize()
    assert_close(out.cpu().numpy(), o_ref, what="varlen O")
    assert_close(w.cpu().numpy(), w_ref, what="varlen W")
    unp = torch.empty(T, D, device="cuda")
    A.unpack_batched_attn_output(out, unp, T, H, hd)
    dq = torch.zeros(T * D, device="cuda")
    dk = torch.full((rows.size * D,), 7.0, device="cuda")  # overwritten, not accumulated
    dv = torch.full((rows.size * D,), 7.0, device="cuda")
    A.batched_varlen_attention_backward(cu(Q), cu(Kp), cu(Vp), w, cu(G), cu(offs), cu(lens), dq,
                                        dk, dv, T, H, hd, max_len, scale)
    dq_r, dk_r, dv_r = ORC.varlen_bwd(Q, Kp, Vp, w_ref, G, offs, lens, T, H, hd, max_len, scale,
                                      rows.size)
    torch.cuda.synchronize()
    assert_close(unp.cpu().numpy().ravel(), o_ref, what="unpack")
    assert_close(dq.cpu().numpy(), dq_r, what="varlen dQ")
    assert_close(dk.cpu().numpy(), dk_r, what="varlen dK")
    assert_close(dv.cpu().numpy(), dv_r, what="varlen dV")


@pytest.mark.parametrize("H,hd,kind", [(2, 16, "small"), (3, 8, "small"), (8, 32, "small"), (4, 64, "small"),
                                       (8, 16, "c2"), (2, 16, "chains"), (32, 4, "deep")])
def test_varlen_L_queries(gpu, H, hd, kind):
    """small: a depth-12 trie; c2: a C2-shaped sample (depth 32, 8 x 16);
    chains: radix nodes of 1..300 queries (blocks of 64 queries cut inside
    a node, more (query, head) pairs than lanes); deep: max_len x H past the
    radix-node kernel's δ table (the per-(node, head) fallback)."""
    import torch

    from agpt_amd import attention as A
    from agpt_amd import trie as T_
    if kind == "small":
        tr = small_trie(n_tokens=500, depth=12, seed=41)
    elif kind == "c2":
        tr = T_.config_trie("C2", scale=0.001)
    elif kind == "chains":
        tok = np.concatenate([T_.uniform_tokens(300, 5, 1), T_.uniform_tokens(40, 5, 2)]).astype(np.int32)
        tr = T_.build_radix_trie(tok, 300)
    else:
        tr = small_trie(n_tokens=400, depth=40, seed=43)
    rpar, elen = tr.radix()
    R = rpar.shape[0]
    D = H * hd
    T = tr.n_nodes
    Q, K, V, G = tensors(T, D, 17)
    scale = scale_of(hd)
    # chunk-packer layout (agpt_train.cu:4456-4479): queries of radix node i
    # are its edge rows; its packed prefix = ancestor rows then edge rows.
    heads = np.flatnonzero(tr.radix_head)
    qoff = np.append(heads, T).astype(np.int32)
    q2n = np.repeat(np.arange(R, dtype=np.int32), elen)
    kv_rows = []
    kv_off = np.zeros(R, np.int32)
    kv_len = np.zeros(R, np.int32)
    for r in range(R):
        last = qoff[r + 1] - 1
        path = []
        a = last
        while a >= 0:
            path.append(a)
            a = tr.parent[a]
        kv_off[r] = len(kv_rows)
        kv_len[r] = len(path)
        kv_rows.extend(path[::-1])
    kv_rows = np.array(kv_rows, np.int64)
    Kp, Vp = K[kv_rows], V[kv_rows]
    max_kv = int(kv_len.max())
    cu = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    out = torch.zeros(T * D, device="cuda")
    w = torch.zeros(T * H * max_kv, device="cuda")
    A.batched_varlen_attention_L_queries(cu(Q), cu(Kp), cu(Vp), cu(q2n), cu(qoff), cu(kv_off),
                                         cu(kv_len), out, w, T, H, hd, max_kv, scale)
    o_ref, w_ref = ORC.varlen_L_fwd(Q, Kp, Vp, q2n, qoff, kv_off, kv_len, T, H, hd, max_kv, scale)
    # the radix layout is the trie semantics: same outputs as the trie oracle
    O_trie, _, _ = ORC.fwd(tr.parent, Q, K, V, H, hd, scale)
    torch.cuda.synchronize()
    assert_close(out.cpu().numpy(), o_ref, what="L O")
    # the saved weights: every visible entry (query t of node r sees
    # kv_len[r] - L_r + j + 1 rows)
    vis = kv_len[q2n] - elen[q2n] + (np.arange(T) - qoff[q2n]) + 1
    mask = (np.arange(max_kv)[None, None, :] < vis[:, None, None]) & np.ones((T, H, 1), bool)
    wg = w.cpu().numpy().reshape(T, H, max_kv)
    assert_close(wg[mask], w_ref.reshape(T, H, max_kv)[mask], what="L weights")
    assert_close(o_ref.reshape(T, D), O_trie, what="L oracle vs trie oracle")
    dq = torch.zeros(T * D, device="cuda")
    seed_k = np.random.default_rng(3).standard_normal(kv_rows.size * D).astype(np.float32)
    dk = cu(seed_k.copy())
    dv = cu(seed_k.copy())
    A.batched_varlen_attention_L_queries_backward(cu(Q), cu(Kp), cu(Vp), w, cu(G), cu(q2n),
                                                  cu(qoff), cu(kv_off), cu(kv_len), dq, dk, dv, T,
                                                  H, hd, max_kv, scale)
    dq_r, dk_r, dv_r = ORC.varlen_L_bwd(Q, Kp, Vp, w_ref, G, q2n, qoff, kv_off, kv_len, T, H, hd,
                                        max_kv, scale, kv_rows.size, dk=seed_k, dv=seed_k)
    torch.cuda.synchronize()
    assert_close(dq.cpu().numpy(), dq_r, what="L dQ")
    assert_close(dk.cpu().numpy(), dk_r, what="L dK")
    assert_close(dv.cpu().numpy(), dv_r, what="L dV")


@pytest.mark.parametrize("H,hd,longest", [(3, 16, 16), (2, 16, 32), (3, 16, 33), (1, 32, 64), (2, 16, 65), (2, 64, 31),
                                          (1, 64, 33)])
def test_varlen_L_queries_row_limits(gpu, H, hd, longest):
    """The backward on both sides of its row limits (32 and 64 keys in one
    pass, more in two): one node of `longest` rows whose queries are its last
    1, 17 or all rows, and short nodes around it; dK/dV add into the caller's
    values."""
    import torch

    from agpt_amd import attention as A
    rng = np.random.default_rng(longest)
    kv_len = np.array([1, longest, longest, longest, 5, 16], np.int32)
    L = np.array([1, 1, min(17, longest), longest, 3, 16], np.int32)
    qoff = np.concatenate([[0], np.cumsum(L)]).astype(np.int32)
    q2n = np.repeat(np.arange(6, dtype=np.int32), L)
    kv_off = np.concatenate([[0], np.cumsum(kv_len)[:-1]]).astype(np.int32)
    T, R, D, scale = int(qoff[-1]), int(kv_len.sum()), H * hd, scale_of(hd)
    Q, G = (rng.standard_normal((T, D)).astype(np.float32) for _ in range(2))
    K, V, S = (rng.standard_normal((R, D)).astype(np.float32) for _ in range(3))
    cu = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    tabs = [cu(x) for x in (q2n, qoff, kv_off, kv_len)]
    out, w = torch.zeros(T * D, device="cuda"), torch.zeros(T * H * longest, device="cuda")
    A.batched_varlen_attention_L_queries(cu(Q), cu(K), cu(V), *tabs, out, w, T, H, hd, longest, scale)
    o_ref, w_ref = ORC.varlen_L_fwd(Q, K, V, q2n, qoff, kv_off, kv_len, T, H, hd, longest, scale)
    assert_close(out.cpu().numpy(), o_ref, what="L O")
    dq, dk, dv = torch.zeros(T * D, device="cuda"), cu(S.ravel().copy()), cu(S.ravel().copy())
    A.batched_varlen_attention_L_queries_backward(cu(Q), cu(K), cu(V), w, cu(G), *tabs, dq, dk, dv, T, H, hd, longest,
                                                  scale)
    want = ORC.varlen_L_bwd(Q, K, V, w_ref, G, q2n, qoff, kv_off, kv_len, T, H, hd, longest, scale, R,
                            dk=S.ravel(), dv=S.ravel())
    for name, got, ref in zip(("dQ", "dK", "dV"), (dq, dk, dv), want):
        assert_close(got.cpu().numpy(), ref, what=name)


def test_varlen_L_queries_node_past_4gib(gpu):
    """A node whose weights alone pass 4 GiB (8,200 queries of 16 heads):
    output and weights of its first and last queries against float64 softmax
    attention, at the fp32 bar."""
    import torch

    from agpt_amd import attention as A
    H, hd, n = 16, 16, 8200
    assert n * H * n * 4 > 1 << 32
    D, scale = H * hd, scale_of(hd)
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    Q, K, V = (torch.randn(n, D, generator=g, device="cuda") for _ in range(3))
    q2n = torch.zeros(n, dtype=torch.int32, device="cuda")
    qoff, off, ln = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, n], [0], [n]))
    out, w = torch.zeros(n * D, device="cuda"), torch.zeros(n * H * n, device="cuda")
    A.batched_varlen_attention_L_queries(Q, K, V, q2n, qoff, off, ln, out, w, n, H, hd, n, scale)
    k64, v64 = (x.view(n, H, hd).double().cpu().numpy() for x in (K, V))
    for rows in (slice(0, 20), slice(n - 20, n)):
        wr = w.view(n, H, n)[rows].cpu().numpy()
        o = out.view(n, H, hd)[rows].cpu().numpy()
        q64 = Q.view(n, H, hd)[rows].double().cpu().numpy()
        for j, row in enumerate(range(n)[rows]):
            s = np.einsum("hd,phd->hp", q64[j], k64[: row + 1]) * scale
            p = np.exp(s - s.max(1, keepdims=True))
            p /= p.sum(1, keepdims=True)
            assert_close(wr[j, :, : row + 1], p, what=f"W of query {row}")
            assert not wr[j, :, row + 1:].any()
            assert_close(o[j], np.einsum("hp,phd->hd", p, v64[: row + 1]), what=f"O of query {row}")


@pytest.mark.parametrize("H,hd,n", [(2, 16, 30), (1, 32, 60), (3, 16, 60), (1, 64, 31)])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_varlen_L_queries_nonfinite_stays(gpu, H, hd, n, bad):
    """A non-finite dO of a node's first query reaches the rows that query
    sees (its own, row 0) and no block of 16 rows past the one it takes part
    in: the backward's blocks end in padding lanes that hold the first
    query's operands (n is no multiple of 16)."""
    import torch

    from agpt_amd import attention as A
    D, scale = H * hd, scale_of(hd)
    Q, K, V, G = tensors(n, D, n + hd)
    q2n, qoff, off, ln = (np.array(x, np.int32) for x in ([0] * n, [0, n], [0], [n]))
    _, w = ORC.varlen_L_fwd(Q, K, V, q2n, qoff, off, ln, n, H, hd, n, scale)
    G[0, 0] = bad
    want = ORC.varlen_L_bwd(Q, K, V, w, G, q2n, qoff, off, ln, n, H, hd, n, scale, n)
    cu = lambda x: torch.from_numpy(np.ascontiguousarray(x)).cuda()
    dq, dk, dv = (torch.zeros(n * D, device="cuda") for _ in range(3))
    A.batched_varlen_attention_L_queries_backward(cu(Q), cu(K), cu(V), cu(w), cu(G), cu(q2n), cu(qoff), cu(off), cu(ln),
                                                  dq, dk, dv, n, H, hd, n, scale)
    for name, got, ref in zip(("dQ", "dK", "dV"), (dq, dk, dv), want):
        got, ref = got.cpu().numpy().reshape(n, D), np.asarray(ref).reshape(n, D)
        assert not np.isfinite(got[~np.isfinite(ref)]).any(), f"{name}: a non-finite value vanished"
        assert np.isfinite(ref[16:]).all()
        assert_close(got[16:], ref[16:], what=f"{name} past the first block")


def _f64_heads(Q, K, V, G, heads, hd, n, scale):
    """float64 (weights, O, dQ, dK, dV) of one node of n queries over its n
    rows, for the given heads: [len(heads), n, ..]."""
    q, k, v, g = (x.view(n, -1, hd)[:, heads].double().cpu().numpy().transpose(1, 0, 2) for x in (Q, K, V, G))
    s = np.einsum("hjd,hpd->hjp", q, k) * scale
    s = np.where(np.tri(n, dtype=bool), s, -np.inf)
    w = np.exp(s - s.max(2, keepdims=True))
    w /= w.sum(2, keepdims=True)
    dw = np.einsum("hjd,hpd->hjp", g, v)
    ds = w * (dw - (w * dw).sum(2, keepdims=True)) * scale
    return (w, np.einsum("hjp,hpd->hjd", w, v), np.einsum("hjp,hpd->hjd", ds, k), np.einsum("hjp,hjd->hpd", ds, q),
            np.einsum("hjp,hjd->hpd", w, g))


@pytest.mark.parametrize("H,hd,n,longest", [(64, 16, 16, 1_200_000), (170_000, 64, 100, 100), (1_100_000, 64, 17, 17)])
def test_varlen_L_queries_spans_past_4gib(gpu, H, hd, n, longest):
    """Forward where a block of 16 weight rows spans 4 GiB (a short node in a
    table of long rows), where one node's queries and packed rows do, and
    where 17 of them do: all rows of sampled heads against float64."""
    import torch

    from agpt_amd import attention as A
    scale = scale_of(hd)
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    Q, K, V = (torch.randn(n, H * hd, generator=g, device="cuda") for _ in range(3))
    q2n = torch.zeros(n, dtype=torch.int32, device="cuda")
    qoff, off, ln = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, n], [0], [n]))
    out = torch.zeros(n * H * hd, device="cuda")
    w = torch.zeros(n * H * longest, device="cuda")
    A.batched_varlen_attention_L_queries(Q, K, V, q2n, qoff, off, ln, out, w, n, H, hd, longest, scale)
    heads = [0, 1, H // 2, H - 1]
    w_ref, o_ref = _f64_heads(Q, K, V, Q, heads, hd, n, scale)[:2]
    got_w = w.view(n, H, longest)[:, heads, :n].cpu().numpy().transpose(1, 0, 2)
    assert_close(got_w, w_ref, what="W")
    assert_close(out.view(n, H, hd)[:, heads].cpu().numpy().transpose(1, 0, 2), o_ref, what="O")


def test_varlen_L_queries_backward_weights_past_4gib(gpu):
    """Backward with rows of 64 keys whose one node's weights pass 4 GiB
    (272,000 heads): all rows of sampled heads against float64."""
    import torch

    from agpt_amd import attention as A
    H, hd, n = 272_000, 16, 64
    assert (n - 1) * n * H * 4 > 1 << 32
    scale = scale_of(hd)
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    Q, K, V, G = (torch.randn(n, H * hd, generator=g, device="cuda") for _ in range(4))
    q2n = torch.zeros(n, dtype=torch.int32, device="cuda")
    qoff, off, ln = (torch.tensor(x, dtype=torch.int32, device="cuda") for x in ([0, n], [0], [n]))
    heads = [0, 1, H // 2, H - 1]
    w_ref, _, *want = _f64_heads(Q, K, V, G, heads, hd, n, scale)
    w = torch.zeros(n, H, n, device="cuda")
    w[:, heads] = torch.from_numpy(w_ref.transpose(1, 0, 2).astype(np.float32)).cuda()
    dq, dk, dv = (torch.zeros(n * H * hd, device="cuda") for _ in range(3))
    A.batched_varlen_attention_L_queries_backward(Q, K, V, w.view(-1), G, q2n, qoff, off, ln, dq, dk, dv, n, H, hd, n,
                                                  scale)
    for name, got, ref in zip(("dQ", "dK", "dV"), (dq, dk, dv), want):
        assert_close(got.view(n, H, hd)[:, heads].cpu().numpy().transpose(1, 0, 2), ref, what=name)
