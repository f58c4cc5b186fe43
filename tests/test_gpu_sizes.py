"""Trie attention at the edges of the kernels' size rules, against the oracle
(test_gpu_parity's comparison and tolerances)."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import (ATOL_BF16, RTOL_BF16, abs_terms, assert_close, assert_close_or_f64, assert_close_terms, f64_key_grads,
                     round_bf16, run_gpu, scale_of, small_trie, tensors)
from oracle import oracle as ORC
from test_gpu_parity import _check

pytestmark = pytest.mark.gpu


def _tree(rows: int, depth: int, seed: int):
    """The first `rows` rows (a preorder prefix is a trie) of a corpus trie."""
    par = small_trie(n_tokens=max(60, 2 * rows // max(1, depth // 2)), order=2, vocab=5, depth=depth, seed=seed).parent
    assert par.shape[0] >= rows
    return par[:rows]


@pytest.mark.parametrize("depth,rows,chunk", [(17, 65, 1), (33, 129, 2), (34, 640, 2), (33, 1601, 24), (64, 900, 3)])
def test_path_carry_hd32(gpu, monkeypatch, depth, rows, chunk):
    """The path carry at head_dim 32: prefix capacities of 16 to 64 slots,
    chunks of one tile and of several, short last tiles."""
    monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    _check(_tree(rows, depth, seed=depth), 3, 32, seed=rows, rope=True, acc=True)


@pytest.mark.parametrize("hd,dtype,depth,rows", [(16, "f32", 1, 5), (16, "f32", 33, 700), (16, "f32", 72, 900),
                                                 (32, "f32", 70, 500), (16, "bf16", 33, 700), (32, "bf16", 17, 200)])
def test_rope_table_in_lds(gpu, monkeypatch, hd, dtype, depth, rows):
    """The backward's rotations from the table in LDS do the operations of the
    caller's tables on the same values: the same bytes, and in fp32 the
    oracle's. Depths past the 64-row tables clamp to their last position."""
    par = _tree(rows, depth, seed=depth) if depth > 1 else np.full(rows, -1, np.int32)
    Q, K, V, G = tensors(rows, 2 * hd, rows)
    res = []
    for staged in ("0", "1"):
        monkeypatch.setenv("AGPT_ATTN_ROPELDS", staged)
        res.append(run_gpu(par, Q, K, V, G, 2, hd, dtype, rope=ORC.rope_table(64, hd)))
    for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), *res):
        np.testing.assert_array_equal(a, b, err_msg=name)
    if dtype == "f32":
        _check(par, 2, hd, seed=rows, rope=True)


@pytest.mark.parametrize("H,hd,dtype,rows,chunk", [(3, 16, "f32", 17 * 64 + 1, 1), (8, 16, "f32", 30 * 64, 1),
                                                   (5, 32, "f32", 40 * 64 + 7, 2), (3, 64, "f32", 36 * 64 + 1, 2),
                                                   (3, 16, "f32", 98 * 64 + 1, 1), (2, 64, "f32", 150 * 64, 2)])
def test_carry_sums_over_many_chunks(gpu, monkeypatch, H, hd, dtype, rows, chunk):
    """One root over every chunk: sums of 16 chunks or fewer (one thread
    each) and longer ones (split over the workgroup's waves, 32 chunks a
    round: one round, one chunk into the next, and several), rows narrower
    and wider than a wave's 64 column groups."""
    monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    par = _tree(rows - 1, 20, seed=rows)
    par = np.concatenate([[-1], par + 1]).astype(np.int32)
    _check(par, H, hd, seed=rows, dtype=dtype, rope=True, acc=True)


_ORACLE: dict = {}


def _oracle(H, hd, dtype, rows):
    """Inputs and the oracle's outputs on the first `rows` rows of one trie."""
    key = (H, hd, dtype, rows)
    if key not in _ORACLE:
        par = small_trie(n_tokens=26000, order=4, vocab=30, depth=12, seed=9).parent[:rows]
        assert par.shape[0] == rows
        inp = tensors(rows, H * hd, 5)
        if dtype == "bf16":
            inp = [round_bf16(x) for x in inp]
        Q, K, V, G = inp
        O, W, lse = ORC.fwd(par, Q, K, V, H, hd, scale_of(hd))
        _ORACLE[key] = par, inp, W, (O, lse, *ORC.bwd(par, Q, K, V, W, G, H, hd, scale_of(hd)))
    return _ORACLE[key]


@pytest.mark.parametrize("H,hd,dtype", [(4, 16, "f32"), (3, 32, "f32"), (4, 16, "bf16")])
@pytest.mark.parametrize("chunk", [1, 3])
def test_more_claims_than_workgroups(gpu, monkeypatch, H, hd, dtype, chunk):
    """Plans on both sides of one claim per workgroup: a few tiles (no
    counter is read), and more (chunk, head group) claims than the chip holds
    workgroups. Two passes of one handle over the same counters, into outputs
    full of NaN: the oracle's values, and the same bytes again."""
    import torch

    from agpt_amd.attention import TrieAttention
    monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    tdt = torch.float32 if dtype == "f32" else torch.bfloat16
    for rows in (100, 3 * 2048 * 64 // 2 + 65):
        par, (Q, K, V, G), W, want = _oracle(H, hd, dtype, rows)
        D = H * hd
        att = TrieAttention(H, hd, max_depth=12, dtype=tdt)
        att.plan(par)
        q, k, v, g = (torch.from_numpy(x).cuda().to(tdt) for x in (Q, K, V, G))
        passes = []
        for _ in range(2):
            nan = lambda *n, dt=torch.float32: torch.full(n, float("nan"), device="cuda", dtype=dt)
            o, lse = att.forward(q, k, v, out=nan(rows, D, dt=tdt), lse=nan(rows, H))
            grads = att.backward(q, k, v, o, lse, g, out=(nan(rows, D), nan(rows, D), nan(rows, D)))
            torch.cuda.synchronize()
            passes.append([x.float().cpu().numpy() for x in (o, lse, *grads)])
        att.close()
        scale = scale_of(hd)
        names = ("O", "lse", "dQ", "dK", "dV")
        if dtype == "f32":
            f64 = lambda r: f64_key_grads(par, Q, K, V, G, H, hd, scale, r)
            for name, x, y in zip(names[:3], passes[0], want):
                assert_close(x, y, what=name)
            assert_close_or_f64(passes[0][3], want[3], lambda r: f64(r)[0], what="dK")
            assert_close_or_f64(passes[0][4], want[4], lambda r: f64(r)[1], what="dV")
        else:
            assert_close(passes[0][1], want[1], RTOL_BF16, ATOL_BF16, "lse")
            for name, x, y in zip(names, passes[0], want):
                if name != "lse":
                    assert_close_terms(x, y, lambda r: abs_terms(name, par, Q, K, V, G, W, H, hd, scale, r), what=name)
        for name, x, y in zip(names, *passes):
            np.testing.assert_array_equal(x, y, err_msg=name)


@pytest.mark.parametrize("H,hd,dtype,rows", [(8, 64, "f32", 65), (8, 64, "f32", 128 * 64 + 1), (2, 32, "f32", 300 * 64),
                                             (8, 16, "f32", 2 * 256 * 64 - 1), (8, 16, "f32", 300 * 64),
                                             (8, 64, "bf16", 128 * 64 + 1), (4, 32, "bf16", 2 * 256 * 64 - 1),
                                             (8, 16, "bf16", 300 * 64), (8, 16, "bf16", 3 * 256 * 64)])
def test_default_chunk_lengths(gpu, H, hd, dtype, rows):
    """Plans around the rule's lines: the deep key side's floor of two tiles,
    fewer claims than workgroups, one claim each, the three-tile floor (in
    bf16 at two claims per tile of four heads)."""
    tr = small_trie(n_tokens=26000, order=4, vocab=30, depth=12, seed=9)
    assert tr.n_nodes >= rows
    _check(tr.parent[:rows], H, hd, seed=rows, dtype=dtype, rope=True)


def _rooted(rows, depth, seed):
    """`rows` rows of depth `depth` under one root."""
    par = small_trie(n_tokens=4 * depth + 100, order=2, vocab=5, depth=depth - 1, seed=seed).parent
    par = np.concatenate([[-1], par[:rows - 1] + 1]).astype(np.int32)
    assert par.shape[0] == rows and ORC.depths(par).max() == depth
    return par


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("depth,chunk,iters", [(64, 2, 0), (65, 3, 0), (66, 2, 0), (128, 3, 0), (129, 2, 0), (134, 2, 0),
                                               (60, 2, 3), (65, 2, 2), (128, 2, 2)])
def test_deep_carry_register_turns(gpu, monkeypatch, dtype, depth, chunk, iters):
    """The deep key side's path carry on both sides of its register rules: two
    turns of four key blocks to depth 65, three to depth 129, past that the
    first slots only; three turns on a shallow plan and two on a deep one by
    the knob. A root over ten tiles and more keeps the subtree-range kernel
    out."""
    monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    if iters:
        monkeypatch.setenv("AGPT_ATTN_REGITERS", str(iters))
    _check(_rooted(11 * 64 + 5, depth, seed=depth), 2, 64, seed=depth, dtype=dtype, rope=True, acc=True)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("depth", [20, 65, 72, 129, 134])
def test_rope_table_in_lds_deep(gpu, monkeypatch, dtype, depth):
    """Head dim 64: the deep kernels' rotations from LDS (the fp32 dQ kernel,
    both carry kernels) give the bytes of the caller's 64-row tables."""
    rows = 11 * 64 + 5
    par = _rooted(rows, depth, seed=depth)
    Q, K, V, G = tensors(rows, 128, rows)
    monkeypatch.setenv("AGPT_ATTN_CHUNK", "2")
    res = []
    for staged in ("0", "1"):
        monkeypatch.setenv("AGPT_ATTN_ROPELDS", staged)
        res.append(run_gpu(par, Q, K, V, G, 2, 64, dtype, rope=ORC.rope_table(64, 64)))
    for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), *res):
        np.testing.assert_array_equal(a, b, err_msg=name)


@pytest.mark.parametrize("dtype,depth,want", [("f32", 20, "1/1"), ("f32", 134, "0/1"), ("bf16", 20, "0/1"), ("bf16", 65, "0/1"),
                                              ("bf16", 129, "0/0"), ("bf16", 134, "0/1")])
def test_deep_rotations_are_placed_by_the_plan(gpu, monkeypatch, dtype, depth, want):
    """Head dim 64: the plan decides once which kernels (dQ / key side) take
    the rotations from LDS: those whose workgroups per CU it leaves alone (the
    bf16 key side's cache from depth 66 to 129 does not). The knob is read there too."""
    import torch

    from agpt_amd.attention import TrieAttention
    monkeypatch.setenv("AGPT_ATTN_CHUNK", "2")
    par = _rooted(11 * 64 + 5, depth, seed=depth)
    for knob, expect in (("1", want), ("0", "0/0")):
        monkeypatch.setenv("AGPT_ATTN_ROPELDS", knob)
        att = TrieAttention(2, 64, max_depth=depth, dtype=torch.float32 if dtype == "f32" else torch.bfloat16)
        att.plan(par)
        assert f"rope_in_lds={expect} " in att.describe()
        att.close()


@pytest.mark.parametrize("H,hd,dtype", [(8, 16, "f32"), (4, 32, "f32"), (2, 64, "f32"), (2, 64, "bf16")])
@pytest.mark.parametrize("where", ["Q", "V", "dO"])
def test_nan_stays_near_with_carry(gpu, monkeypatch, H, hd, dtype, where):
    """A NaN in a plan whose backward carries path sums over chunks of two
    tiles reaches what the oracle says and no tile away from it."""
    from test_gpu_nan import test_nan_surfaces
    monkeypatch.setenv("AGPT_ATTN_CHUNK", "2")
    test_nan_surfaces(gpu, dtype, H, hd, where)


@pytest.mark.parametrize("H,hd,dtype,rows", [(3, 16, "f32", 33 * 64 + 5), (1, 16, "f32", 32 * 64), (2, 32, "f32", 70 * 64 + 1),
                                             (2, 64, "f32", 70 * 64 + 1),
                                             (4, 64, "bf16", 65 * 64)])
def test_partial_sums_over_chunks(gpu, monkeypatch, H, hd, dtype, rows):
    """Without the carry: chunk sums of the per-tile partials over whole and
    short 32-tile chunks, one root over all of them."""
    monkeypatch.setenv("AGPT_ATTN_CARRY", "0")
    par = _tree(rows - 1, 20, seed=rows)
    par = np.concatenate([[-1], par + 1]).astype(np.int32)
    _check(par, H, hd, seed=rows, dtype=dtype, rope=dtype == "f32", acc=dtype == "f32")


@pytest.mark.parametrize("chunk", [0, 3])
def test_static_plan_past_the_carry(gpu, monkeypatch, chunk):
    """A batch at head_dim 32 whose carry partials would not fit the static
    scratch at the default chunk length (3 tiles), but whose per-tile partials
    do: planned there with longer chunks, or, with the length set by hand, with
    per-tile partials. The allocated plan does the same: equal bytes."""
    import torch

    from agpt_amd import trie
    from agpt_amd.attention import TrieAttention
    if chunk:
        monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    par = trie.build_radix_trie(trie.markov_corpus(6800, 3, 65, 1.1, 4), 32).parent
    rows = par.shape[0]
    acc = [torch.from_numpy(x).cuda() for x in tensors(rows, 128, 4, n=2)]
    rope = [torch.from_numpy(x).cuda() for x in ORC.rope_table(64, 32)]
    q, k, v, g = (torch.from_numpy(x).cuda() for x in tensors(rows, 128, 3))
    outs = []
    for static in (True, False):
        att = TrieAttention(4, 32, max_depth=32)
        (att.plan_static if static else att.plan)(par)
        assert ("path-carry" in att.describe()) == (chunk == 0)
        o, lse = att.forward(q, k, v)
        outs.append((o, lse) + tuple(att.backward(q, k, v, o, lse, g, acc_dk=acc[0], acc_dv=acc[1], rope=rope)))
        torch.cuda.synchronize()
        att.close()
    for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), *outs):
        assert torch.equal(a, b), name
