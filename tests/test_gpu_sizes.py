"""Trie attention at the edges of the kernels' size rules, against the oracle
(test_gpu_parity's comparison and tolerances)."""
from __future__ import annotations

import numpy as np
import pytest

from helpers import run_gpu, small_trie, tensors
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
                                                   (5, 32, "f32", 40 * 64 + 7, 2), (3, 64, "f32", 36 * 64 + 1, 2)])
def test_carry_sums_over_many_chunks(gpu, monkeypatch, H, hd, dtype, rows, chunk):
    """One root over every chunk: sums of 16 chunks or fewer (one thread
    each) and longer ones (split over the workgroup's waves), rows narrower
    and wider than a wave's 64 column groups."""
    monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    par = _tree(rows - 1, 20, seed=rows)
    par = np.concatenate([[-1], par + 1]).astype(np.int32)
    _check(par, H, hd, seed=rows, dtype=dtype, rope=True, acc=True)


@pytest.mark.parametrize("H,hd,dtype", [(4, 16, "f32"), (3, 32, "f32"), (4, 16, "bf16")])
@pytest.mark.parametrize("chunk", [1, 3])
def test_more_claims_than_workgroups(gpu, monkeypatch, H, hd, dtype, chunk):
    """Plans on both sides of one claim per workgroup: a few tiles (no
    counter is read), and more (chunk, head group) claims than the chip
    holds workgroups, twice over the same counters, the same bytes."""
    monkeypatch.setenv("AGPT_ATTN_CHUNK", str(chunk))
    tr = small_trie(n_tokens=26000, order=4, vocab=30, depth=12, seed=9)
    for rows in (100, 3 * 2048 * 64 // 2 + 65):
        par = tr.parent[:rows]
        assert par.shape[0] == rows
        Q, K, V, G = tensors(rows, H * hd, 5)
        a = run_gpu(par, Q, K, V, G, H, hd, dtype)
        b = run_gpu(par, Q, K, V, G, H, hd, dtype)
        for name, x, y in zip(("O", "lse", "dQ", "dK", "dV"), a, b):
            np.testing.assert_array_equal(x, y, err_msg=name)
    _check(tr.parent[:3000], H, hd, seed=6, dtype="f32")


@pytest.mark.parametrize("H,hd,dtype,rows", [(8, 64, "f32", 65), (8, 64, "f32", 128 * 64 + 1), (2, 32, "f32", 300 * 64),
                                             (8, 16, "f32", 2 * 256 * 64 - 1), (8, 16, "f32", 300 * 64)])
def test_default_chunk_lengths(gpu, H, hd, dtype, rows):
    """Plans around the rule's lines: the deep key side's floor of two tiles,
    fewer claims than workgroups, one claim each, the three-tile floor."""
    tr = small_trie(n_tokens=26000, order=4, vocab=30, depth=12, seed=9)
    assert tr.n_nodes >= rows
    _check(tr.parent[:rows], H, hd, seed=rows, dtype=dtype, rope=True)


@pytest.mark.parametrize("H,hd,dtype,rows", [(3, 16, "f32", 33 * 64 + 5), (1, 16, "f32", 32 * 64), (2, 64, "f32", 70 * 64 + 1),
                                             (4, 64, "bf16", 65 * 64)])
def test_partial_sums_over_chunks(gpu, monkeypatch, H, hd, dtype, rows):
    """Without the carry: chunk sums of the per-tile partials over whole and
    short 32-tile chunks, one root over all of them."""
    monkeypatch.setenv("AGPT_ATTN_CARRY", "0")
    par = _tree(rows - 1, 20, seed=rows)
    par = np.concatenate([[-1], par + 1]).astype(np.int32)
    _check(par, H, hd, seed=rows, dtype=dtype, rope=dtype == "f32", acc=dtype == "f32")


def test_static_plan_past_the_carry(gpu):
    """A batch at head_dim 32 whose carry partials would not fit the static
    scratch, but whose per-tile partials do, is still planned there. Its dK/dV
    sums are grouped by tile instead of by chunk: equal to the allocated
    plan's within the sums' fp32 rounding (root keys sum ~1e5 terms)."""
    import torch

    from agpt_amd import trie
    from agpt_amd.attention import TrieAttention
    par = trie.build_radix_trie(trie.markov_corpus(6800, 3, 65, 1.1, 4), 32).parent
    q, k, v, g = (torch.from_numpy(x).cuda() for x in tensors(par.shape[0], 128, 3))
    outs = []
    for static in (True, False):
        att = TrieAttention(4, 32, max_depth=32)
        (att.plan_static if static else att.plan)(par)
        assert ("path-carry" in att.describe()) != static
        o, lse = att.forward(q, k, v)
        outs.append((o, lse) + tuple(att.backward(q, k, v, o, lse, g)))
        torch.cuda.synchronize()
        att.close()
    for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), *outs):
        assert (a - b).norm() <= 2e-6 * b.norm(), name
