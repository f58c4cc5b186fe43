"""Trie attention at the edges of the kernels' size rules, against the oracle
(test_gpu_parity's comparison and tolerances)."""
from __future__ import annotations

import pytest

from helpers import small_trie
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
