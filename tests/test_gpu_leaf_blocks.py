"""Merkle layers whose nodes take one to six blocks of columns, whole and partial last ones, with and
without children, strided columns and a table, against the oracle: the leaf kernel's two sets of column
words change roles from block to block, so the last block may lie in either."""
import numpy as np
import pytest

import oracle_lib as O
from hip_lib import SH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hb():
    b = SH.HipBackend(0)
    yield b
    b.close()


@pytest.mark.parametrize("kids", [False, True])
@pytest.mark.parametrize("n", [17, 31, 32, 33, 47, 48, 49, 64, 65, 81])
@pytest.mark.parametrize("log_n", [0, 5, 9])
def test_leaf_blocks(hb, log_n, n, kids):
    print("leaf blocks", log_n, n, kids, flush=True)
    rng = np.random.default_rng(100 * n + log_n + kids)
    words = 1 << log_n
    flat = rng.integers(0, (1 << 31) - 1, n * (words + 1), dtype=np.uint32)
    src = hb.from_cpu(flat)
    prev = rng.integers(0, 1 << 32, 16 * words, dtype=np.uint64).astype(np.uint32) if kids else None
    order = rng.permutation(n)
    for offs in ([i * words for i in range(n)], [int(i) * (words + 1) for i in order]):
        data = [flat[o:o + words] for o in offs]
        exp = O.commit_on_layer(log_n, prev.view(np.uint8) if kids else None, data).view(np.uint32)
        got = hb.commit_on_layer(log_n, hb.from_cpu(prev) if kids else None, [src.ptr + 4 * o for o in offs])
        assert np.array_equal(got.to_cpu(), exp)
