"""Poseidon252 layers on both sides of the node count where the kernel with a node on 16 lanes hands
over to the one with a node on a lane: children alone, columns alone and both, whole last waves and
partial ones, against the restatement at the first, the last and some nodes between; children at the
ends of the word range, where the carries of the signed limbs are longest; the two kernels agree on
the nodes that a small layer shares with a large one."""
import numpy as np
import pytest

import p252 as Q
from hip_lib import SH

pytestmark = pytest.mark.gpu
M31 = (1 << 31) - 1


@pytest.fixture(scope="module")
def hb():
    b = SH.HipBackend(0)
    yield b
    b.close()


def felts_at(col, nodes):
    w = col.to_cpu()
    return [SH.felt252_from_words(w[8 * i:8 * i + 8]) for i in nodes]


@pytest.mark.parametrize("log_size,n_cols,kids", [
    (0, 7, True), (1, 0, True), (1, 17, False), (2, 24, True), (6, 0, True),
    (13, 3, False), (13, 9, True), (14, 0, True), (14, 9, True), (15, 0, True), (15, 16, False)])
def test_layers_around_the_handover(hb, log_size, n_cols, kids):
    print("poseidon252 rows", log_size, n_cols, kids, flush=True)
    rng = np.random.default_rng(900 + log_size * 40 + n_cols)
    n = 1 << log_size
    prev = None
    if kids:
        words = rng.integers(0, 1 << 32, (2 * n, 8), dtype=np.uint64).astype(np.uint32)
        words[:, 7] >>= 5  # below 2^251
        prev = hb.from_cpu(words.reshape(-1))
    cols = [rng.integers(0, M31, n, dtype=np.uint32) for _ in range(n_cols)]
    out = hb.commit_on_layer_poseidon252(log_size, prev, [hb.from_cpu(c) for c in cols])
    nodes = sorted({0, n - 1, n // 2, n // 3} | {int(x) for x in rng.integers(0, n, 4)})
    exp = []
    for i in nodes:
        pair = tuple(SH.felt252_from_words(words[2 * i + j]) for j in (0, 1)) if kids else None
        exp.append(Q.hash_node(pair, [int(c[i]) for c in cols]))
    assert felts_at(out, nodes) == exp


def test_children_at_the_ends_of_the_range(hb):
    print("poseidon252 rows, extreme children", flush=True)
    p = Q.P
    limbs = [sum(v << 29 * i for i in range(8)) for v in ((1 << 29) - 1, 1 << 28, (1 << 28) - 1)]
    ends = [0, 1, 2, p - 1, p - 2, p >> 1, (p >> 1) + 1, (1 << 251) - 1, 17 << 192] + limbs
    kids = [(a, b) for a in ends for b in ends][:128]
    flat = [k for pair in kids for k in pair]
    prev = hb.from_cpu(np.concatenate([SH.felt252_to_words(k) for k in flat]))
    out = hb.commit_on_layer_poseidon252(7, prev, [])
    assert felts_at(out, range(128)) == [Q.hash_node(pair, []) for pair in kids]


def test_small_layer_is_a_prefix_of_a_large_one(hb):
    print("poseidon252 rows, prefix", flush=True)
    rng = np.random.default_rng(77)
    big, small = 16, 12
    words = rng.integers(0, 1 << 32, (2 << big, 8), dtype=np.uint64).astype(np.uint32)
    words[:, 7] >>= 5
    cols = [rng.integers(0, M31, 1 << big, dtype=np.uint32) for _ in range(11)]
    for c in (cols, []):
        full = hb.commit_on_layer_poseidon252(big, hb.from_cpu(words.reshape(-1)), [hb.from_cpu(x) for x in c])
        part = hb.commit_on_layer_poseidon252(small, hb.from_cpu(words[:2 << small].reshape(-1)),
                                              [hb.from_cpu(x[:1 << small]) for x in c])
        assert (full.to_cpu()[:8 << small] == part.to_cpu()[:8 << small]).all()
