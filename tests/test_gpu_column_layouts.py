"""How a call's columns lie in memory never changes its results: rows of one allocation (no address
table), the same rows backwards, one source column given several times, scattered columns, columns at an
odd distance, and more columns than a launch's arguments hold, against the oracle. Transforms in one
kernel, in several passes and below the LDS kernels' sizes; Merkle layers of 0..17 and 40 columns on both
sides of the 16 that travel as arguments."""
import numpy as np
import pytest

import oracle_lib as O
from hip_lib import SH

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


@pytest.fixture(scope="module")
def hb():
    b = SH.HipBackend(0)
    yield b
    b.close()


def layouts(n, words):
    """name -> word offsets of n columns in one allocation."""
    rng = np.random.default_rng(words + n)
    gap = words + 3
    return {"rows": [i * words for i in range(n)], "backwards": [(n - 1 - i) * words for i in range(n)],
            "odd distance": [1 + i * gap for i in range(n)], "scattered": [int(x) * gap for x in rng.permutation(n)]}


@pytest.mark.parametrize("log_n,n", [(3, 5), (7, 6), (12, 5), (16, 3), (11, 300)])
def test_transforms(hb, log_n, n):
    print("layouts", log_n, n, flush=True)
    words = 1 << log_n
    rng = np.random.default_rng(log_n * 1000 + n)
    data = rng.integers(0, P, (n, words), dtype=np.uint32)
    check = sorted({0, 1, n // 2, n - 1})
    coeffs = {i: O.interpolate(data[i]) for i in check}
    evals = {i: O.evaluate(coeffs[i], log_n + 1) for i in check}
    src_l, mid_l, dst_l = layouts(n, words), layouts(n, words), layouts(n, 2 * words)
    for name in src_l:
        flat = np.zeros((words + 3) * n + 8, np.uint32)
        for i, o in enumerate(src_l[name]):
            flat[o:o + words] = data[i]
        src = hb.from_cpu(flat)
        mid, dst = hb.column((words + 3) * n + 8), hb.column((2 * words + 3) * n + 8)
        # inputs and outputs laid out differently, so that both kinds meet in one call
        other = {"rows": "scattered", "scattered": "rows", "backwards": "odd distance", "odd distance": "backwards"}[name]
        mids = [mid.ptr + 4 * o for o in mid_l[other]]
        hb.interpolate_columns([src.ptr + 4 * o for o in src_l[name]], log_n, out=mids)
        hb.evaluate_polynomials(mids, log_n, 1, out=[dst.ptr + 4 * o for o in dst_l[name]])
        got_c, got_e = mid.to_cpu(), dst.to_cpu()
        for i in check:
            o = mid_l[other][i]
            assert np.array_equal(got_c[o:o + words], coeffs[i]), (name, i)
            o = dst_l[name][i]
            assert np.array_equal(got_e[o:o + 2 * words], evals[i]), (name, i)


def test_one_source_for_every_column(hb):
    log_n, n = 11, 4
    rng = np.random.default_rng(3)
    c = rng.integers(0, P, 1 << log_n, dtype=np.uint32)
    src, out = hb.from_cpu(c), hb.column(n << (log_n + 1))
    hb.evaluate_polynomials([src.ptr] * n, log_n, 1, out=[out.ptr + 4 * (i << (log_n + 1)) for i in range(n)])
    exp = O.evaluate(c, log_n + 1)
    assert np.array_equal(out.to_cpu(), np.tile(exp, n))


@pytest.mark.parametrize("n", [0, 1, 2, 15, 16, 17, 40])
@pytest.mark.parametrize("with_prev", [False, True])
def test_merkle_layers(hb, n, with_prev):
    log_n = 5
    words = 1 << log_n
    rng = np.random.default_rng(n)
    data = rng.integers(0, P, (n, words), dtype=np.uint32)
    prev = rng.integers(0, 1 << 32, 16 << log_n, dtype=np.uint64).astype(np.uint32) if with_prev else None
    exp = O.commit_on_layer(log_n, None if prev is None else prev.view(np.uint8), list(data)).view(np.uint32)
    for name, offs in layouts(n, words).items():
        flat = np.zeros((words + 3) * n + 8, np.uint32)
        for i, o in enumerate(offs):
            flat[o:o + words] = data[i]
        src = hb.from_cpu(flat)
        got = hb.commit_on_layer(log_n, hb.from_cpu(prev) if with_prev else None, [src.ptr + 4 * o for o in offs])
        assert np.array_equal(got.to_cpu(), exp), name
