"""Small reads of device memory (batch_at_multi within the argument block, copy_d2h of a column's first
words), which the host awaits by a flag: every size where the route changes, addresses inside a column
and alignment, single words by every route, many reads in a row with work between them that outlasts the
polling, and reads interleaved over two contexts on two threads, each against the same words kept on the
host."""
import ctypes
import threading

import numpy as np
import pytest

from hip_lib import SH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hb():
    b = SH.HipBackend(0)
    yield b
    b.close()


@pytest.mark.parametrize("n_cols,n_rows", [(1, 1), (1, 48), (16, 1), (15, 17), (16, 16), (16, 48), (17, 48), (16, 49), (3, 700)])
def test_gathers(hb, n_cols, n_rows):
    print("gather", n_cols, n_rows, flush=True)
    rng = np.random.default_rng(n_cols * 1000 + n_rows)
    data = rng.integers(0, 1 << 32, (n_cols, 1 << 11), dtype=np.uint64).astype(np.uint32)
    cols = [hb.from_cpu(c) for c in data]
    for _ in range(3):
        rows = rng.integers(0, 1 << 11, n_rows).astype(np.uint32)
        got = np.asarray(hb.batch_at_multi(cols, rows)).reshape(n_rows, n_cols)
        assert (got == data[:, rows].T).all()


@pytest.mark.parametrize("n", [1, 8, 255, 257, 4095, 4096, 4097, 20000])
def test_reads(hb, n):
    print("read", n, flush=True)
    data = np.random.default_rng(n).integers(0, 1 << 32, n + 64, dtype=np.uint64).astype(np.uint32)
    col = hb.from_cpu(data)
    for off in (0, 1, 63):  # an address inside the column is the copy engine's
        out = np.full(n, 7, np.uint32)
        hb._check(hb.lib.stwo_hip_copy_d2h(hb.ctx, out.ctypes.data, col.ptr + 4 * off, n))
        assert (out == data[off:off + n]).all()


@pytest.mark.parametrize("n", [1, 9, 64, 5000])
def test_single_words_by_every_route(hb, n):
    """column_at and channel_read of a column's own address (a kernel reads it) and of addresses that are
    not one of the context's columns: inside a column, and another context's."""
    print("column_at", n, flush=True)
    data = np.random.default_rng(n).integers(0, 1 << 32, n + 1, dtype=np.uint64).astype(np.uint32)
    other = SH.HipBackend(0)
    try:
        mine, theirs = hb.from_cpu(data), other.from_cpu(data)
        other.synchronize()
        word = np.zeros(1, np.uint32)
        digest, draws = ctypes.create_string_buffer(32), ctypes.c_uint32()
        for base in (mine.ptr, theirs.ptr):
            for off in (0, 1):
                for i in sorted({0, n // 2, n - off}):
                    hb._check(hb.lib.stwo_hip_column_at(hb.ctx, base + 4 * off, i, word.ctypes.data_as(SH._U32P)))
                    assert word[0] == data[off + i]
                if n >= 9:
                    hb._check(hb.lib.stwo_hip_channel_read(hb.ctx, base + 4 * off, digest, ctypes.byref(draws)))
                    assert digest.raw == data[off:off + 8].tobytes() and draws.value == data[off + 8]
    finally:
        other.close()


def test_reads_behind_long_work(hb):
    """100 reads (several synchronising ones among them), each of what a transform of 2^22 values left."""
    big = np.random.default_rng(5).integers(0, (1 << 31) - 1, 1 << 22, dtype=np.uint32)
    col = hb.from_cpu(big)
    exp = None
    for i in range(100):
        if i % 10 == 0:
            outs = [hb.interpolate_columns([col], 22)[0] for _ in range(12)]
        got = np.asarray(hb.batch_at_multi([outs[-1]], np.array([0, 1, (1 << 22) - 1], np.uint32))).reshape(-1)
        if exp is None:
            exp = outs[0].to_cpu()
        assert (got == exp[[0, 1, -1]]).all(), i


def test_two_contexts_on_two_threads():
    fails = []

    def work(seed):
        b = SH.HipBackend(0)
        try:
            rng = np.random.default_rng(seed)
            data = rng.integers(0, 1 << 32, (5, 300), dtype=np.uint64).astype(np.uint32)
            cols = [b.from_cpu(c) for c in data]
            for i in range(150):
                rows = rng.integers(0, 300, 1 + i % 48).astype(np.uint32)
                got = np.asarray(b.batch_at_multi(cols, rows)).reshape(len(rows), 5)
                if not (got == data[:, rows].T).all():
                    fails.append((seed, i))
                    return
        finally:
            b.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not fails
