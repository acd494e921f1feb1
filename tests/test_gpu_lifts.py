"""AccumulationOps in one pass: sums of lifted secure columns of many sizes (more than one launch's
sources among them), equal sizes, the smallest ones, columns off the vector form's alignment, and a source that
holds the destination's own columns, against the
definition out[i] = sum over the columns of col[(i >> (r + 1) << 1) + (i & 1)], r the difference of the log
sizes; and the sums of block results in out-of-domain evaluation, from one block to several waves' worth."""
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


@pytest.mark.parametrize("logs", [[1], [2], [1, 2], [1, 1, 1], [3, 6], [6, 6], [2, 5, 5, 9], [1, 2, 3, 4, 5, 6, 7, 11],
                                  [4] * 13 + [5] * 13 + [7]])
@pytest.mark.parametrize("off", [0, 1, 2])
def test_lift_and_accumulate(hb, logs, off):
    print("lifts", logs, off, flush=True)
    rng = np.random.default_rng(len(logs) * 10 + off)
    L = logs[-1]
    i = np.arange(1 << L)
    cols, exp = [], np.zeros((4, 1 << L), np.uint64)
    for lg in logs:
        data = rng.integers(0, P, (4, 1 << lg), dtype=np.uint32)
        data[:, 0] = P - 1
        r = L - lg
        exp += data[:, i if r == 0 else ((i >> (r + 1)) << 1) + (i & 1)]
        cols.append(data)
    keep = [[hb.from_cpu(np.concatenate([np.zeros(off, np.uint32), c])) for c in d] for d in cols]
    out = [hb.column(off + (1 << L)) for _ in range(4)]
    flat = SH._ptrs([c.ptr + 4 * off for d in keep for c in d])
    ls = np.array(logs, np.uint32)
    hb._check(hb.lib.stwo_hip_lift_and_accumulate(hb.ctx, flat, ls.ctypes.data_as(SH._U32P), len(logs),
                                                  SH._ptrs([c.ptr + 4 * off for c in out])))
    for k in range(4):
        assert np.array_equal(out[k].to_cpu()[off:], (exp[k] % P).astype(np.uint32))


@pytest.mark.parametrize("log_size", [0, 1, 2, 7, 10])
@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("order", [(0, 1, 2, 3), (1, 2, 3, 0), (0, 0, 0, 0)])
def test_accumulate_of_its_own_coordinates(hb, log_size, off, order):
    """The source holds the destination's columns, in any order: every sum is of the old values."""
    print("accumulate own", log_size, off, order, flush=True)
    data = np.random.default_rng(log_size).integers(0, P, (4, 1 << log_size), dtype=np.uint64)
    cols = [hb.from_cpu(np.concatenate([np.zeros(off, np.uint32), c.astype(np.uint32)])) for c in data]
    dst = SH._ptrs([c.ptr + 4 * off for c in cols])
    hb._check(hb.lib.stwo_hip_accumulate(hb.ctx, log_size, dst, SH._ptrs([cols[k].ptr + 4 * off for k in order])))
    for k in range(4):
        assert np.array_equal(cols[k].to_cpu()[off:], ((data[k] + data[order[k]]) % P).astype(np.uint32)), k


@pytest.mark.parametrize("log_size", [3, 11, 12, 17, 19])
def test_block_sums_of_evaluations(hb, log_size):
    rng = np.random.default_rng(log_size)
    n = 3
    cols = [rng.integers(0, P, 1 << log_size, dtype=np.uint32) for _ in range(n)]
    cols[1][:] = P - 1
    point = tuple(int(x) for x in rng.integers(0, P, 8))
    got = hb.batch_eval_at_point([hb.from_cpu(c) for c in cols], log_size, point)
    for c, g in zip(cols, got):
        assert tuple(int(x) for x in O.eval_at_point(c, point)) == g
