"""The low-stage transform kernel on doubles, at the values and sizes where its arithmetic or its tile
loop could go wrong: columns of zeros, of P - 1 and of both in turn (the largest magnitudes that sums and
differences reach), at every tile size, with a single tile, with more tiles than the device holds
workgroups (each loops over several), and on columns 4 bytes off 16-byte alignment."""
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


def extreme_columns(log_n, rng):
    n = 1 << log_n
    i = np.arange(n)
    return [np.full(n, P - 1, np.uint32), np.zeros(n, np.uint32),
            np.where(i & 1, P - 1, 0).astype(np.uint32), np.where(i >> (log_n - 1), P - 1, 1).astype(np.uint32),
            np.where(rng.integers(0, 2, n), P - 1, rng.integers(0, 3, n)).astype(np.uint32)]


@pytest.mark.parametrize("low", [11, 12, 13, 14, 15])
@pytest.mark.parametrize("extra", [0, 1])
def test_extreme_values(hb, low, extra):
    log_n = low + extra
    print("fft extremes", low, log_n, flush=True)
    cols = extreme_columns(log_n, np.random.default_rng(low))
    hb.set_fft_low_log(low)
    try:
        coeffs = hb.interpolate_columns([hb.from_cpu(c) for c in cols], log_n)
        again = hb.evaluate_polynomials(coeffs, log_n, 0)
        wide = hb.evaluate_polynomials([hb.from_cpu(c) for c in cols], log_n, 1)
    finally:
        hb.set_fft_low_log(0)
    for c, cf, a, w in zip(cols, coeffs, again, wide):
        assert np.array_equal(cf.to_cpu(), O.interpolate(c))
        assert np.array_equal(a.to_cpu(), c)
        assert np.array_equal(w.to_cpu(), O.evaluate(c, log_n + 1))


@pytest.mark.parametrize("low,n_cols", [(11, 141), (13, 37), (15, 9)])
def test_more_tiles_than_workgroups(hb, low, n_cols):
    """About 4500 tiles of 2^11, 1180 of 2^13 and 290 of 2^15 on unaligned columns."""
    log_n = 16 if low < 15 else 20
    print("fft loop", low, log_n, n_cols, flush=True)
    n = 1 << log_n
    rng = np.random.default_rng(n_cols)
    data = rng.integers(0, P, 1 + n_cols * n, dtype=np.uint32)
    src = hb.from_cpu(data)
    mid, dst = hb.column(1 + n_cols * n), hb.column(1 + n_cols * n)
    at = [[c.ptr + 4 * (1 + i * n) for i in range(n_cols)] for c in (src, mid, dst)]
    hb.set_fft_low_log(low)
    try:
        hb.interpolate_columns(at[0], log_n, out=at[1])
        hb.evaluate_polynomials(at[1], log_n, 0, out=at[2])
    finally:
        hb.set_fft_low_log(0)
    assert np.array_equal(dst.to_cpu()[1:], data[1:])
    coeffs = mid.to_cpu()[1:]
    for i in (0, n_cols // 2, n_cols - 1):
        assert np.array_equal(coeffs[i * n:(i + 1) * n], O.interpolate(data[1 + i * n:1 + (i + 1) * n]))
