"""The low-stage transform kernel on doubles, at the values and sizes where its arithmetic or its tile
loop could go wrong: columns of zeros, of P - 1 and of both in turn (the largest magnitudes that sums and
differences reach), at every tile size, with a single tile, with more tiles than the device holds
workgroups (each loops over several), and on columns 4 bytes off 16-byte alignment."""
import glob

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


def compute_units():
    """Of the largest GPU that the kernel driver lists."""
    best = 0
    for f in glob.glob("/sys/class/kfd/kfd/topology/nodes/*/properties"):
        v = dict(line.split() for line in open(f) if len(line.split()) == 2)
        best = max(best, int(v.get("simd_count", 0)) // max(1, int(v.get("simd_per_cu", 4))))
    return best or 256


@pytest.mark.parametrize("low", [11, 12, 13, 14, 15])
@pytest.mark.parametrize("above", [0, 2])
def test_more_tiles_than_workgroups(hb, low, above):
    """Foreground launches have at most as many workgroups as the device holds at once: here each runs two
    or three tiles, an uneven number to an XCD; tiles that are whole columns, and four to a column; unaligned
    columns; forward onto the same domain and, where a tile is a column, onto the twice larger one (two tiles
    that read the same coefficients)."""
    resident = (compute_units() // 8 * 8) << (15 - low)
    n_cols = (resident * 9 // 4 >> above) | 1
    tiles, log_n = n_cols << above, low + above
    assert 2 * resident < tiles < 3 * resident and tiles % 8
    print("fft loop", low, log_n, n_cols, resident, flush=True)
    n = 1 << log_n
    data = np.random.default_rng(n_cols).integers(0, P, 1 + n_cols * n, dtype=np.uint32)
    blow = 1 if above == 0 else 0
    src, mid, dst = hb.from_cpu(data), hb.column(1 + n_cols * n), hb.column(1 + (n_cols * n << blow))
    at = lambda c, b=0: [c.ptr + 4 * (1 + (i * n << b)) for i in range(n_cols)]
    hb.set_fft_low_log(low)
    try:
        hb.interpolate_columns(at(src), log_n, out=at(mid))
        hb.evaluate_polynomials(at(mid), log_n, 0, out=at(dst))
        again = dst.to_cpu()[1:1 + n_cols * n]
        if blow:
            hb.evaluate_polynomials(at(mid), log_n, 1, out=at(dst, 1))
    finally:
        hb.set_fft_low_log(0)
    assert np.array_equal(again, data[1:])
    coeffs, wide = mid.to_cpu()[1:], dst.to_cpu()[1:]
    # columns at the ends of the XCDs' ranges
    for i in sorted({min(n_cols - 1, (n_cols * x >> 3) + d) for x in range(9) for d in (0, 1)} | {n_cols - 2}):
        c = O.interpolate(data[1 + i * n:1 + (i + 1) * n])
        assert np.array_equal(coeffs[i * n:(i + 1) * n], c), i
        if blow:
            assert np.array_equal(wide[2 * i * n:2 * (i + 1) * n], O.evaluate(c, log_n + 1)), i
