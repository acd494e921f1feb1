"""Proofs whose FRI layers and Merkle levels cross every hand-over of the latency-bound hash kernels (layers
in one launch, chunks of 2^7 leaves and more, one or many chunk roots, levels on quads and on lanes, even
and odd numbers of levels in a subtree), byte for byte the oracle's."""
import pytest

import oracle_lib as O
from hip_lib import SH

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hb():
    b = SH.HipBackend(0)
    yield b
    b.close()


@pytest.mark.parametrize("log_n,fold_step,last", [(k, 1, 0) for k in range(4, 18)] +
                         [(k, s, s - 1) for k in range(6, 13) for s in (2, 3)])
def test_every_fri_size(hb, log_n, fold_step, last):
    print("fri sizes", log_n, fold_step, last, flush=True)
    cfg = dict(pow_bits=3, log_blowup=1, log_last_layer=last, n_queries=4, fold_step=fold_step)
    trace = hb.gen_trace_wide_fibonacci(5, log_n, 1, log_n)
    pr = hb.prove_wide_fibonacci(trace, log_n, SH.PcsConfig.make(3, 1, last, 4, fold_step, 0))
    st, proof, dig, _, _ = O.prove(air="wide_fib", log_n_rows=log_n, n_cols=5, input_mode=1, seed=log_n, **cfg)
    assert pr.status == st == 0
    assert pr.bytes == proof and pr.digest == dig
