"""The small-batch GEMM of Q4_K and Q5_K, whose waves ask for a round's operands a round ahead: rows of one super-block, of a
round of eight or sixteen less one, exactly, and more by one, of two rounds and the first remainder behind them (where Q5_K
changes over), with idle waves in the last round, activations row by row (few tokens) and in operand chunks, one to three token
tiles and rows that end inside a tile -- bit for bit the CPU path's results."""
import numpy as np
import pytest

import oracle
from helpers import Q4_K, Q5_K, synth_weights, synth_x

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


@pytest.mark.parametrize("waves", [8, 16])
@pytest.mark.parametrize("t", [Q4_K, Q5_K])
@pytest.mark.parametrize("nsb,rows,tokens", [(1, 70, 9), (2, 33, 40), (7, 32, 17), (8, 100, 31), (9, 64, 32), (15, 40, 65), (16, 96, 33),
                                             (17, 33, 20), (24, 64, 12), (31, 32, 64), (32, 70, 9), (33, 40, 77), (43, 64, 33)])
def test_rounds(be, t, waves, nsb, rows, tokens):
    from orangu_amd import QuantMatrix
    in_dim = 256 * nsb
    raw = np.ascontiguousarray(synth_weights(t, in_dim, rows, seed=nsb * 100 + rows))
    x = synth_x(tokens, in_dim, seed=tokens)
    want = np.asarray(oracle.matmul(t, raw, in_dim, rows, x, tokens), np.float32).reshape(-1)
    tuning = {"gemm_min_tokens": 2, "gemm_small_max_tokens": 512, "gemm_sb_waves": waves, "gemv_mma": 0}
    try:
        for k, v in tuning.items():
            be.set_tuning(k, v)
        got = np.asarray(be.matmul(x, tokens, QuantMatrix(raw, t, in_dim, rows)), np.float32).reshape(-1)
        assert be.last_kernel() == f"ogm_gemm_sb_{'q4k' if t == Q4_K else 'q5k'}{'_w16' if waves == 16 else ''}_kernel"
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        for k, v in {"gemm_min_tokens": 0, "gemm_small_max_tokens": 0, "gemm_sb_waves": 0, "gemv_mma": 1}.items():
            be.set_tuning(k, v)
