"""Batches over the per-32 types' rows of any number of blocks: one block, odd counts in tiles one block wide, counts that fill
a tile of four with zero blocks, and counts that leave the tiled kernel's last piece of four short -- through the small-batch
kernel, both widths of the tiled kernel (four row blocks of 32 a workgroup need the launch of many) and the f16 one.  Every bit
of the CPU restatement; scales of infinities in a row's last block must not meet the blocks the piece does not have."""
import numpy as np
import pytest

import oracle
from helpers import BLOCK, IQ4_NL, Q4_0, Q5_0, Q5_1, Q8_0, TYPE_NAME, synth_weights, synth_x

pytestmark = pytest.mark.gpu

FLAT = (Q8_0, Q4_0, Q5_0, IQ4_NL)


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


def check(be, t, in_dim, out_dim, tokens, kernel, tiled, raw=None, x=None):
    from orangu_amd import QuantMatrix
    print(TYPE_NAME[t], in_dim, out_dim, tokens, kernel, flush=True)
    raw = synth_weights(t, in_dim, out_dim, seed=in_dim + t) if raw is None else raw
    x = synth_x(tokens, in_dim, seed=tokens) if x is None else x
    be.set_tuning("gemm_small_max_tokens", 1 if tiled else 0)
    try:
        y = be.matmul(x, tokens, QuantMatrix(raw, t, in_dim, out_dim)).reshape(tokens, out_dim)
        assert be.last_kernel() == kernel
    finally:
        be.set_tuning("gemm_small_max_tokens", 0)
    want = oracle.matmul(t, raw, in_dim, out_dim, x, tokens).reshape(tokens, out_dim)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(y[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("nblk,out_dim,tokens", [(1, 3, 9), (3, 70, 17), (5, 33, 40), (27, 40, 33), (43, 31, 20)])
@pytest.mark.parametrize("t", FLAT + (Q5_1,))
def test_small_batches(be, t, nblk, out_dim, tokens):
    if t == Q5_1:
        nblk = max(nblk, 9)   # (rows of a few blocks stay on the GEMV kernel)
    check(be, t, 32 * nblk, out_dim, tokens, "ogm_gemm_sb_flat_kernel", False)


@pytest.mark.parametrize("nblk,out_dim,tokens", [(1, 3, 17), (3, 70, 129), (5, 65, 33), (6, 130, 64), (27, 128, 97), (31, 129, 32), (43, 61, 200)])
@pytest.mark.parametrize("t", FLAT)
def test_two_row_blocks(be, t, nblk, out_dim, tokens):
    check(be, t, 32 * nblk, out_dim, tokens, "ogm_gemm_flat_kernel", True)


@pytest.mark.parametrize("t,nblk,kernel", [(Q8_0, 1, "ogm_gemm_flat_kernel"), (Q8_0, 3, "ogm_gemm_flat_kernel"), (Q8_0, 6, "ogm_gemm_flat_kernel"),
                                           (Q8_0, 7, "ogm_gemm_flat_kernel"), (Q4_0, 3, "ogm_gemm_flat_kernel"), (Q5_0, 5, "ogm_gemm_flat_kernel"),
                                           (IQ4_NL, 3, "ogm_gemm_flat_kernel"), (Q4_0, 2, "ogm_gemm_flat_f16_kernel"),
                                           (Q5_0, 4, "ogm_gemm_flat_f16_kernel"), (IQ4_NL, 2, "ogm_gemm_flat_f16_kernel")])
def test_four_row_blocks_and_f16(be, t, nblk, kernel):
    check(be, t, 32 * nblk, 4101, 1701, kernel, False)   # 33 x 14 tiles of 128 x 128


@pytest.mark.parametrize("t", FLAT)
def test_blocks_past_the_end(be, t):
    """Infinite and not-a-number scales in the last block, whose bytes the missing blocks of the last piece repeat."""
    nblk, out_dim, tokens = 5, 66, 40
    raw = np.array(synth_weights(t, 32 * nblk, out_dim, seed=t), np.uint8)
    blocks = raw.reshape(out_dim, nblk, BLOCK[t][0])
    blocks[3, -1, :2] = np.frombuffer(np.float16(np.inf).tobytes(), np.uint8)
    blocks[40, -1, :2] = np.frombuffer(np.float16(65504).tobytes(), np.uint8)
    x = synth_x(tokens, 32 * nblk, seed=5).reshape(tokens, 32 * nblk)
    x[7, -1] = np.inf
    x[9, -2] = np.float32(3e38)
    check(be, t, 32 * nblk, out_dim, tokens, "ogm_gemm_flat_kernel", True, raw=raw, x=x)
