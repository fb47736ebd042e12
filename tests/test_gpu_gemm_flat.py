"""The tiled GEMM of the symmetric per-32 types, whose scale products ad * dw come from a matrix instruction: every bit of
the CPU restatement at the edges of its tiles (128 rows x 128 tokens, two blocks a stage), with scales whose product is
subnormal, zero or beyond the range, and with rows and tokens of infinities that must not reach their neighbours."""
import numpy as np
import pytest

import oracle
from helpers import BLOCK, IQ4_NL, Q4_0, Q5_0, Q8_0, synth_weights

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    b.set_tuning("gemm_small_max_tokens", 1)   # the tiled kernel whatever the batch
    yield b
    b.close()


@pytest.mark.parametrize("t", [Q8_0, Q5_0, Q4_0, IQ4_NL])
@pytest.mark.parametrize("in_dim,out_dim,tokens", [(64, 5, 17), (192, 128, 129), (1024, 200, 33), (4160, 129, 128)])
def test_scale_products(be, t, in_dim, out_dim, tokens):
    from orangu_amd import QuantMatrix
    print(t, in_dim, out_dim, tokens, flush=True)
    rng = np.random.default_rng(in_dim + t)
    raw = np.array(synth_weights(t, in_dim, out_dim, seed=t + in_dim), np.uint8)
    blocks = raw.reshape(out_dim, in_dim // 32, BLOCK[t][0])
    d = (2e-3 * rng.standard_normal(blocks.shape[:2])).astype(np.float16)
    d[0] = np.float16(6e-8)                       # the smallest subnormal
    d[min(3, out_dim - 1)] = np.float16(65504)
    d[min(4, out_dim - 1), 0] = np.float16(np.inf)
    d[1, :] = np.float16(-0.0)
    blocks[:, :, :2] = d[..., None].view(np.uint8)
    x = rng.standard_normal((tokens, in_dim)).astype(np.float32)
    x[1] *= np.float32(1e-36)                     # scales of about 1e-38: products with dw are subnormal
    x[2] *= np.float32(1e-41)                     # a subnormal scale
    x[3] *= np.float32(1e36)
    x[4] = 0.0
    x[5, 7] = np.inf
    x[6, 9] = np.nan
    y = be.matmul(x, tokens, QuantMatrix(raw, t, in_dim, out_dim)).reshape(tokens, out_dim)
    assert be.last_kernel() == "ogm_gemm_flat_kernel"
    want = oracle.matmul(t, raw, in_dim, out_dim, x, tokens).reshape(tokens, out_dim)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(y[~nan].view(np.uint32), want[~nan].view(np.uint32))
