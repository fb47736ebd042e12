"""The K-quant GEMMs over prebuilt planes (128-row and 64-row tiles) at the edges of what they are built from: one to five
super-blocks a row (the ring of pieces, the two register sets of a super-block's activations and the table slots turn at
different numbers of them), row blocks of 32 past the matrix, token blocks of 32 that are ragged or missing (their waves
only fetch), several matrices a launch, and scales whose product with dmin, formed on the matrix cores, is subnormal,
infinite or not a number.  Every bit of the CPU restatement."""
import numpy as np
import pytest
import torch

import oracle
from helpers import BLOCK, F16_FIELDS, IQ4_XS, Q3_K, Q4_K, Q5_K, Q6_K, TYPE_NAME, captured_launches, synth_weights, synth_x

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    b.set_tuning("gemm_small_max_tokens", 1)   # the kernels over planes whatever the launch
    b.set_tuning("gemm_medium", 1)
    b.set_tuning("gemm_plane_kernel", 2)
    yield b
    b.close()


def check(be, t, raw, in_dim, out_dim, x, tokens, rows64):
    from orangu_amd import QuantMatrix
    print(TYPE_NAME[t], in_dim, out_dim, tokens, rows64, flush=True)
    be.set_tuning("gemm_interleave", 2 if rows64 else 1)
    y = be.matmul(x, tokens, QuantMatrix(raw, t, in_dim, out_dim)).reshape(tokens, out_dim)
    assert be.last_kernel().endswith("_dmx_kernel" if rows64 else "_dma_kernel")
    want = oracle.matmul(t, raw, in_dim, out_dim, x, tokens).reshape(tokens, out_dim)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(y), nan)
    assert np.array_equal(y[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("rows64", [False, True])
@pytest.mark.parametrize("nsb,out_dim,tokens", [(1, 1, 32), (2, 33, 65), (3, 97, 128), (4, 129, 33), (5, 200, 161), (7, 64, 300)])
@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, IQ4_XS, Q3_K])
def test_edges(be, t, nsb, out_dim, tokens, rows64):
    if t == Q3_K and rows64:
        pytest.skip("Q3_K has 128-row tiles only")
    raw = synth_weights(t, 256 * nsb, out_dim, seed=nsb + t)
    check(be, t, raw, 256 * nsb, out_dim, synth_x(tokens, 256 * nsb, seed=tokens), tokens, rows64)


@pytest.mark.parametrize("rows64", [False, True])
@pytest.mark.parametrize("t", [Q4_K, Q5_K])
def test_min_products(be, t, rows64):
    nsb, out_dim, tokens = 3, 70, 40
    rng = np.random.default_rng(t)
    raw = np.array(synth_weights(t, 256 * nsb, out_dim, seed=t + 1), np.uint8)
    blocks = raw.reshape(out_dim, nsb, BLOCK[t][0])
    at = F16_FIELDS[t][1]
    dmin = (2e-3 * rng.standard_normal((out_dim, nsb))).astype(np.float16)
    dmin[0] = np.float16(6e-8)                    # the smallest subnormal
    dmin[1] = np.float16(-0.0)
    dmin[2] = np.float16(65504)
    dmin[3, 1] = np.float16(np.inf)
    blocks[:, :, at:at + 2] = dmin[..., None].view(np.uint8)
    x = rng.standard_normal((tokens, 256 * nsb)).astype(np.float32)
    x[1] *= np.float32(1e-36)                     # scales of about 1e-38: products with dmin are subnormal
    x[2] *= np.float32(1e-41)                     # a subnormal scale
    x[3] *= np.float32(1e36)
    x[4] = 0.0
    x[5, 7] = np.inf
    x[6, 9] = np.nan
    check(be, t, raw, 256 * nsb, out_dim, x, tokens, rows64)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K, IQ4_XS, Q3_K])
def test_planes_are_one_launch(be, t):
    """A matrix's first tiled call: the quantizer, one launch that builds all that the GEMM reads of the matrix, the GEMM."""
    from orangu_amd import hiprt
    in_dim, out_dim, tokens = 512, 200, 130
    raw = synth_weights(t, in_dim, out_dim, seed=t)
    first, second = (be.upload_raw(raw, t, in_dim, out_dim) for _ in range(2))
    x, y = torch.ones(tokens, in_dim, device="cuda"), torch.empty(tokens, out_dim, device="cuda")
    torch.cuda.synchronize()
    stream = hiprt.Stream()
    be.set_tuning("gemm_interleave", 1)
    be.matmul_dev(first, x.data_ptr(), tokens, y.data_ptr(), False, stream.ptr)   # (allocates the scratch)
    stream.synchronize()
    ran = captured_launches(stream.ptr, lambda: be.matmul_dev(second, x.data_ptr(), tokens, y.data_ptr(), False, stream.ptr), relaxed=True)
    be.free_weight(first)
    be.free_weight(second)   # (its planes were never filled)
    stream.destroy()
    print(t, [k[0] for k in ran], flush=True)
    assert [k[0] for k in ran[1:]] == ["ogm_gemm_build_planes_kernel", "ogm_gemm_dma_kernel"]
