"""Gate and up of a batch in one launch that leaves silu(gate) * up alone (128-row tiles over planes): bit for bit the hidden
states of the two products stored and multiplied by a launch of their own (64-row tiles; Q3_K: the feeding waves' kernel), for
every type with planes, one to five super-blocks, a last row block of 32, token tiles of one to 128 tokens, a down projection
that quantizes h per 256 and per 32, and -- by size alone, no forced route -- a grid that fills the device."""
import numpy as np
import pytest

from helpers import IQ4_XS, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0
from test_gpu_llama import build, f32

pytestmark = pytest.mark.gpu
KEYS = ("gemm_plane_kernel", "gemm_small_max_tokens", "gemm_interleave")


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


def hidden(be, dev, x, one_launch, **tuning):
    """The hidden states, and that both layers' gate and up ran as one launch (or neither's)."""
    try:
        for k, v in tuning.items():
            be.set_tuning(k, v)
        be.kernels_run()
        states = dev.hidden_states(x)
        ran = be.kernels_run()
        print(ran, flush=True)
        assert ran.count("ogm_gemm_swiglu_kernel") == (2 if one_launch else 0)
        return states
    finally:
        for k in KEYS:
            be.set_tuning(k, 0)


@pytest.mark.parametrize("gate,down,n_embd,n_ff,n_tokens", [
    (Q4_K, Q4_K, 256, 512, 33), (Q4_K, Q6_K, 512, 768, 129), (Q4_K, Q8_0, 768, 1056, 257), (Q4_K, Q6_K, 1280, 1280, 65),
    (Q5_K, Q6_K, 512, 512, 128), (Q5_K, Q8_0, 256, 288, 160), (Q6_K, Q6_K, 256, 512, 32), (Q6_K, Q8_0, 768, 800, 130),
    (IQ4_XS, Q4_K, 512, 512, 100), (IQ4_XS, Q8_0, 256, 352, 256), (Q3_K, Q6_K, 512, 512, 96), (Q3_K, Q8_0, 256, 288, 161)])
def test_one_launch_leaves_the_product(be, gate, down, n_embd, n_ff, n_tokens):
    ref, dev, rng = build(be, n_embd=n_embd, n_head=4, n_kv=2, hd=64, n_ff=n_ff, n_vocab=320, n_layer=2,
                          types=(gate, Q8_0, down, Q8_0), max_ctx=n_tokens + 4, seed=n_ff + n_tokens)
    x = rng.standard_normal((n_tokens, n_embd)).astype(f32)
    try:
        got = hidden(be, dev, x, True, gemm_plane_kernel=2, gemm_small_max_tokens=1, gemm_interleave=1)
        want = hidden(be, dev, x, False, gemm_plane_kernel=0 if gate == Q3_K else 2, gemm_small_max_tokens=1, gemm_interleave=2)
        assert np.isfinite(want).all() and np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        dev.close()


def test_by_size(be):
    """1100 tokens over 2 x 2048 rows: 288 workgroups of 128 rows."""
    ref, dev, rng = build(be, n_embd=512, n_head=4, n_kv=2, hd=64, n_ff=2048, n_vocab=320, n_layer=2,
                          types=(Q4_K, Q6_K, Q6_K, Q6_K), max_ctx=1104, seed=3)
    x = rng.standard_normal((1100, 512)).astype(f32)
    try:
        got, want = hidden(be, dev, x, True), hidden(be, dev, x, False, gemm_interleave=2)
        assert np.isfinite(want).all() and np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        dev.close()
