"""Which kernel a K-quant batch takes by its size alone, on both sides of each line between the small-batch kernel, the 64-row
and the 128-row tiles over planes and the kernels without planes (weights of zero bytes; the kernels' values are compared in
their own tests)."""
import numpy as np
import pytest
import torch

from helpers import BLOCK, IQ4_XS, Q4_K, Q5_K, Q6_K, TYPE_NAME

pytestmark = pytest.mark.gpu
SB, X64, X128, MED, FEED = "ogm_gemm_sb_%s_kernel", "ogm_gemm_%s_dmx_kernel", "ogm_gemm_%s_dma_kernel", "ogm_gemm_sbw_%s_kernel", "ogm_gemm_%s_i8p"


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


def kernel(be, t, in_dim, outs, tokens):
    bytes_, elems = BLOCK[t]
    ws = [be.upload_raw(np.zeros(o * (in_dim // elems) * bytes_, np.uint8), t, in_dim, o) for o in outs]
    x, ys = torch.ones(tokens, in_dim, device="cuda"), [torch.empty(tokens, o, device="cuda") for o in outs]
    torch.cuda.synchronize()
    be.matmul_multi_dev(ws, x.data_ptr(), tokens, [y.data_ptr() for y in ys], False)
    torch.cuda.synchronize()
    name = be.last_kernel()
    for w in ws:
        be.free_weight(w)
    print(t, in_dim, outs, tokens, name, flush=True)
    return name


# (rounds of the small-batch kernel's workgroups of 32 rows x 32 tokens: three, Q4_K from 6144 inputs on four)
@pytest.mark.parametrize("t,in_dim,outs,tokens,want", [
    (Q4_K, 4096, (4096,), 192, SB), (Q4_K, 4096, (4096,), 193, X64), (Q5_K, 4096, (4096,), 192, SB), (Q5_K, 11008, (4096,), 193, X64),
    (Q4_K, 11008, (4096,), 256, SB), (Q4_K, 14336, (5120,), 192, SB), (Q4_K, 14336, (5120,), 193, X64), (Q5_K, 14336, (5120,), 160, X64),
    (Q4_K, 6144, (6144,), 160, SB), (Q4_K, 6144, (6144,), 161, X64), (Q4_K, 5120, (4608,), 160, SB), (Q5_K, 5120, (4608,), 160, SB),
    (Q4_K, 5120, (4608,), 161, X64), (Q4_K, 4096, (3072, 1024), 130, SB), (Q4_K, 8192, (5000,), 160, SB), (Q5_K, 8192, (5000,), 160, X64),
    (Q4_K, 2048, (5120,), 160, X64), (Q4_K, 2048, (5056,), 160, MED)])
def test_two_token_tiles(be, t, in_dim, outs, tokens, want):
    assert kernel(be, t, in_dim, outs, tokens) == want % TYPE_NAME[t].replace("_", "")


# (64-row workgroups: from 160, Q6_K 128, to 512, Q4_K and Q5_K over rows of 4096 inputs and more to 256, and 128-row ones beyond)
@pytest.mark.parametrize("t,in_dim,outs,tokens,want", [
    (Q4_K, 4096, (4096,), 512, X64), (Q4_K, 4096, (4160,), 512, X128), (Q5_K, 8192, (5440,), 300, X64), (Q5_K, 8192, (5504,), 300, X128),
    (Q4_K, 2048, (8192,), 512, X64), (Q4_K, 2048, (8256,), 512, X128), (Q4_K, 2048, (3456,), 300, X64), (Q4_K, 2048, (3392,), 300, FEED),
    (Q6_K, 4096, (4096,), 160, X64), (Q6_K, 4096, (4032,), 160, SB), (Q6_K, 4096, (8192,), 512, X64), (Q6_K, 4096, (8256,), 512, X128),
    (IQ4_XS, 4096, (8192,), 512, X64), (IQ4_XS, 4096, (8256,), 512, X128)])
def test_row_tiles_over_planes(be, t, in_dim, outs, tokens, want):
    got = kernel(be, t, in_dim, outs, tokens)
    assert got.startswith(want % TYPE_NAME[t].replace("_", "")) if want == FEED else got == want % TYPE_NAME[t].replace("_", "")
