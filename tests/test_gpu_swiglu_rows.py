"""Gate and up of a decode step in one launch, two row blocks a workgroup: from the first size that takes it (769 and more row
blocks of sixteen rows at 4096 inputs, Q4_K 745) against the last that doesn't, with a down projection per 32 (12320 rows) and per 256, for
each K-quant -- the bits of the step whose norm, products and SwiGLU are launches of their own, and the workgroups launched."""
import numpy as np
import pytest
import torch

from helpers import IQ4_XS, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, Q8_0, captured_launches
from test_gpu_llama import build, f32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


@pytest.mark.parametrize("gate,down,n_ff,workgroups", [(Q4_K, Q6_K, 10240, 640), (Q4_K, Q8_0, 10272, 642), (Q6_K, Q6_K, 10496, 656),
                                                       (Q4_K, Q6_K, 11776, 736), (Q4_K, Q6_K, 12288, 384), (Q6_K, Q6_K, 12288, 768), (Q4_K, Q4_K, 14336, 448),
                                                       (Q5_K, Q8_0, 12320, 385), (Q6_K, Q6_K, 12544, 392), (Q3_K, Q8_0, 12352, 386),
                                                       (IQ4_XS, Q6_K, 12544, 392), (Q2_K, Q6_K, 16384, 512)])
def test_two_row_blocks(be, gate, down, n_ff, workgroups):
    from orangu_amd import hiprt
    _, dev, rng = build(be, n_embd=4096, n_head=4, n_kv=2, hd=64, n_ff=n_ff, n_vocab=320, n_layer=2, types=(gate, gate, down, Q8_0),
                        max_ctx=8, seed=n_ff)
    stream = hiprt.Stream()
    xs = rng.standard_normal((3, 4096)).astype(f32)
    try:
        got = {}
        for mode in (1, 2):
            be.set_tuning("gemv_prologue", mode)
            got[mode] = [a for pos in range(3) for a in (dev.decode(xs[pos], pos)[0], dev.hidden())]
        for one, two in zip(got[1], got[2]):
            assert np.isfinite(one).all() and np.array_equal(one.view(np.uint32), two.view(np.uint32))
        xd, lg, tok = torch.from_numpy(xs[0]).cuda(), torch.empty(320, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        ran = captured_launches(stream.ptr, lambda: dev.decode_dev(xd.data_ptr(), 3, lg.data_ptr(), tok.data_ptr(), stream.ptr))
        swiglu = [k for k in ran if k[0] == "ogm_gemv_fused_kernel" and "Lb1EEv" in k[1]]
        assert [k[2][0] for k in swiglu] == 2 * [workgroups], swiglu
    finally:
        be.set_tuning("gemv_prologue", 0)
        stream.destroy()
        dev.close()
