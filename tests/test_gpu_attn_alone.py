"""The decode step's attention where one workgroup holds a head's whole cache and finishes it by itself: at the first and the
last context of each chunk (64, 128 and, with heads of 64, 256 positions, two to four threads) and just beyond, over head
counts that fill the kernel's head slots in runs of the quantizer's 256 or 32 -- against the forward pass of the oracle, as
every decode step is checked, and by the workgroups the launch has."""
import numpy as np
import pytest
import torch

from helpers import Q4_K, Q6_K, Q8_0, captured_launches
from test_gpu_llama import build, f32, fill_cache_both, step_both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


# (n_pre: cached positions before the first of two steps; splits: workgroups a K/V head at the second)
@pytest.mark.parametrize("hd,group,n_kv,wo,n_pre,splits", [
    (64, 4, 2, Q4_K, 0, 1), (64, 4, 2, Q4_K, 62, 1), (64, 4, 2, Q4_K, 63, 1), (64, 4, 2, Q4_K, 126, 1), (64, 4, 2, Q4_K, 127, 1),
    (64, 8, 1, Q4_K, 180, 1), (64, 4, 1, Q4_K, 253, 1), (64, 4, 2, Q4_K, 254, 1), (64, 4, 2, Q4_K, 255, 5),
    (64, 1, 8, Q8_0, 130, 1), (64, 2, 4, Q8_0, 254, 1), (64, 2, 2, Q4_K, 100, 2),
    (128, 4, 2, Q4_K, 63, 1), (128, 2, 2, Q4_K, 126, 1), (128, 4, 1, Q4_K, 127, 3), (128, 8, 1, Q4_K, 90, 1), (128, 1, 2, Q8_0, 70, 1)])
def test_one_workgroup_a_head(be, hd, group, n_kv, wo, n_pre, splits):
    from orangu_amd import hiprt
    n_head, n_embd = group * n_kv, 256
    types = (Q4_K, Q6_K, Q6_K, Q6_K) if wo == Q4_K else (Q8_0, Q8_0, Q8_0, Q8_0)
    ref, dev, rng = build(be, n_embd=n_embd, n_head=n_head, n_kv=n_kv, hd=hd, n_ff=512, n_vocab=320, n_layer=1, types=types,
                          max_ctx=n_pre + 4, seed=23)
    stream = hiprt.Stream()
    try:
        if n_pre:
            fill_cache_both(ref, dev, rng, 1, n_pre, n_kv * hd)
        x = rng.standard_normal((2, n_embd)).astype(f32)
        for i in range(2):
            step_both(ref, dev, x[i], n_pre + i, f"context {n_pre + i}", attn_rtol=1e-5)
        xd, lg, tok = torch.from_numpy(x[1]).cuda(), torch.empty(320, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
        torch.cuda.synchronize()
        ran = captured_launches(stream.ptr, lambda: dev.decode_dev(xd.data_ptr(), n_pre + 1, lg.data_ptr(), tok.data_ptr(), stream.ptr))
        attn = [k for k in ran if k[0] == "ogm_attn_kernel"]
        assert len(attn) == 1 and tuple(attn[0][2][:2]) == (n_kv, splits), attn
    finally:
        stream.destroy()
        dev.close()
