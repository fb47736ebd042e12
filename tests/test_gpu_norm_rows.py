"""RMSNorm + quantize over rows of every width: how a row is cut over waves (ogm_launch_norm_quant's rule) against the
one-token launch that prepares the row itself, which is cut another way, and against the rule's own figures."""
import numpy as np
import pytest
import torch

from helpers import Q8_0, captured_launches
from test_gpu_llama import build

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


@pytest.fixture(scope="module")
def stream():
    from orangu_amd import hiprt
    s = hiprt.Stream()
    yield s
    s.destroy()


# (the edges of 1, 2, 3 and 4 runs of 256 a wave; a last run that is partly empty)
@pytest.mark.parametrize("n_embd,waves", [(4096, 16), (4128, 9), (5120, 10), (8192, 16), (8224, 16), (10240, 16), (12288, 16),
                                          (12320, 16), (16384, 16)])
def test_wide_rows(be, stream, n_embd, waves):
    """One token through one layer with norms of their own, and with the norms inside the launches behind them."""
    print(n_embd, flush=True)
    _, dev, rng = build(be, n_embd=n_embd, n_head=2, n_kv=1, hd=64, n_ff=64, n_vocab=40, n_layer=1,
                        types=(Q8_0, Q8_0, Q8_0, Q8_0), max_ctx=8, seed=n_embd)
    x = rng.standard_normal(n_embd).astype(f32)
    xd, lg, tok = torch.from_numpy(x).cuda(), torch.empty(40, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    step = lambda: dev.decode_dev(xd.data_ptr(), 0, lg.data_ptr(), tok.data_ptr(), stream.ptr)
    got = {}
    try:
        for mode in (2, 1):
            be.set_tuning("gemv_prologue", mode)
            step()
            stream.synchronize()
            got[mode] = lg.cpu().numpy(), dev.hidden()
            norms = [k[3] // 64 for k in captured_launches(stream.ptr, step) if k[0] == "ogm_norm_quant_kernel"]
            assert norms == [waves] * (3 if mode == 1 else 1)   # before q/k/v, before gate/up, the output norm
    finally:
        be.set_tuning("gemv_prologue", 0)
        dev.close()
    for a, b in zip(got[1], got[2]):
        assert np.isfinite(a).all()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("n_embd", [4128, 8192, 8224, 12320])
def test_wide_rows_of_a_batch(be, n_embd):
    """Cache rows of 300 tokens (rows of more than 48 runs: two workgroups a compute unit) against parts of 100."""
    print(n_embd, flush=True)
    n = 300
    _, dev, rng = build(be, n_embd=n_embd, n_head=2, n_kv=1, hd=64, n_ff=64, n_vocab=40, n_layer=1,
                        types=(Q8_0, Q8_0, Q8_0, Q8_0), max_ctx=n, seed=n_embd)
    X = rng.standard_normal((n, n_embd)).astype(f32)
    dev.prefill(X, 0)
    whole = [a.copy() for a in dev.kv_read(0, 0, n)]
    for at in range(0, n, 100):
        dev.prefill(X[at:at + 100], at)
    parts = dev.kv_read(0, 0, n)
    dev.close()
    for a, b in zip(whole, parts):
        assert np.array_equal(np.asarray(a), np.asarray(b))
