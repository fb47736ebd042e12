"""The quantizers' largest magnitude skips a NaN whatever its payload (`fold(0f32, |m, v| m.max(v.abs()))`,
vecdot.rs:103 / 3037): a signalling NaN in a caller's row leaves its group's scale, and so every other value, as a quiet
one does.  (v_max_f32 answers a signalling NaN with a NaN, so a maximum without care would lose what came before it.)"""
import numpy as np
import pytest
import torch

import oracle
from helpers import Q2_K, Q4_K, Q5_1, Q6_K, Q8_0, synth_weights

pytestmark = pytest.mark.gpu
SIGNALLING, QUIET = np.uint32(0x7FA00001), np.uint32(0x7FC00000)


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


def rows(n_tokens, n, payload, seed):
    """Rows whose largest value of each 32 (and a larger one of each 256) has NaNs before, beside and after it."""
    x = np.random.default_rng(seed).standard_normal((n_tokens, n)).astype(np.float32)
    for t in range(n_tokens):
        for g in range(0, n, 32):
            k = g // 32 + t
            x[t, g + k % 32] = 20.0 if k % 8 == t % 8 else 9.0
            for step in (1, 2, 3, 5, 17)[:1 + k % 5]:
                x.view(np.uint32)[t, g + (k + step) % 32] = payload | np.uint32(0x80000000 * (k & 1))
    return x


# (one token: prepared inside the GEMV and after a quantizer launch; a few; batches with and without operand chunks)
@pytest.mark.parametrize("t", [Q4_K, Q6_K, Q2_K, Q8_0, Q5_1])
@pytest.mark.parametrize("n_tokens,prologue", [(1, 2), (1, 1), (5, 0), (24, 0), (40, 0)])
def test_a_signalling_nan_is_skipped(be, t, n_tokens, prologue):
    in_dim, out_dim = 1280, 70
    print(t, n_tokens, prologue, flush=True)
    raw = synth_weights(t, in_dim, out_dim, seed=t)
    want = oracle.matmul(t, raw, in_dim, out_dim, rows(n_tokens, in_dim, QUIET, 3), n_tokens).reshape(-1)
    xd = torch.from_numpy(rows(n_tokens, in_dim, SIGNALLING, 3)).cuda()
    w = be.upload_raw(raw, t, in_dim, out_dim)
    y = torch.empty(n_tokens * out_dim, device="cuda")
    torch.cuda.synchronize()
    be.set_tuning("gemv_prologue", prologue)
    try:
        be.matmul_dev(w, xd.data_ptr(), n_tokens, y.data_ptr(), False, 0)
        torch.cuda.synchronize()
    finally:
        be.set_tuning("gemv_prologue", 0)
        be.free_weight(w)
    assert np.isfinite(want).all()
    got = y.cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), np.nonzero(got.view(np.uint32) != want.view(np.uint32))[0][:8]
