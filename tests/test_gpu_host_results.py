"""A model call's results on their way to pageable host memory: in chunks of 4096 words through two halves of pinned staging
of 2 MiB, each chunk announced by its own word.  At vocabularies around one chunk and with a remainder behind the last sixteen
bytes, at results of one piece, of exactly two, and of more pieces than there are halves, into plain and into pinned memory,
and with words that never come: always the bytes that one transfer of the runtime brings (host_flag_wait 0)."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import Q6_K
from test_gpu_llama import build, f32

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.set_tuning("host_flag_wait", 1)
    b.close()


def results(be, dev, x, n_vocab):
    """(everything a model hands back, as bytes): a decode step, a verify batch, a prompt and hidden states."""
    out = []
    for i in range(2):
        logits, tok = dev.decode(x[i], i)
        out += [logits.tobytes(), tok]
    logits, toks = dev.forward_all_logits(x, 2)
    out += [logits.tobytes(), np.asarray(toks).tobytes()]
    logits, tok = dev.prefill(x, 0)
    out += [logits.tobytes(), tok, dev.hidden_states(x).tobytes()]
    pinned = torch.zeros(n_vocab, pin_memory=True)
    tok = C.c_uint32()
    be._check(be._lib.ogm_llama_decode(be._ctx, dev._h, x[0].ctypes.data, len(x), pinned.data_ptr(), C.byref(tok)), "decode")
    return out + [pinned.numpy().tobytes(), tok.value]


@pytest.mark.parametrize("n_vocab,n_tokens", [
    (4095, 3), (4096, 2), (4097, 5), (4099, 64), (12291, 3),      # below, at and past a chunk; remainders of 1 to 3 words
    (16384, 32), (16384, 64), (20003, 64), (20003, 27)])          # half a staging, all of it, and three pieces
def test_results_arrive_whole(be, n_vocab, n_tokens):
    ref, dev, rng = build(be, n_embd=256, n_head=4, n_kv=2, hd=64, n_ff=512, n_vocab=n_vocab, n_layer=1,
                          types=(Q6_K, Q6_K, Q6_K, Q6_K), max_ctx=n_tokens + 8, seed=n_vocab)
    x = rng.standard_normal((n_tokens, 256)).astype(f32)
    try:
        be.set_tuning("host_flag_wait", 0)
        be.kernels_run()
        want = results(be, dev, x, n_vocab)
        assert "ogm_host_copy_kernel" not in be.kernels_run()
        for wait in (1, 1, 2):
            be.set_tuning("host_flag_wait", wait)
            be.kernels_run()
            got = results(be, dev, x, n_vocab)
            assert [g == w for g, w in zip(got, want)] == [True] * len(want), wait
            # the copies by kernel: of 2 MiB at most, from 16 KiB of pageable memory on (two steps, a batch, a prompt, the states)
            sizes = [n_vocab, n_vocab, n_vocab * n_tokens, n_vocab, 256 * n_tokens]
            assert be.kernels_run().count("ogm_host_copy_kernel") == sum(-(-n // 524288) for n in sizes if n >= 4096), wait
    finally:
        be.set_tuning("host_flag_wait", 1)
        dev.close()


def test_wide_hidden_states_take_their_pieces_in_turn(be):
    """600 rows of 2048: 4.9 MB, three pieces; and a run of different calls whose pieces reuse the same staging."""
    ref, dev, rng = build(be, n_embd=2048, n_head=8, n_kv=2, hd=64, n_ff=2048, n_vocab=4200, n_layer=1,
                          types=(Q6_K, Q6_K, Q6_K, Q6_K), max_ctx=640, seed=5)
    x = [rng.standard_normal((n, 2048)).astype(f32) for n in (600, 255, 256, 513)]
    try:
        be.set_tuning("host_flag_wait", 0)
        want = [dev.hidden_states(a).tobytes() for a in x]
        be.set_tuning("host_flag_wait", 1)
        for rep in range(70):      # past the call that synchronizes after 256 polled ones
            for a, w in zip(x, want):
                be.kernels_run()
                assert dev.hidden_states(a).tobytes() == w, (rep, len(a))
                assert be.kernels_run().count("ogm_host_copy_kernel") == -(-a.size // 524288)
    finally:
        be.set_tuning("host_flag_wait", 1)
        dev.close()
