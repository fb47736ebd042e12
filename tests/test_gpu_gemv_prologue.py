"""One-token launches that prepare their own activations (quantizer, or residual add + RMSNorm + quantizer, inside the
GEMV) against the same call after a launch that does: the arithmetic is the same sequence of roundings, so outputs, the
quantized row left in the scratch and a decode step's logits are equal to the bit."""
import numpy as np
import pytest
import torch

import oracle
from helpers import IQ4_NL, IQ4_XS, Q2_K, Q3_K, Q4_0, Q4_K, Q5_0, Q5_1, Q5_K, Q6_K, Q8_0, captured_launches, synth_weights
from test_gpu_llama import build

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module")
def be():
    from orangu_amd import Mi355xBackend
    b = Mi355xBackend()
    yield b
    b.close()


def special_row(n, seed):
    """Ties and near-ties of the int8 rounding, a run of zeros, one of subnormals, NaN and infinities."""
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(n).astype(f32)
    x[:32] = (np.arange(32) - 16).astype(f32) + f32(0.5)      # with 127 as the group's maximum: exact ties
    x[31] = 127.0
    x[5] = np.nextafter(f32(2.5), f32(0))
    if n >= 1024:
        x[256:512] = 0.0
        x[512:544] = f32(1e-42)
        x[768], x[780] = np.nan, 3.0
        x[800] = np.inf
    return x


# (edges: one block; a last run of 1024 partly empty; a row of 43 blocks; one run a wave, two runs a wave; rows that end
# inside a row block; several row blocks a workgroup with an odd number of them)
SHAPES_K = [(256, 5), (1024, 48), (1280, 33), (4096, 8192 + 272), (11008, 40), (14336, 17)]
SHAPES_32 = [(32, 3), (1056, 40), (4096, 300), (14336, 65)]


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q3_K, Q6_K, Q2_K, IQ4_XS, Q8_0, Q4_0, Q5_0, IQ4_NL, Q5_1])
def test_prepared_rows_give_the_same_bits(be, t):
    per_256 = t in (Q4_K, Q5_K, Q3_K, Q6_K, Q2_K, IQ4_XS)
    for in_dim, out_dim in SHAPES_K if per_256 else SHAPES_32:
        print(t, in_dim, out_dim, flush=True)
        raw = synth_weights(t, in_dim, out_dim, seed=in_dim)
        raw2 = synth_weights(t, in_dim, 19, seed=in_dim + 1)
        ws = [be.upload_raw(raw, t, in_dim, out_dim), be.upload_raw(raw2, t, in_dim, 19)]
        for x in (np.random.default_rng(1).standard_normal(in_dim).astype(f32), special_row(in_dim, 2)):
            xd = torch.from_numpy(x).cuda()
            got = {}
            for mode in (1, 2):
                be.set_tuning("gemv_prologue", mode)
                y = [torch.full((o,), 7.0, device="cuda") for o in (out_dim, 19, out_dim, 19)]
                torch.cuda.synchronize()
                ran = "ogm_gemv_fused_kernel<" if mode == 2 else "ogm_gemv_kernel<"
                be.matmul_dev(ws[0], xd.data_ptr(), 1, y[0].data_ptr(), False, 0)
                assert be.last_kernel().startswith(ran)
                be.matmul_multi_dev(ws, xd.data_ptr(), 1, [y[2].data_ptr(), y[1].data_ptr()], True, 0)
                assert be.last_kernel().startswith(ran)
                be.matmul_act_dev(ws[1], 1, y[3].data_ptr(), True, 0)   # over the scratch that call left
                torch.cuda.synchronize()
                got[mode] = [v.cpu().numpy() for v in y]
            for a, b in zip(got[1], got[2]):
                assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (t, in_dim, out_dim)
            if np.isfinite(x).all() and out_dim < 1000:
                want = oracle.matmul(t, raw, in_dim, out_dim, x, 1).reshape(-1)
                assert np.array_equal(got[2][0].view(np.uint32), want.view(np.uint32)), (t, in_dim, out_dim)
        for w in ws:
            be.free_weight(w)
    be.set_tuning("gemv_prologue", 0)


def test_output_over_its_input(be):
    """y may lie over x: such a call quantizes first, by one element at either end too; beside it, it prepares its own."""
    n = 1024
    raw = synth_weights(Q4_K, n, n, seed=3)
    w = be.upload_raw(raw, Q4_K, n, n)
    x = np.random.default_rng(4).standard_normal(n).astype(f32)
    want = oracle.matmul(Q4_K, raw, n, n, x, 1).reshape(-1)
    be.set_tuning("gemv_prologue", 2)
    for x_at, y_at in ((0, 0), (64, 0), (n - 1, 0), (n, 0), (0, n - 1), (0, n)):
        buf = torch.zeros(2 * n, device="cuda")
        buf[x_at:x_at + n] = torch.from_numpy(x).cuda()
        torch.cuda.synchronize()
        be.matmul_dev(w, buf.data_ptr() + 4 * x_at, 1, buf.data_ptr() + 4 * y_at, False, 0)
        torch.cuda.synchronize()
        assert be.last_kernel().startswith("ogm_gemv_fused_kernel<" if abs(x_at - y_at) == n else "ogm_gemv_kernel<")
        assert np.array_equal(buf[y_at:y_at + n].cpu().numpy().view(np.uint32), want.view(np.uint32))
    be.set_tuning("gemv_prologue", 0)
    be.free_weight(w)


# A layer's launches: F prepares its own row, P two types' too, S with SwiGLU besides; G the plain GEMV, A attention, N norm,
# s SwiGLU + quantize.
LETTER = {"ogm_gemv_kernel": "G", "ogm_gemv_fused_pair_kernel": "P", "ogm_attn_kernel": "A", "ogm_norm_quant_kernel": "N",
          "ogm_swiglu_quant_kernel": "s", "ogm_quantize_kernel": "q"}


def route(ran):
    """A decode step's launches as letters."""
    return "".join("S" if k[0] == "ogm_gemv_fused_kernel" and "Lb1EEv" in k[1] else
                   "F" if k[0] == "ogm_gemv_fused_kernel" else LETTER.get(k[0], "") for k in ran)


# (types: q/k/gate/up, v, down, output; a group of two types leaves its second launch the first one's scratch; Q5_0's
# 1056 inputs end inside a run of 256; 2304 / 6400: an odd number of blocks a row, whose row blocks of 64 leave SwiGLU out)
@pytest.mark.parametrize("types,n_embd,n_ff,layer", [((Q4_K, Q4_K, Q6_K, Q6_K), 2048, 8192, "FAGSF"),
                                                     ((Q4_K, Q6_K, Q4_K, Q6_K), 1024, 2816, "PAGSF"),
                                                     ((Q8_0, Q8_0, Q8_0, Q8_0), 1024, 3072, "FAGSF"),
                                                     ((Q5_0, Q8_0, Q5_1, Q8_0), 1056, 2080, "FGAGFsG"),
                                                     ((Q5_K, Q6_K, Q3_K, Q4_K), 4096, 4352, "PAGSF"),
                                                     ((Q6_K, Q6_K, IQ4_XS, Q4_K), 2304, 6400, "FAGFsG")])
def test_decode_steps_give_the_same_bits(be, types, n_embd, n_ff, layer):
    _, dev, rng = build(be, n_embd=n_embd, n_head=4, n_kv=2, hd=64, n_ff=n_ff, n_vocab=500, n_layer=3, types=types,
                        max_ctx=16, seed=n_embd)
    from orangu_amd import hiprt
    stream = hiprt.Stream()
    xs = rng.standard_normal((4, n_embd)).astype(f32)
    got = {}
    for mode in (1, 2):
        be.set_tuning("gemv_prologue", mode)
        out = []
        for pos in range(4):
            if pos % 2 == 0:
                out.append(dev.decode(xs[pos], pos)[0])
            else:
                xd, lg, tok = torch.from_numpy(xs[pos]).cuda(), torch.empty(500, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
                torch.cuda.synchronize()
                dev.decode_dev(xd.data_ptr(), pos, lg.data_ptr(), tok.data_ptr(), 0)
                torch.cuda.synchronize()
                out.append(lg.cpu().numpy())
                assert np.array_equal(xd.cpu().numpy(), xs[pos])   # the caller's row stays as it was
            out.append(dev.hidden())
        got[mode] = out
        launched = captured_launches(stream.ptr, lambda: dev.decode_dev(xd.data_ptr(), 3, lg.data_ptr(), tok.data_ptr(), stream.ptr))
        ran = route(launched)
        assert all(k[4] == 0 for k in launched if "fused" in k[0])
        v_apart = "G" if types[0] != types[1] else ""
        assert ran == 3 * (layer if mode == 2 else "NG" + v_apart + "AGNGsG") + "NG"
    be.set_tuning("gemv_prologue", 0)
    stream.destroy()
    dev.close()
    for a, b in zip(got[1], got[2]):
        assert np.isfinite(a).all()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# (each type's share of q/k + v within the line of 4096 row blocks x runs; q/k above it)
@pytest.mark.parametrize("n_head,n_kv,layer,wgs", [(32, 32, "PAGSF", 512 + 256), (64, 8, "PAGSF", 576 + 64), (128, 8, "NGGAGSF", 1024 + 64)])
def test_two_types_at_the_line(be, n_head, n_kv, layer, wgs):
    from orangu_amd import hiprt
    _, dev, rng = build(be, n_embd=4096, n_head=n_head, n_kv=n_kv, hd=128, n_ff=256, n_vocab=300, n_layer=1,
                        types=(Q4_K, Q6_K, Q4_K, Q6_K), max_ctx=8, seed=n_head)
    x = rng.standard_normal(4096).astype(f32)
    xd, lg, tok = torch.from_numpy(x).cuda(), torch.empty(300, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    stream = hiprt.Stream()
    step = lambda: dev.decode_dev(xd.data_ptr(), 0, lg.data_ptr(), tok.data_ptr(), stream.ptr)
    got = {}
    for mode in (1, 0):
        be.set_tuning("gemv_prologue", mode)
        step()
        stream.synchronize()
        got[mode] = lg.cpu().numpy(), dev.hidden()
        ran = captured_launches(stream.ptr, step)
        assert route(ran) == (layer if mode == 0 else "NGGAGNGsG") + "NG"
        if mode == 0:
            assert ran[0 if layer[0] == "P" else 1][2][0] == wgs
    be.set_tuning("gemv_prologue", 0)
    stream.destroy()
    dev.close()
    for a, b in zip(got[0], got[1]):
        assert np.isfinite(a).all()
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


# (the kernel between the projections and the attention takes several tokens a wave from 12288 waves of one on at heads of
# 64, from 20480 at 128; the norm two runs of 256 a wave from 1024 rows)
@pytest.mark.parametrize("n_embd,n_head,n_kv,hd,rope_dim,neox,pre,n_tokens", [
    (256, 32, 8, 64, 64, False, (), 257), (256, 4, 1, 64, 64, True, ("q_bias", "k_bias", "v_bias"), 263),
    (256, 2, 2, 128, 128, False, ("q_norm", "k_norm"), 259), (512, 4, 4, 64, 64, False, ("q_norm", "k_norm"), 1027),
    (1280, 32, 4, 128, 128, True, (), 1025), (256, 32, 8, 64, 24, False, ("q_norm", "k_norm"), 258),
    (256, 32, 8, 64, 48, True, ("q_bias", "k_bias", "v_bias"), 261), (512, 64, 8, 128, 96, True, (), 260),
    (512, 4, 2, 128, 2, False, (), 262)])
def test_batches_leave_the_rows_of_smaller_ones(be, n_embd, n_head, n_kv, hd, rope_dim, neox, pre, n_tokens):
    """Cache rows of a batch against those of the same tokens in parts of at most 100 (a wave a token).  The second
    layer's rows carry q through the first one's attention, by the kernel that works token by token whatever the batch."""
    _, dev, rng = build(be, n_embd=n_embd, n_head=n_head, n_kv=n_kv, hd=hd, n_ff=512, n_vocab=300, n_layer=2,
                        types=(Q8_0, Q8_0, Q8_0, Q8_0), max_ctx=n_tokens + 8, seed=n_tokens, neox=neox, pre=pre, rope_dim=rope_dim)
    X = rng.standard_normal((n_tokens, n_embd)).astype(f32)
    be.set_tuning("attn_prefill_variant", 1)
    be.set_tuning("attn_decode_chunks", 1)
    try:
        dev.prefill(X, 3)
        whole = [a.copy() for l in (0, 1) for a in dev.kv_read(l, 3, n_tokens)]
        for at in range(0, n_tokens, 100):
            dev.prefill(X[at:at + 100], 3 + at)
        parts = [a for l in (0, 1) for a in dev.kv_read(l, 3, n_tokens)]
    finally:
        be.set_tuning("attn_prefill_variant", 0)
        be.set_tuning("attn_decode_chunks", 0)
        dev.close()
    for a, b in zip(whole, parts):
        assert np.isfinite(np.asarray(a, np.float32)).all()
        assert np.array_equal(np.asarray(a), np.asarray(b))
