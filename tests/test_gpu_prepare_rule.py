"""Which one-token launches prepare their own rows: the families of shapes that the limit on row blocks times runs of 1024
inputs alone gets wrong, each on both sides of its own line -- read from a capture of the call, over weights of zero bytes
(both routes give the same bits; test_gpu_gemv_prologue.py and test_gpu_llama.py compare them)."""
import numpy as np
import pytest
import torch

from helpers import BLOCK, IQ4_NL, IQ4_XS, Q2_K, Q3_K, Q4_0, Q4_K, Q5_0, Q5_1, Q5_K, Q6_K, Q8_0, captured_launches

pytestmark = pytest.mark.gpu
PREPARED, SEPARATE = ["ogm_gemv_fused_kernel"], ["ogm_quantize_kernel", "ogm_gemv_kernel"]


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


def zeros(be, t, in_dim, out_dim):
    bytes_, elems = BLOCK[t]
    return be.upload_raw(np.zeros(out_dim * (in_dim // elems) * bytes_, np.uint8), t, in_dim, out_dim)


def check(be, stream, t, in_dim, out_dim, prepared):
    w = zeros(be, t, in_dim, out_dim)
    x, y = torch.ones(in_dim, device="cuda"), torch.empty(out_dim, device="cuda")
    torch.cuda.synchronize()
    be.matmul_dev(w, x.data_ptr(), 1, y.data_ptr(), True, stream.ptr)   # (its scratch is there before the capture)
    stream.synchronize()
    ran = captured_launches(stream.ptr, lambda: be.matmul_dev(w, x.data_ptr(), 1, y.data_ptr(), True, stream.ptr))
    be.free_weight(w)
    print(t, in_dim, out_dim, [k[0] for k in ran], flush=True)
    assert [k[0] for k in ran] == (PREPARED if prepared else SEPARATE)


# (48 Mi weights of rows without padded tiles, 2048 row blocks of sixteen rows with)
@pytest.mark.parametrize("t,in_dim,out_dim,prepared", [
    (Q8_0, 1024, 49152, True), (Q8_0, 1024, 49153, False), (Q4_0, 512, 98304, True), (Q4_0, 512, 98305, False),
    (IQ4_NL, 768, 65536, True), (IQ4_NL, 768, 65537, False), (Q5_1, 864, 32768, True), (Q5_1, 864, 32769, False),
    (Q8_0, 1056, 32768, True), (Q5_0, 256, 131072, True)])
def test_one_run_of_per_32_blocks(be, stream, t, in_dim, out_dim, prepared):
    check(be, stream, t, in_dim, out_dim, prepared)


# (two runs a wave: 256 row blocks of sixteen rows)
@pytest.mark.parametrize("t", [Q4_K, Q6_K, IQ4_XS])
@pytest.mark.parametrize("in_dim,prepared_to", [(10240, 4096), (11008, 4096), (14336, 4096)])
def test_two_runs_a_wave(be, stream, t, in_dim, prepared_to):
    check(be, stream, t, in_dim, prepared_to, True)
    check(be, stream, t, in_dim, prepared_to + 1, False)


# (rows of three tiles, up to two row blocks in each of 512 workgroups; by type beyond)
@pytest.mark.parametrize("t,in_dim,out_dim,prepared", [
    (IQ4_XS, 3072, 16384, True), (IQ4_XS, 3072, 16385, False), (Q3_K, 2816, 16384, True), (Q3_K, 2816, 16385, False),
    (Q6_K, 3072, 16385, True), (Q4_K, 3072, 21840, True), (Q2_K, 3072, 16385, True), (IQ4_XS, 1536, 32768, True),
    (IQ4_XS, 1536, 40992, False), (Q6_K, 1536, 40992, False), (Q5_K, 1536, 40992, True), (Q4_K, 768, 131072, True),
    (Q4_K, 768, 163904, False)])
def test_three_tiles(be, stream, t, in_dim, out_dim, prepared):
    check(be, stream, t, in_dim, out_dim, prepared)


LETTER = {"ogm_norm_quant_kernel": "n", "ogm_gemv_kernel": "m", "ogm_attn_kernel": "a", "ogm_swiglu_quant_kernel": "s",
          "ogm_attn_combine_quant_kernel": "c", "ogm_quantize_kernel": "q", "ogm_gemv_fused_kernel": "F"}


def decode_launches(be, stream, t, n_embd, n_head, n_kv, hd, n_ff):
    """The launches of a decode step's one layer, every matrix of one type, as letters: norm, matmul, attention (and its merge),
    SwiGLU and quantizer launches small, matmuls that prepare their row F, gate and up that leave silu(gate) * up G."""
    from orangu_amd import LlamaDecoder
    shapes = {"wq": (n_embd, n_head * hd), "wk": (n_embd, n_kv * hd), "wv": (n_embd, n_kv * hd), "wo": (n_head * hd, n_embd),
              "w_gate": (n_embd, n_ff), "w_up": (n_embd, n_ff), "w_down": (n_ff, n_embd)}
    layer = {k: zeros(be, t, *s) for k, s in shapes.items()}
    ws = [*layer.values(), zeros(be, t, n_embd, 32)]
    layer["attn_norm"] = layer["ffn_norm"] = np.ones(n_embd, np.float32)
    dev = LlamaDecoder(be, n_embd=n_embd, n_head=n_head, n_head_kv=n_kv, head_dim=hd, n_ff=n_ff, n_vocab=32, layers=[layer],
                       output_norm=np.ones(n_embd, np.float32), output=ws[-1], max_ctx=8, rms_eps=1e-5,
                       rope_freq_base=10000.0, upload=lambda handle: handle)
    x, lg, tok = torch.ones(n_embd, device="cuda"), torch.empty(32, device="cuda"), torch.empty(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    ran = captured_launches(stream.ptr, lambda: dev.decode_dev(x.data_ptr(), 2, lg.data_ptr(), tok.data_ptr(), stream.ptr))
    dev.close()
    for w in ws:
        be.free_weight(w)
    assert [k[0] for k in ran[-2:]] == ["ogm_argmax_kernel"] * 2   # behind the last norm and the output matrix
    return "".join("G" if k[0] == "ogm_gemv_fused_kernel" and "Lb1EEv" in k[1] else LETTER[k[0]] for k in ran[:-4])


# (row blocks of sixteen rows times runs of 1024: up to 512 the launch prepares the normed row, beyond it the norm has a launch
# of its own; silu(gate) * up, of rows of at most 1024 inputs, beyond it too)
@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q5_0, Q5_1, IQ4_NL])
@pytest.mark.parametrize("n_embd,n_head,n_kv,hd,n_ff,want", [
    (2048, 32, 16, 64, 2048, "FamFsm"), (2048, 32, 32, 64, 2080, "nmamnmsm"), (4096, 32, 8, 128, 4096, "nmamnmsm"),
    (1024, 16, 8, 64, 8192, "FamGF")])
def test_norms_before_per_32_matrices(be, stream, t, n_embd, n_head, n_kv, hd, n_ff, want):
    got = decode_launches(be, stream, t, n_embd, n_head, n_kv, hd, n_ff)
    print(t, n_embd, n_ff, got, flush=True)
    assert got == want


@pytest.mark.parametrize("t,n_embd,n_head,n_kv,hd,n_ff,want", [
    (IQ4_XS, 3072, 24, 8, 128, 8192, "FacmGF"), (IQ4_XS, 3072, 24, 8, 128, 8704, "Facmnmsm"), (Q5_K, 3072, 24, 8, 128, 8704, "FacmGF"),
    (Q2_K, 1536, 24, 8, 64, 20480, "Facmnmsm"), (Q4_K, 1536, 24, 8, 64, 16384, "FacmGF")])
def test_three_tiles_gate_and_up(be, stream, t, n_embd, n_head, n_kv, hd, n_ff, want):
    got = decode_launches(be, stream, t, n_embd, n_head, n_kv, hd, n_ff)
    print(t, n_embd, n_ff, got, flush=True)
    assert got == want


# (512 workgroups run at once; the heavier types' second round from a quarter of it on)
@pytest.mark.parametrize("t", [Q4_K, Q2_K, Q3_K, Q5_K, Q6_K, IQ4_XS])
def test_gate_and_up_of_4096_inputs(be, stream, t):
    light = t in (Q4_K, Q2_K, Q3_K)
    for n_ff, prepared in ((8192, True), (8448, light), (9984, light), (10240, True), (14336, True), (16384, True), (16640, False)):
        got = decode_launches(be, stream, t, 4096, 32, 8, 128, n_ff)
        print(t, n_ff, got, flush=True)
        assert got.startswith("FamG") if prepared else got == "Famnmsm", n_ff
