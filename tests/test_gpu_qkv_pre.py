"""The kernel between a batch's projections and its attention (ogm_launch_qkv_pre: bias, per-head norm, RoPE, cache rows), in
its two forms: a wave a token and head, and a wave over several tokens where the launch is large.  Called as the prefill
calls it, on whole batches and on the same tokens in parts too small for the second form: the same bits in q and in both
caches; against numpy in 64 bits within the roundings; and the line between the forms."""
import ctypes as C

import numpy as np
import pytest
import torch

from helpers import captured_launches

pytestmark = pytest.mark.gpu
f32 = np.float32


class Pre(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("q_bias", "k_bias", "v_bias", "q_norm", "k_norm")] + [("eps", C.c_float), ("neox", C.c_uint32)]


@pytest.fixture(scope="module")
def launch():
    from orangu_amd import capi
    torch.cuda.init()
    fn = capi.load_library()._Z18ogm_launch_qkv_prePfPKfS1_PKvjRK10OgmAttnPrejjjPvS7_jjP12ihipStream_t
    vp, u = C.c_void_p, C.c_uint32
    fn.argtypes = [vp, vp, vp, vp, u, C.POINTER(Pre), u, u, u, vp, vp, u, u, vp]
    return fn


@pytest.fixture(scope="module")
def stream():
    from orangu_amd import hiprt
    s = hiprt.Stream()
    yield s
    s.destroy()


EPS = 1e-5


def run(launch, stream, x, cs, rope_dim, vecs, neox, n_head, n_kv, hd, pos0, parts):
    """q, K cache and V cache after launches over the given parts of the tokens; and the kernels of the first."""
    q, k, v = (torch.from_numpy(a).cuda() for a in x)
    n_tokens = q.shape[0]
    caches = [torch.full((pos0 + n_tokens + 1, n_kv * hd), 7.0, dtype=torch.float16, device="cuda") for _ in range(2)]
    cs_d = torch.from_numpy(cs).cuda()
    dev = {n: torch.from_numpy(a).cuda() for n, a in vecs.items()}
    pre = Pre(**{n: a.data_ptr() for n, a in dev.items()}, eps=EPS, neox=neox)
    torch.cuda.synchronize()

    def enqueue(at, n):
        assert launch(q[at:].data_ptr(), k[at:].data_ptr(), v[at:].data_ptr(), cs_d[at:].data_ptr() if rope_dim else cs_d.data_ptr(),
                      rope_dim, C.byref(pre), n_head, n_kv, hd, caches[0].data_ptr(), caches[1].data_ptr(), pos0 + at, n, stream.ptr) == 0

    ran = captured_launches(stream.ptr, lambda: enqueue(*parts[0]))
    for at, n in parts:
        enqueue(at, n)
    stream.synchronize()
    return [a.cpu().numpy() for a in (q, *caches)], [r[0] for r in ran]


def reference(x, cs, rope_dim, vecs, neox, n_head, n_kv, hd):
    out = []
    for name, a in zip("qkv", x):
        heads = n_head if name == "q" else n_kv
        a = a.astype(np.float64).reshape(len(a), heads, hd)
        if name + "_bias" in vecs:
            a = a + vecs[name + "_bias"].astype(np.float64).reshape(heads, hd)
        if name + "_norm" in vecs:
            a = a / np.sqrt((a * a).mean(-1, keepdims=True) + EPS) * vecs[name + "_norm"].astype(np.float64)
        half = rope_dim // 2
        if name != "v" and half:
            c, s = (cs[:, None, :, j].astype(np.float64) for j in (0, 1))
            i = np.arange(half) if neox else 2 * np.arange(half)
            j = i + half if neox else i + 1
            r = a.copy()
            r[..., i], r[..., j] = a[..., i] * c - a[..., j] * s, a[..., i] * s + a[..., j] * c
            a = r
        out.append(a.reshape(len(a), heads * hd))
    return out


# (tokens: one more than whole waves of four or eight; 12288 and 20480 waves of one token are the line at heads of 64 and 128)
@pytest.mark.parametrize("n_head,n_kv,hd,n_tokens", [(32, 8, 64, 257), (9, 3, 64, 821), (64, 8, 128, 257), (5, 5, 128, 1366)])
@pytest.mark.parametrize("neox", [0, 1])
@pytest.mark.parametrize("pre,rotated", [((), 1.0), (("q_bias", "k_bias", "v_bias"), 0.75), (("q_norm", "k_norm"), 0.375), (("k_bias", "q_norm"), 0.0)])
def test_both_forms(launch, stream, n_head, n_kv, hd, n_tokens, neox, pre, rotated):
    rng = np.random.default_rng(n_tokens + hd)
    pos0, rope_dim = 3, int(rotated * hd)
    x = [rng.standard_normal((n_tokens, h * hd)).astype(f32) for h in (n_head, n_kv, n_kv)]
    ang = rng.uniform(-3, 3, (n_tokens, max(1, rope_dim // 2)))
    cs = np.stack([np.cos(ang), np.sin(ang)], -1).astype(f32)
    sizes = {"q_bias": n_head * hd, "k_bias": n_kv * hd, "v_bias": n_kv * hd, "q_norm": hd, "k_norm": hd}
    vecs = {n: (rng.standard_normal(sizes[n]) + n.endswith("norm")).astype(f32) for n in pre}
    args = (x, cs, rope_dim, vecs, neox, n_head, n_kv, hd)
    whole, ran = run(launch, stream, *args, pos0, [(0, n_tokens)])
    assert ran == ["ogm_qkv_pre_tokens_kernel"]
    parts, ran = run(launch, stream, *args, pos0, [(at, min(100, n_tokens - at)) for at in range(0, n_tokens, 100)])
    assert ran == ["ogm_qkv_pre_kernel"]
    for a, b in zip(whole, parts):
        assert np.array_equal(a.view(np.uint16), b.view(np.uint16))
    want = reference(*args)
    # f32: a norm's sum of 128 squares and its root, then five roundings of values of up to the row's largest
    err = np.abs(whole[0] - want[0]).max() / np.abs(want[0]).max()
    assert err < 2e-6, err
    for got, w in zip(whole[1:], want[1:]):
        assert (got[:pos0] == 7.0).all() and (got[pos0 + n_tokens:] == 7.0).all()
        rows = got[pos0:pos0 + n_tokens].astype(np.float64)
        # half a step of f16 (2^-11 of the value) on top
        assert (np.abs(rows - w) <= 2.0 ** -11 * np.abs(w) + 2e-6 * np.abs(w).max() + 2.0 ** -25).all()


@pytest.mark.parametrize("n_head,n_kv,hd,n_tokens,many", [(32, 8, 64, 255, False), (32, 8, 64, 256, True), (4, 2, 64, 1535, False),
                                                          (4, 2, 64, 1536, True), (64, 8, 128, 255, False), (64, 8, 128, 256, True),
                                                          (16, 2, 128, 512, False), (2, 1, 128, 2048, False)])
def test_the_line(launch, stream, n_head, n_kv, hd, n_tokens, many):
    x = [np.zeros((n_tokens, h * hd), f32) for h in (n_head, n_kv, n_kv)]
    cs = np.zeros((n_tokens, hd // 2, 2), f32)
    _, ran = run(launch, stream, x, cs, hd, {}, 0, n_head, n_kv, hd, 0, [(0, n_tokens)])
    assert ran == ["ogm_qkv_pre_tokens_kernel" if many else "ogm_qkv_pre_kernel"]
