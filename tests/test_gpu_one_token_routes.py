"""Which kernels one-token calls run: read from a capture of the call (helpers.captured_launches), so that a comparison of
two routes elsewhere is known to compare two routes."""
import numpy as np
import pytest
import torch

from helpers import BLOCK, IQ4_NL, IQ4_XS, Q2_K, Q3_K, Q4_0, Q4_K, Q5_0, Q5_1, Q5_K, Q6_K, Q8_0, captured_launches, synth_weights

pytestmark = pytest.mark.gpu
FMT = {Q4_K: "FmtQ4K", Q5_K: "FmtQ5K", Q3_K: "FmtQ3K", Q6_K: "FmtQ6K", Q2_K: "FmtQ2K", IQ4_XS: "FmtIQ4XS", Q8_0: "FmtQ80",
       Q4_0: "FmtQ40", Q5_0: "FmtQ50", IQ4_NL: "FmtIQ4NL", Q5_1: "FmtQ51"}
# the template argument of the types whose Fmt name is an alias
MANGLED = {Q4_0: "8FmtNib32ILi0E", Q5_0: "8FmtNib32ILi1E", IQ4_NL: "8FmtNib32ILi2E", Q5_1: "8FmtNib32ILi3E", Q2_K: "7FmtQ2KTILb0E"}


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


def launches(stream, call):
    """The call's launches; it runs once before, so that its scratch is there."""
    call()
    stream.synchronize()
    return captured_launches(stream.ptr, call)


@pytest.mark.parametrize("t", sorted(FMT))
@pytest.mark.parametrize("prologue", [1, 2])
def test_last_kernel_names_the_kernel_that_ran(be, stream, t, prologue):
    in_dim, out_dim = 1024, 40
    w = be.upload_raw(synth_weights(t, in_dim, out_dim, seed=t), t, in_dim, out_dim)
    x, y = torch.ones(in_dim, device="cuda"), torch.empty(out_dim, device="cuda")
    torch.cuda.synchronize()
    be.set_tuning("gemv_prologue", prologue)
    try:
        ran = launches(stream, lambda: be.matmul_dev(w, x.data_ptr(), 1, y.data_ptr(), False, stream.ptr))
    finally:
        be.set_tuning("gemv_prologue", 0)
    name = be.last_kernel()
    be.free_weight(w)
    print(t, prologue, name, ran, flush=True)
    assert [k[0] for k in ran] == (["ogm_quantize_kernel", "ogm_gemv_kernel"] if prologue == 1 else ["ogm_gemv_fused_kernel"])
    assert name.split("<")[0] == ran[-1][0]
    assert name.split("<")[1].rstrip(">").split(",")[0] == FMT[t]
    assert ran[-1][1].startswith("I" + MANGLED.get(t, str(len(FMT[t])) + FMT[t]))


def test_a_row_behind_the_bus_is_read_once(be, stream):
    """A caller's pinned row goes through a quantizer launch, alone and for several matrices; one in device memory (also
    from the middle of an allocation) is prepared by the launch.  Same bits."""
    in_dim, out_dim = 4096, 600
    ws = [be.upload_raw(synth_weights(Q4_K, in_dim, o, seed=o), Q4_K, in_dim, o) for o in (out_dim, 40)]
    x = torch.randn(8 + in_dim)
    on_device, pinned = x.cuda(), x.pin_memory()
    got = []
    for rows in (on_device, pinned):
        y = [torch.zeros(o, device="cuda") for o in (out_dim, out_dim, 40)]
        torch.cuda.synchronize()
        ran = launches(stream, lambda: (be.matmul_dev(ws[0], rows.data_ptr() + 32, 1, y[0].data_ptr(), False, stream.ptr),
                                        be.matmul_multi_dev(ws, rows.data_ptr() + 32, 1, [y[1].data_ptr(), y[2].data_ptr()],
                                                            True, stream.ptr)))
        stream.synchronize()
        assert [k[0] for k in ran] == 2 * (["ogm_gemv_fused_kernel"] if rows is on_device else
                                           ["ogm_quantize_kernel", "ogm_gemv_kernel"])
        got.append([v.cpu().numpy().view(np.uint32) for v in y])
    for w in ws:
        be.free_weight(w)
    for a, b in zip(*got):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("t", sorted(FMT))
def test_prepared_rows_use_no_private_memory(be, stream, t):
    """Alone and several matrices at a time, at row lengths that are constants of the kernel and at others, a wave
    preparing one run of 1024 or two.  (An array indexed by a lane's own number ends there: every wave stored it at its
    start, and at the line calls took up to an eighth longer than after a quantizer launch.)"""
    be.set_tuning("gemv_prologue", 2)
    try:
        for in_dim in (1024, 4096, 8960, 14336):
            ws = [be.upload_raw(synth_weights(t, in_dim, o, seed=o), t, in_dim, o) for o in (33, 20)]
            x, y = torch.ones(in_dim, device="cuda"), [torch.empty(33, device="cuda") for _ in ws]
            torch.cuda.synchronize()
            ran = launches(stream, lambda: (be.matmul_dev(ws[0], x.data_ptr(), 1, y[0].data_ptr(), False, stream.ptr),
                                            be.matmul_multi_dev(ws, x.data_ptr(), 1, [v.data_ptr() for v in y], True, stream.ptr)))
            for w in ws:
                be.free_weight(w)
            assert [(k[0], k[4]) for k in ran] == 2 * [("ogm_gemv_fused_kernel", 0)], (in_dim, ran)
    finally:
        be.set_tuning("gemv_prologue", 0)


# (row blocks x runs of 1024 up to 4096, 8192 at 4096 inputs and for the per-32 types; row blocks of 16 rows, of 64 at 7 blocks a
# row; the shapes that end earlier are in test_gpu_prepare_rule.py)
@pytest.mark.parametrize("t,in_dim,out_dim,prepared", [
    (Q4_K, 4096, 512 * 16, True), (Q4_K, 4096, 512 * 16 + 1, True), (Q4_K, 4096, 2048 * 16, True), (Q4_K, 4096, 2048 * 16 + 1, False),
    (Q6_K, 2816, 682 * 16, True), (Q6_K, 2816, 682 * 16 + 1, True), (Q6_K, 2816, 1365 * 16, True), (Q6_K, 2816, 1365 * 16 + 1, False),
    (Q4_K, 1792, 1024 * 64, True), (Q4_K, 1792, 2048 * 64, True), (Q4_K, 1792, 2048 * 64 + 1, False),
    (Q8_0, 2048, 256 * 16, True), (Q8_0, 2048, 256 * 16 + 1, True), (Q8_0, 2048, 4096 * 16, True), (Q8_0, 2048, 4096 * 16 + 1, False)])
def test_the_line(be, stream, t, in_dim, out_dim, prepared):
    bytes_, elems = BLOCK[t]
    raw = np.zeros(out_dim * (in_dim // elems) * bytes_, np.uint8)
    w = be.upload_raw(raw, t, in_dim, out_dim)
    x, y = torch.ones(in_dim, device="cuda"), torch.empty(out_dim, device="cuda")
    torch.cuda.synchronize()
    ran = launches(stream, lambda: be.matmul_dev(w, x.data_ptr(), 1, y.data_ptr(), False, stream.ptr))
    be.free_weight(w)
    assert [k[0] for k in ran] == (["ogm_gemv_fused_kernel"] if prepared else ["ogm_quantize_kernel", "ogm_gemv_kernel"])
