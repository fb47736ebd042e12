"""The performance cases of the quantized matmul path and of the Llama forward pass around it.

Every case goes through the package's public entry points as a program that serves a model calls them:

* ``linear``   device-resident activations through uploaded matrices (``Mi355xBackend.matmul_dev`` for one matrix,
               ``matmul_multi_dev`` for several that read the same input), in matmul's or matmul_decode's float order;
* ``ffn``      one token through a feed-forward block's three matrices: gate and up together, then down;
* ``host``     ``Backend::matmul`` itself: a host slice in, a host slice out;
* ``decode``   one token through a model with a filled cache, device pointers (``decode_dev``) or host ones (``decode``);
* ``verify``   a speculative-decode verify batch: every position's logits and greedy token (``forward_all_logits``);
* ``prefill``  a prompt from an empty cache, the last position's logits (``prefill_tokens``);
* ``embed``    an embeddings request: every token's final hidden state (``hidden_states``).

The models are the 8B-shaped Llama of the benchmark (hidden 4096, 32 heads over 8 K/V heads, FFN 14336, vocabulary
128256; 8 of its layers, so that a state is made quickly) and a 1B-shaped one (hidden 2048, 32 heads of 64 over 8,
FFN 8192; all 16 layers).  Weights are random blocks whose values have the spread of a trained matrix.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from orangu_amd import LlamaDecoder, Mi355xBackend, QuantMatrix

Q4_0, Q5_0, Q5_1, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K, IQ4_NL, IQ4_XS = 2, 6, 7, 8, 10, 11, 12, 13, 14, 20, 23
TYPES = {"q4_0": Q4_0, "q5_0": Q5_0, "q5_1": Q5_1, "q8_0": Q8_0, "q2_k": Q2_K, "q3_k": Q3_K, "q4_k": Q4_K, "q5_k": Q5_K,
         "q6_k": Q6_K, "iq4_nl": IQ4_NL, "iq4_xs": IQ4_XS}
BLOCK = {Q4_0: (18, 32), Q5_0: (22, 32), Q5_1: (24, 32), Q8_0: (34, 32), Q2_K: (84, 256), Q3_K: (110, 256),
         Q4_K: (144, 256), Q5_K: (176, 256), Q6_K: (210, 256), IQ4_NL: (18, 32), IQ4_XS: (136, 256)}
# the f16 scale fields of a block: (offset of the scale, its typical value, offset of the minimum's, its multiple of
# the scale); the typical values give weights with a standard deviation of about 0.03
SCALES = {Q4_0: (0, 6.5e-3, None, 0.0), Q5_0: (0, 3.2e-3, None, 0.0), Q5_1: (0, 3.2e-3, 2, -15.5), Q8_0: (0, 4.0e-4, None, 0.0),
          IQ4_NL: (0, 4.5e-4, None, 0.0), Q2_K: (80, 2.4e-3, 82, 1.5), Q3_K: (108, 7.0e-4, None, 0.0), Q4_K: (0, 1.5e-4, 2, 7.5),
          Q5_K: (0, 7.0e-5, 2, 15.5), Q6_K: (208, 2.2e-5, None, 0.0), IQ4_XS: (0, 2.4e-5, None, 0.0)}

MODELS = {  # layers run, hidden, heads, K/V heads, head width, FFN, vocabulary
    "8b": (8, 4096, 32, 8, 128, 14336, 128256),
    "1b": (16, 2048, 32, 8, 64, 8192, 128256),
}
RESIDUAL = 1 / 32   # of the matrices that write the residual stream: a block's update is then about a sixth of it
EMBEDDINGS = 8192
MAX_LINEAR_FLOPS = 3.0e11   # of a drawn matmul: the slowest types then take no longer than the largest listed case


def listed():
    return [
        # the smallest call a layer makes: a K or V projection at one token
        {"name": "linear_q4k_4096x1024_t1", "kind": "linear", "type": "q4_k", "in": 4096, "outs": "1024", "tokens": 1, "decode": True},
        # the headline: an 8B feed-forward block at one token
        {"name": "ffn_q4k_4096x14336_t1", "kind": "ffn", "type": "q4_k", "in": 4096, "ff": 14336, "tokens": 1},
        # the backend seam itself, one token, host slices
        {"name": "host_q8_0_4096x4096_t1", "kind": "host", "type": "q8_0", "in": 4096, "outs": "4096", "tokens": 1, "decode": True},
        # the vocabulary projection of a small decode batch
        {"name": "linear_q6k_4096x128256_t4", "kind": "linear", "type": "q6_k", "in": 4096, "outs": "128256", "tokens": 4, "decode": True},
        # a short prompt through a Q5_K matrix of an awkward width (43 blocks a row)
        {"name": "linear_q5k_11008x4096_t77", "kind": "linear", "type": "q5_k", "in": 11008, "outs": "4096", "tokens": 77, "decode": False},
        # a prompt through a per-32 type's gate and up projections
        {"name": "linear_q8_0_4096x14336_t512", "kind": "linear", "type": "q8_0", "in": 4096, "outs": "14336,14336", "tokens": 512, "decode": False},
        # token generation: the usual chat context, a long one, and a small model driven from the host
        {"name": "decode_8b_ctx2048", "kind": "decode", "model": "8b", "ctx": 2048, "host": False},
        {"name": "decode_8b_ctx16000", "kind": "decode", "model": "8b", "ctx": 16000, "host": False},
        {"name": "decode_1b_ctx333_host", "kind": "decode", "model": "1b", "ctx": 333, "host": True},
        # speculative decoding: the last accepted token and a draft of four
        {"name": "verify_8b_t5_ctx2048", "kind": "verify", "model": "8b", "ctx": 2048, "tokens": 5},
        # a prompt of a usual length, and an embeddings request over a longer text
        {"name": "prefill_8b_t512", "kind": "prefill", "model": "8b", "tokens": 512},
        {"name": "embed_1b_t1901", "kind": "embed", "model": "1b", "tokens": 1901},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear"] * 6 + ["ffn", "host"] + ["decode"] * 4 + ["verify"] * 2 + ["prefill"] * 2 + ["embed"])
    if kind in ("linear", "host"):
        name = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0", "q5_k"] + sorted(TYPES))
        be = BLOCK[TYPES[name]][1]
        width = be * max(1, round(_log_int(rng, 512, 14336) / be))
        tokens = rng.choice([1, _log_int(rng, 2, 16), _log_int(rng, 17, 2048)]) if kind == "linear" else rng.choice([1, _log_int(rng, 2, 64)])
        rows = [_log_int(rng, 256, 16384) for _ in range(rng.choice([1, 1, 2, 3]) if kind == "linear" else 1)]
        tokens = max(1, min(tokens, int(MAX_LINEAR_FLOPS / (2 * width * sum(rows)))))
        return {"kind": kind, "type": name, "in": width, "outs": ",".join(map(str, rows)), "tokens": tokens,
                "decode": bool(tokens == 1 or (tokens <= 16 and rng.random() < 0.3))}
    if kind == "ffn":
        name = rng.choice(["q4_k", "q5_k", "q6_k", "q8_0", "iq4_xs"])
        return {"kind": kind, "type": name, "in": 256 * rng.randint(4, 24), "ff": 256 * rng.randint(12, 56), "tokens": rng.choice([1, 1, 2, 4])}
    model = rng.choice(sorted(MODELS))
    if kind == "decode":
        return {"kind": kind, "model": model, "ctx": _log_int(rng, 1, 16000), "host": rng.random() < 0.5}
    if kind == "verify":
        return {"kind": kind, "model": model, "ctx": _log_int(rng, 16, 4096), "tokens": rng.randint(2, 16)}
    if kind == "prefill":
        return {"kind": kind, "model": model, "tokens": _log_int(rng, 17, 512 if model == "8b" else 1850)}
    return {"kind": kind, "model": model, "tokens": _log_int(rng, 17, 512 if model == "8b" else 1901)}


# ---- states ------------------------------------------------------------------------------------------------------

_shared = {}


def _backend():
    """The process's backend and the stream its device-pointer calls go to."""
    if not _shared:
        torch.cuda.init()
        _shared["be"] = Mi355xBackend()
        _shared["stream"] = torch.cuda.Stream()
    return _shared["be"], _shared["stream"]


class State:
    """What one case keeps between passes; gives its device copies back when it goes."""

    def __init__(self, be):
        self.be, self.weights, self.matrices, self.decoder = be, [], [], None

    def __del__(self):
        torch.cuda.synchronize()
        if self.decoder is not None:
            self.decoder.close()
        for w in self.weights:
            self.be.free_weight(w)
        for m in self.matrices:
            self.be.evict(m)


def _raw(gen, type_id, width, rows, scale=1.0):
    """Blocks of a random matrix: uniform payload bytes, scales around the type's typical value."""
    bytes_, elems = BLOCK[type_id]
    n = rows * (width // elems)
    # (a whole number of 64-bit words for the generator)
    words = torch.randint(-2**63, 2**63 - 1, ((n * bytes_ + 7) // 8,), generator=gen, device="cuda", dtype=torch.int64)
    raw = words.view(torch.uint8)[:n * bytes_].view(n, bytes_)
    at, value, at_min, times = SCALES[type_id]
    d = scale * value * (0.5 + torch.rand(n, generator=gen, device="cuda"))
    raw[:, at:at + 2] = d.half().view(torch.uint8).view(n, 2)
    if at_min is not None:
        raw[:, at_min:at_min + 2] = (times * d).half().view(torch.uint8).view(n, 2)
    return raw.view(-1).cpu().numpy()


def _upload(s, gen, type_id, width, rows, scale=1.0):
    s.weights.append(s.be.upload_raw(_raw(gen, type_id, width, rows, scale), type_id, width, rows))
    return s.weights[-1]


def _model(s, gen, case):
    n_layer, n_embd, n_head, n_kv, hd, n_ff, n_vocab = MODELS[case["model"]]
    kvd = n_kv * hd
    rng = np.random.default_rng(int(torch.randint(0, 2**31, (1,), generator=gen, device="cuda")))
    layers = []
    for i in range(n_layer):
        # the 8B-shaped model: everything Q4_K but down (and the output) Q6_K; the 1B-shaped one as Q4_K_M files mix
        # them, V and down in Q6_K in every other layer
        more = Q6_K if case["model"] == "8b" or i % 2 == 0 else Q4_K
        v_type = Q4_K if case["model"] == "8b" else more
        shapes = {"wq": (Q4_K, n_embd, n_head * hd), "wk": (Q4_K, n_embd, kvd), "wv": (v_type, n_embd, kvd),
                  "wo": (Q4_K, n_head * hd, n_embd), "w_gate": (Q4_K, n_embd, n_ff), "w_up": (Q4_K, n_embd, n_ff),
                  "w_down": (more, n_ff, n_embd)}
        layer = {k: _upload(s, gen, *v, scale=RESIDUAL if k in ("wo", "w_down") else 1.0) for k, v in shapes.items()}
        layer["attn_norm"] = (1 + 0.05 * rng.standard_normal(n_embd)).astype(np.float32)
        layer["ffn_norm"] = (1 + 0.05 * rng.standard_normal(n_embd)).astype(np.float32)
        layers.append(layer)
    s.output = _upload(s, gen, Q6_K, n_embd, n_vocab)
    if case["kind"] in ("prefill", "embed"):
        # (embedding rows of the residual stream's own size, for the part of the vocabulary that the prompts use)
        s.embedding = _upload(s, gen, Q4_K, n_embd, EMBEDDINGS, scale=1 / 0.03)
    ctx = case.get("ctx", 0)
    s.decoder = LlamaDecoder(s.be, n_embd=n_embd, n_head=n_head, n_head_kv=n_kv, head_dim=hd, n_ff=n_ff, n_vocab=n_vocab,
                             layers=layers, output_norm=np.ones(n_embd, np.float32), output=s.output,
                             max_ctx=ctx + max(64, case.get("tokens", 1)), rms_eps=1e-5, rope_freq_base=500000.0,
                             upload=lambda handle: handle)
    if ctx:
        # the cache of a conversation: every layer its own rows, cut from one pool
        pool = rng.standard_normal((2 * ctx + 64 * n_layer) * kvd, dtype=np.float32)
        for i in range(n_layer):
            rows = pool[64 * i * kvd:(64 * i + 2 * ctx) * kvd].reshape(2, ctx, kvd)
            s.decoder.kv_write(i, 0, rows[0], rows[1])
    return rng, n_embd, n_vocab


def prepare(case, seed):
    be, stream = _backend()
    gen = torch.Generator("cuda")
    gen.manual_seed(seed * 7919 + 13)
    s = State(be)
    s.case, s.stream = case, stream.cuda_stream
    kind, tokens = case["kind"], case.get("tokens", 1)
    if kind == "linear":
        outs = [int(o) for o in case["outs"].split(",")]
        s.w = [_upload(s, gen, TYPES[case["type"]], case["in"], o) for o in outs]
        s.x = torch.randn(tokens, case["in"], generator=gen, device="cuda")
        s.y = [torch.empty(tokens, o, device="cuda") for o in outs]
    elif kind == "ffn":
        t, n, ff = TYPES[case["type"]], case["in"], case["ff"]
        s.w = [_upload(s, gen, t, n, ff), _upload(s, gen, t, n, ff), _upload(s, gen, t, ff, n)]
        s.x = torch.randn(tokens, n, generator=gen, device="cuda")
        s.h = torch.randn(tokens, ff, generator=gen, device="cuda")
        s.y = [torch.empty(tokens, o, device="cuda") for o in (ff, ff, n)]
    elif kind == "host":
        t, out = TYPES[case["type"]], int(case["outs"])
        s.matrices.append(QuantMatrix(_raw(gen, t, case["in"], out), t, case["in"], out))
        be.upload(s.matrices[0])
        s.x = torch.randn(tokens * case["in"], generator=gen, device="cuda").cpu().numpy()
    else:
        rng, n_embd, n_vocab = _model(s, gen, case)
        if kind in ("prefill", "embed"):
            s.x = rng.integers(0, EMBEDDINGS, tokens).astype(np.uint32)
        else:
            s.x = rng.standard_normal((tokens, n_embd), dtype=np.float32)
        if kind == "decode" and not case["host"]:
            s.x = torch.from_numpy(s.x).cuda()
            s.logits = torch.empty(n_vocab, device="cuda")
            s.greedy = torch.empty(1, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


def run(s):
    # (a model's greedy tokens are made but not compared: over random weights the two largest of 128256 logits are
    # often closer than a tipped rounding, see tolerance; the logits that they are picked from are the output)
    case, be, kind = s.case, s.be, s.case["kind"]
    tokens = case.get("tokens", 1)
    if kind == "linear":
        if len(s.w) == 1:
            be.matmul_dev(s.w[0], s.x.data_ptr(), tokens, s.y[0].data_ptr(), case["decode"], s.stream)
        else:
            be.matmul_multi_dev(s.w, s.x.data_ptr(), tokens, [y.data_ptr() for y in s.y], case["decode"], s.stream)
        return s.y
    if kind == "ffn":
        be.matmul_multi_dev(s.w[:2], s.x.data_ptr(), tokens, [s.y[0].data_ptr(), s.y[1].data_ptr()], True, s.stream)
        be.matmul_dev(s.w[2], s.h.data_ptr(), tokens, s.y[2].data_ptr(), True, s.stream)
        return s.y
    if kind == "host":
        return (be.matmul_decode if case["decode"] else be.matmul)(s.x, tokens, s.matrices[0])
    if kind == "decode":
        if case["host"]:
            return s.decoder.decode(s.x, case["ctx"])[0]
        s.decoder.decode_dev(s.x.data_ptr(), case["ctx"], s.logits.data_ptr(), s.greedy.data_ptr(), s.stream)
        return s.logits
    if kind == "verify":
        return s.decoder.forward_all_logits(s.x, case["ctx"])[0]
    if kind == "prefill":
        return s.decoder.prefill_tokens(s.embedding, s.x, 0)[0]
    return s.decoder.hidden_states(tok_embd=s.embedding, tokens=s.x)


# ---- what a pass cannot do without -------------------------------------------------------------------------------

def _matrix_bytes(type_id, width, rows):
    bytes_, elems = BLOCK[type_id]
    return rows * (width // elems) * bytes_


def work(case):
    kind, tokens = case["kind"], case.get("tokens", 1)
    if kind in ("linear", "host"):
        rows = sum(int(o) for o in case["outs"].split(","))
        return {"bytes": _matrix_bytes(TYPES[case["type"]], case["in"], rows) + 4 * tokens * (case["in"] + rows),
                "flops": 2 * tokens * case["in"] * rows}
    if kind == "ffn":
        t, n, ff = TYPES[case["type"]], case["in"], case["ff"]
        return {"bytes": 2 * _matrix_bytes(t, n, ff) + _matrix_bytes(t, ff, n) + 4 * tokens * (2 * n + 3 * ff),
                "flops": 6 * tokens * n * ff}
    n_layer, n_embd, n_head, n_kv, hd, n_ff, n_vocab = MODELS[case["model"]]
    qd, kvd, ctx = n_head * hd, n_kv * hd, case.get("ctx", 0)
    weights = flops = 0
    for i in range(n_layer):
        more = Q6_K if case["model"] == "8b" or i % 2 == 0 else Q4_K
        v_type = Q4_K if case["model"] == "8b" else more
        weights += _matrix_bytes(Q4_K, n_embd, qd + kvd) + _matrix_bytes(v_type, n_embd, kvd) + _matrix_bytes(Q4_K, qd, n_embd)
        weights += _matrix_bytes(Q4_K, n_embd, 2 * n_ff) + _matrix_bytes(more, n_ff, n_embd)
        flops += 2 * tokens * (n_embd * (qd + 2 * kvd) + qd * n_embd + 3 * n_embd * n_ff)
        flops += 4 * qd * (tokens * ctx + tokens * (tokens + 1) // 2)          # scores and weighted sum
    cache = 2 * n_layer * kvd * 2 * (ctx + tokens)                             # f16 rows read, the new ones written
    rows = tokens if kind == "verify" else 0 if kind == "embed" else 1         # rows through the output matrix
    if rows:
        weights += _matrix_bytes(Q6_K, n_embd, n_vocab)
        flops += 2 * rows * n_embd * n_vocab
    if kind in ("prefill", "embed"):
        weights += _matrix_bytes(Q4_K, n_embd, tokens)                         # the tokens' embedding rows
        io = 4 * tokens
    else:
        io = 4 * tokens * n_embd
    io += 4 * rows * n_vocab if rows else 4 * tokens * n_embd
    return {"bytes": weights + cache + io, "flops": flops}


def tolerance(case):
    # A matmul quantizes its input to int8 exactly and sums f32 terms; another order of the sums shows 2e-7 to 4e-7.
    if case["kind"] in ("linear", "ffn", "host"):
        return {"rel": 1.5e-6}
    # Through a model a last-bit difference tips an int8 rounding now and then, which is 1/254 of the largest of 256
    # values, and the tip travels on and tips others until the two results are as far apart as the quantized path is
    # from an exact one: the library's own attention kernels and its two float orders of a GEMM are 1 % to 2 % apart.
    return {"rel": 3e-2}
