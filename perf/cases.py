"""The work this library is timed on: what a program that serves one chat on one GPU has it do.

A case is a plain dict; `listed()` gives the named ones and `draw()` more of the same ranges. The
kinds, from the smallest call to the largest:

decode_attention  one layer's rope, cache append and attention of one token, over short and long
                  caches (muyo_rope_append_f16kv, muyo_attention_decode_f16kv)
head              the reference's node chain that ends every token: final norm, LM-head GEMV and
                  greedy argmax, as separate launchers
sample            the sampler on one token's logits (muyo_sample_f32)
decode            one whole decode step (Decoder.step), as a chat that streams its answer runs it
mlp               a prefill's feed-forward block: norm, gate/up GEMM with swiglu, down GEMM + residual
attention_block   a prefill's attention block: rope and append, causal attention over the cache,
                  o_proj GEMM + residual
prefill           a whole prompt or chat turn (Decoder.prefill)
rows              the element-wise and reduction launchers on a batch of rows

Widths are the two configurations the binding names (QWEN25_05B, QWEN25_7B). The whole-model kinds
run the 0.5B one at its full depth; the 7B one at a few of its layers, which repeat.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "muyo-llm_amd"))
import muyo_hip as mh  # noqa: E402

MODELS = {"0.5b": mh.QWEN25_05B, "7b": mh.QWEN25_7B}
EPS, ROPE_BASE = 1e-6, 1e6


def listed():
    return [
        # The first tokens of an answer: a short cache, one layer at a time. Launches and latency.
        dict(name="decode_attention_short", kind="decode_attention", model="0.5b", position=301, max_seq=2048),
        # The same call late in a long document.
        dict(name="decode_attention_long", kind="decode_attention", model="7b", position=20011, max_seq=32768),
        # A program that drives the reference's nodes itself: the end of a token.
        dict(name="head_nodes", kind="head", model="0.5b"),
        # The usual chat settings of the sampler, with a repetition penalty.
        dict(name="sample_chat", kind="sample", vocab=151936, temperature=0.7, top_k=40, top_p=0.95,
             repeat_penalty=1.1, repeat_last_n=64, history=777),
        # One streamed token in the middle of a 2048-token context.
        dict(name="decode_05b", kind="decode", model="0.5b", layers=24, position=1023, max_seq=2048),
        # The same at the wide configuration, near the end of the context.
        dict(name="decode_7b", kind="decode", model="7b", layers=3, position=1999, max_seq=2048),
        # A short user turn after a longer conversation: few rows, every weight read.
        dict(name="prefill_7b_turn", kind="prefill", model="7b", layers=4, count=45, position=700, max_seq=2048),
        # An ordinary prompt, odd in length.
        dict(name="prefill_05b_prompt", kind="prefill", model="0.5b", layers=24, count=613, position=0, max_seq=2048),
        # A prompt that fills the context.
        dict(name="prefill_7b_full", kind="prefill", model="7b", layers=4, count=2048, position=0, max_seq=2048),
        # One layer's feed-forward block of an ordinary prompt.
        dict(name="mlp_05b", kind="mlp", model="0.5b", rows=301),
        # One layer's attention block of a later part of a long document.
        dict(name="attention_block_7b", kind="attention_block", model="7b", rows=777, position=5003, max_seq=8192),
        # The launchers that take many rows at once, at the batched shapes of the element-wise set.
        dict(name="rows_batch", kind="rows", model="0.5b", rows=4096, keys=2048),
    ]


def _log_int(rng, low, high):
    """An integer of [low, high], spread over its logarithm."""
    return min(high, max(low, int(math.exp(rng.uniform(math.log(low), math.log(high + 1))))))


def draw(rng):
    kind = rng.choice(["decode_attention", "head", "sample", "decode", "prefill", "prefill", "mlp", "mlp",
                       "attention_block", "rows"])
    model = rng.choice(["0.5b", "7b"])
    if kind == "decode_attention":
        max_seq = _log_int(rng, 128, 32768)
        return dict(kind=kind, model=model, position=_log_int(rng, 1, max_seq - 1), max_seq=max_seq)
    if kind == "head":
        return dict(kind=kind, model=model)
    if kind == "sample":
        return dict(kind=kind, vocab=_log_int(rng, 8000, 152064), temperature=round(rng.uniform(0.2, 1.5), 2),
                    top_k=_log_int(rng, 1, 200), top_p=round(rng.uniform(0.5, 1.0), 2),
                    repeat_penalty=rng.choice([1.0, 1.05, 1.1, 1.3]), repeat_last_n=rng.choice([0, 16, 64, 256, -1]),
                    history=_log_int(rng, 1, 2000))
    if kind == "decode":
        max_seq = _log_int(rng, 256, 8192)
        return dict(kind=kind, model=model, layers=rng.randint(2, 24) if model == "0.5b" else rng.randint(1, 3),
                    position=_log_int(rng, 1, max_seq - 1), max_seq=max_seq)
    if kind == "prefill":
        count = _log_int(rng, 2, 2048)
        position = rng.choice([0, _log_int(rng, 1, 3000)])
        return dict(kind=kind, model=model, layers=rng.randint(2, 24) if model == "0.5b" else rng.randint(1, 3),
                    count=count, position=position, max_seq=max(256, position + count + rng.randint(0, 1000)))
    if kind == "mlp":
        return dict(kind=kind, model=model, rows=_log_int(rng, 1, 2048))
    if kind == "attention_block":
        rows = _log_int(rng, 8, 2048)
        position = rng.choice([0, _log_int(rng, 1, 6000)])
        return dict(kind=kind, model=model, rows=rows, position=position,
                    max_seq=position + rows + rng.randint(0, 1000))
    return dict(kind=kind, model=model, rows=_log_int(rng, 1, 4096 if model == "0.5b" else 1024),
                keys=_log_int(rng, 16, 2048))


# --------------------------------------------------------------------------------------------
# Inputs: everything from the seed alone, made on the GPU.

def _rand(seed, what, shape, std=1.0, mean=0.0, dtype=torch.float32):
    """N(mean, std): the tensor that (seed, what) names."""
    g = torch.Generator(device="cuda").manual_seed((seed * 1000003 + what * 7919 + 17) % (1 << 60))
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean).to(dtype)


def _tokens(seed, count, vocab):
    g = torch.Generator().manual_seed(seed * 31 + 5)
    return torch.randint(0, vocab, (count,), generator=g).numpy().astype(np.int32)


def _model(case):
    c = dict(MODELS[case["model"]])
    for key in ("layers", "max_seq"):
        c[key] = case.get(key, c[key])
    c["qdim"], c["kvdim"] = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    c["group"] = c["heads"] // c["kv_heads"]
    return c


_KINDS = ["ATTN_NORM", "ATTN_QKV", "ATTN_QKV_B", "ATTN_OUTPUT", "FFN_NORM", "FFN_GATE", "FFN_UP", "FFN_DOWN"]


def _weight(c, seed, kind, layer=0):
    """One weight tensor: matrices, embedding and biases N(0, 0.02), norms N(1, 0.1)."""
    h, f, q, kv = c["hidden"], c["ffn"], c["qdim"], c["kvdim"]
    shape = {"TOKEN_EMBD": (c["vocab"], h), "OUTPUT_NORM": (h,), "ATTN_NORM": (h,), "ATTN_QKV": (q + 2 * kv, h),
             "ATTN_QKV_B": (q + 2 * kv,), "ATTN_OUTPUT": (h, q), "FFN_NORM": (h,), "FFN_GATE": (f, h),
             "FFN_UP": (f, h), "FFN_DOWN": (h, f)}[kind]
    what = 100 + 16 * layer + mh.TENSOR[kind]
    if kind.endswith("NORM"):
        return _rand(seed, what, shape, 0.1, 1.0)
    return _rand(seed, what, shape, 0.02, dtype=torch.float32 if kind == "ATTN_QKV_B" else torch.float16)


def _cache(c, seed, layer, which, rows):
    """A cache [kv_heads][max_seq][head_dim] of which `rows` rows are filled with N(0, 1)."""
    t = torch.zeros((c["kv_heads"], c["max_seq"], c["head_dim"]), dtype=torch.float16, device="cuda")
    t[:, :rows] = _rand(seed, 50000 + 2 * layer + which, (c["kv_heads"], rows, c["head_dim"]), dtype=torch.float16)
    return t


class _Owner:
    """Closes a decoder with the last view of its memory."""

    def __init__(self, decoder):
        self.decoder = decoder

    def __del__(self):
        self.decoder.close()


class _Memory:
    """One of a decoder's tensors as the array interface torch reads; keeps the decoder."""

    def __init__(self, owner, kind, layer, shape, f16):
        self.owner = owner
        address, nbytes = owner.decoder.tensor(kind, layer)
        assert nbytes == math.prod(shape) * (2 if f16 else 4)
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f2" if f16 else "<f4",
                                             data=(address, False), strides=None, version=3)


def _view(owner, kind, layer, shape, f16=True):
    return torch.as_tensor(_Memory(owner, kind, layer, shape, f16), device="cuda")


def _decoder(case, seed, filled):
    """A decoder with its weights and `filled` cache rows, and the views that a pass returns."""
    c = _model(case)
    config = {k: c[k] for k in ("layers", "hidden", "ffn", "heads", "kv_heads", "head_dim", "vocab", "max_seq")}
    owner = _Owner(mh.Decoder(mh.qwen2_config(**config, eps=EPS, rope_base=ROPE_BASE)))
    cache = (c["kv_heads"], c["max_seq"], c["head_dim"])
    out = {"logits": _view(owner, "LOGITS", 0, (c["vocab"],), False), "k": [], "v": []}
    for kind in ("TOKEN_EMBD", "OUTPUT_NORM"):
        w = _weight(c, seed, kind)
        _view(owner, kind, 0, w.shape, w.dtype == torch.float16).copy_(w)
    for layer in range(c["layers"]):
        for kind in _KINDS:
            w = _weight(c, seed, kind, layer)
            _view(owner, kind, layer, w.shape, w.dtype == torch.float16).copy_(w)
        for which, (name, kind) in enumerate((("k", "KCACHE"), ("v", "VCACHE"))):
            view = _view(owner, kind, layer, cache)
            view.copy_(_cache(c, seed, layer, which, filled))
            out[name].append(view)
    torch.cuda.synchronize()
    return owner.decoder, out


def _split(x):
    hi = x.to(torch.float16)
    return hi, (x - hi.float()).to(torch.float16)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        decoder, out = _decoder(case, seed, case["position"])
        count = case.get("count", 1)
        return dict(kind=kind, decoder=decoder, out=out, tokens=_tokens(seed, count, _model(case)["vocab"]),
                    position=case["position"])
    lib = mh.load()
    s = dict(kind=kind, lib=lib)
    if kind == "sample":
        vocab = case["vocab"]
        p = mh.sampler_params(**{k: case[k] for k in ("temperature", "top_k", "top_p", "repeat_penalty",
                                                      "repeat_last_n")}, seed=seed)
        s.update(vocab=vocab, params=p, logits=_rand(seed, 1, (vocab,), 3.0),
                 work=torch.empty(vocab, device="cuda"), token=torch.zeros(1, dtype=torch.int32, device="cuda"),
                 history=torch.from_numpy(_tokens(seed, case["history"], vocab)).cuda(),
                 state=torch.zeros(lib.muyo_sampler_state_bytes(), dtype=torch.uint8, device="cuda"),
                 space=torch.zeros(lib.muyo_sample_workspace_bytes(vocab, mh.ref(p)), dtype=torch.uint8,
                                   device="cuda"))
        mh.check(lib.muyo_sampler_seed(s["state"].data_ptr(), seed, torch.cuda.current_stream().cuda_stream))
        return s
    c = _model(case)
    s["c"] = c
    h, f, q, kv, hd = c["hidden"], c["ffn"], c["qdim"], c["kvdim"], c["head_dim"]
    if kind == "head":
        vocab = c["vocab"]
        s.update(x=_rand(seed, 1, (h,)), norm=_weight(c, seed, "OUTPUT_NORM"), w=_weight(c, seed, "TOKEN_EMBD"),
                 y=torch.empty(h, device="cuda"), logits=torch.empty(vocab, device="cuda"),
                 token=torch.empty(1, dtype=torch.int32, device="cuda"), norm_pc=mh.rows_push_constants(h, 1, EPS),
                 head_pc=mh.mat_vec_push_constants(h, vocab), argmax_pc=mh.argmax_push_constants(vocab),
                 spec=mh.MuyoMatVecSpec(32, 1, 1))
    elif kind == "decode_attention":
        size = lib.muyo_attention_decode_f16kv_workspace_bytes(c["heads"], c["kv_heads"], hd, c["max_seq"])
        s.update(q=_rand(seed, 1, (q,)), k=_rand(seed, 2, (kv,)), v=_rand(seed, 3, (kv,)),
                 kcache=_cache(c, seed, 0, 0, case["position"]), vcache=_cache(c, seed, 0, 1, case["position"]),
                 q_out=torch.empty(q, device="cuda"), out=torch.empty(q, device="cuda"),
                 position=torch.tensor([case["position"]], dtype=torch.int32, device="cuda"),
                 space=torch.empty(size, dtype=torch.uint8, device="cuda"), theta=mh.theta_scale(ROPE_BASE, hd))
    elif kind == "mlp":
        rows = case["rows"]
        s.update(rows=rows, x=_rand(seed, 1, (rows, h)), norm=_weight(c, seed, "FFN_NORM"),
                 gate=_weight(c, seed, "FFN_GATE"), up=_weight(c, seed, "FFN_UP"),
                 down=_weight(c, seed, "FFN_DOWN"), out=torch.empty((rows, h), device="cuda"),
                 planes=[torch.empty((rows, n), dtype=torch.float16, device="cuda") for n in (h, h, f, f)])
    elif kind == "attention_block":
        rows, theta = case["rows"], np.float32(mh.theta_scale(ROPE_BASE, hd))
        size = lib.muyo_prefill_attention_workspace_bytes(rows, c["heads"], hd)
        powers = np.power(theta, np.arange(hd // 2, dtype=np.float32), dtype=np.float32)
        s.update(rows=rows, pos0=case["position"], qkv=_rand(seed, 1, (rows, q + 2 * kv)),
                 residual=_rand(seed, 2, (rows, h)), w=_weight(c, seed, "ATTN_OUTPUT"),
                 powers=torch.from_numpy(powers).cuda(), out=torch.empty((rows, h), device="cuda"),
                 kcache=_cache(c, seed, 0, 0, case["position"]), vcache=_cache(c, seed, 0, 1, case["position"]),
                 planes=[torch.empty((rows, q), dtype=torch.float16, device="cuda") for _ in range(4)],
                 space=torch.empty(size, dtype=torch.uint8, device="cuda"))
    else:
        rows, heads, keys = case["rows"], c["heads"] + c["kv_heads"], case["keys"]
        new = {n: _rand(seed, i, shape, std) for i, (n, shape, std) in enumerate((
            ("x", (rows, h), 1.0), ("b", (rows, h), 1.0), ("gate", (rows, f), 1.0), ("up", (rows, f), 1.0),
            ("qk", (rows, heads * hd), 1.0), ("scores", (rows * c["heads"], keys), 3.0)))}
        g = torch.Generator(device="cuda").manual_seed(seed + 77)
        s.update(new, rows=rows, heads=heads, keys=keys, norm=_rand(seed, 9, (h,), 0.1, 1.0, torch.float16),
                 positions=torch.randint(0, 2048, (rows,), dtype=torch.int32, device="cuda", generator=g),
                 out={n: torch.empty_like(new[m]) for n, m in (("norm", "x"), ("sum", "x"), ("act", "gate"),
                                                               ("roped", "qk"), ("probs", "scores"))},
                 norm_pc=mh.rows_push_constants(h, rows, EPS), add_pc=mh.add_push_constants(rows * h, row=h),
                 glu_pc=mh.glu_push_constants(rows * f, f),
                 rope_pc=mh.rope_push_constants(heads, hd, ROPE_BASE, tokens=rows),
                 soft_pc=mh.soft_max_push_constants(rows * c["heads"], keys, 1.0))
    return s


# --------------------------------------------------------------------------------------------
# One pass.

def run(s):
    kind = s["kind"]
    if kind == "decode":
        token = s["decoder"].step(int(s["tokens"][0]), s["position"])
        return dict(s["out"], token=token)
    if kind == "prefill":
        token = s["decoder"].prefill(s["tokens"], s["position"])
        return dict(s["out"], token=token)
    lib, check, ref = s["lib"], mh.check, mh.ref
    stream = torch.cuda.current_stream().cuda_stream
    if kind == "sample":
        # A token's logits arrive in a buffer of their own; the sampler works on them in place.
        s["work"].copy_(s["logits"])
        check(lib.muyo_sample_f32(s["work"].data_ptr(), s["vocab"], s["history"].data_ptr(), s["history"].numel(),
                                  ref(s["params"]), s["state"].data_ptr(), s["space"].data_ptr(),
                                  s["token"].data_ptr(), stream))
        return {"logits": s["work"], "token": s["token"]}
    c = s["c"]
    h, q, hd = c["hidden"], c["qdim"], c["head_dim"]
    if kind == "head":
        check(lib.muyo_rms_norm_f32(ref(s["norm_pc"]), 1, s["x"].data_ptr(), s["norm"].data_ptr(),
                                    s["y"].data_ptr(), None, 1, 1, 1, stream))
        check(lib.muyo_mul_mat_vec_f16_f32_f32(ref(s["head_pc"]), ref(s["spec"]), s["w"].data_ptr(),
                                               s["y"].data_ptr(), s["logits"].data_ptr(), None, None, c["vocab"], 1,
                                               1, stream))
        check(lib.muyo_argmax_f32(ref(s["argmax_pc"]), s["logits"].data_ptr(), s["token"].data_ptr(), 1, 1, 1,
                                  stream))
        return {"norm": s["y"], "logits": s["logits"], "token": s["token"]}
    if kind == "decode_attention":
        sizes = (c["heads"], c["kv_heads"], hd, c["max_seq"])
        check(lib.muyo_rope_append_f16kv(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                         s["q_out"].data_ptr(), s["kcache"].data_ptr(), s["vcache"].data_ptr(),
                                         s["position"].data_ptr(), *sizes, s["theta"], stream))
        check(lib.muyo_attention_decode_f16kv(s["q_out"].data_ptr(), s["kcache"].data_ptr(), s["vcache"].data_ptr(),
                                              s["out"].data_ptr(), s["position"].data_ptr(), *sizes,
                                              1.0 / math.sqrt(hd), s["space"].data_ptr(), s["space"].numel(),
                                              stream))
        return {k: s[k] for k in ("q_out", "out", "kcache", "vcache")}
    if kind == "mlp":
        nhi, nlo, ahi, alo = (p.data_ptr() for p in s["planes"])
        rows, f = s["rows"], c["ffn"]
        check(lib.muyo_rms_norm_split_f16x2(s["x"].data_ptr(), s["norm"].data_ptr(), rows, h, EPS, nhi, nlo, stream))
        check(lib.muyo_gemm_swiglu_split_f16(nhi, nlo, s["gate"].data_ptr(), s["up"].data_ptr(), ahi, alo, rows, f,
                                             h, stream))
        check(lib.muyo_gemm_split_f16(ahi, alo, s["down"].data_ptr(), None, s["x"].data_ptr(), s["out"].data_ptr(),
                                      rows, h, f, stream))
        return s["out"]
    if kind == "attention_block":
        qhi, qlo, ohi, olo = (p.data_ptr() for p in s["planes"])
        rows, sizes = s["rows"], (c["heads"], c["kv_heads"], hd, c["max_seq"])
        check(lib.muyo_rope_split_append_f16kv(s["qkv"].data_ptr(), rows, s["pos0"], *sizes, s["powers"].data_ptr(),
                                               qhi, qlo, s["kcache"].data_ptr(), s["vcache"].data_ptr(), stream))
        check(lib.muyo_prefill_attention_f16kv_ws(qhi, qlo, s["kcache"].data_ptr(), s["vcache"].data_ptr(), ohi, olo,
                                                  rows, s["pos0"], *sizes, 1.0 / math.sqrt(hd),
                                                  s["space"].data_ptr(), s["space"].numel(), stream))
        check(lib.muyo_gemm_split_f16(ohi, olo, s["w"].data_ptr(), None, s["residual"].data_ptr(),
                                      s["out"].data_ptr(), rows, h, q, stream))
        return {k: s[k] for k in ("out", "kcache", "vcache")}
    rows, out = s["rows"], {k: t.data_ptr() for k, t in s["out"].items()}
    check(lib.muyo_rms_norm_f32_f16w(ref(s["norm_pc"]), 1, s["x"].data_ptr(), s["norm"].data_ptr(), out["norm"],
                                     None, rows, 1, 1, stream))
    check(lib.muyo_add_f32(ref(s["add_pc"]), 1, s["x"].data_ptr(), s["b"].data_ptr(), out["sum"], None,
                           *mh.add_dispatch(rows * h), stream))
    check(lib.muyo_swiglu_f32(ref(s["glu_pc"]), s["gate"].data_ptr(), s["up"].data_ptr(), out["act"],
                              *mh.add_dispatch(rows * c["ffn"]), stream))
    check(lib.muyo_rope_neox_f32(ref(s["rope_pc"]), s["qk"].data_ptr(), s["positions"].data_ptr(), None,
                                 out["roped"], None, s["heads"] * rows, 1, 1, stream))
    check(lib.muyo_soft_max_f32(ref(s["soft_pc"]), s["scores"].data_ptr(), None, None, out["probs"],
                                *mh.row_dispatch(rows * c["heads"]), stream))
    return s["out"]


# --------------------------------------------------------------------------------------------
# What a pass cannot do without.

def work(case):
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": 4 * 2 * case["vocab"] + 4 * case["history"], "flops": 0}
    c = _model(case)
    h, f, q, kv, hd = c["hidden"], c["ffn"], c["qdim"], c["kvdim"], c["head_dim"]
    if kind == "head":
        return {"bytes": 2 * c["vocab"] * h + 4 * (3 * h + c["vocab"]), "flops": 2 * c["vocab"] * h}
    if kind == "decode_attention":
        keys = case["position"] + 1
        return {"bytes": 4 * kv * keys + 4 * (3 * q + 2 * kv), "flops": 4 * q * keys}
    if kind == "mlp":
        # Both planes of every activation meet every weight: two products each.
        return {"bytes": 6 * f * h + 4 * (2 * case["rows"] * h + h), "flops": 2 * 2 * case["rows"] * 3 * f * h}
    if kind == "attention_block":
        rows, pos = case["rows"], case["position"]
        pairs = rows * pos + rows * (rows + 1) // 2
        return {"bytes": 4 * rows * (q + 2 * kv + 2 * h) + 4 * kv * (pos + 2 * rows) + 2 * h * q,
                "flops": 2 * 4 * q * pairs + 2 * 2 * rows * h * q}
    if kind == "rows":
        rows = case["rows"]
        return {"bytes": rows * 4 * (2 * h + 3 * h + 3 * f + 2 * (q + kv) + 2 * c["heads"] * case["keys"]),
                "flops": 0}
    layer = (q + 2 * kv) * h + h * q + 3 * f * h
    rows, pos = case.get("count", 1), case["position"]
    pairs = rows * pos + rows * (rows + 1) // 2
    return {"bytes": c["layers"] * (2 * layer + 4 * kv * (pos + rows) + 4 * (q + 2 * kv + 2 * h))
            + 2 * c["vocab"] * h + 2 * rows * h + 4 * c["vocab"],
            "flops": c["layers"] * (2 * rows * layer + 4 * q * pairs) + 2 * c["vocab"] * h}


def tolerance(case):
    """About four times what each kind's outputs are off their 64-bit values at the listed sizes."""
    return {
        # Angles are an f32 power times the position: 1.4e-4 of q at row 20011. The cache rows are
        # fp16, and a value at a rounding boundary may fall to either side of it.
        "decode_attention": {"rel": 6e-4, "max": 1e-2},
        "head": {"rel": 1e-6, "max": 2e-5},
        "sample": {"rel": 2e-7, "max": 1e-6},
        # fp16 cache rows again: in a whole model one value's rounding reaches every later layer.
        "decode": {"rel": 2e-4, "max": 1e-2},
        "mlp": {"rel": 2e-6, "max": 4e-5},
        "attention_block": {"rel": 2e-4, "max": 1e-2},
        "prefill": {"rel": 8e-4, "max": 2e-2},
        "rows": {"rel": 2e-5, "max": 4e-4},
    }[case["kind"]]


# --------------------------------------------------------------------------------------------
# The same results in 64 bits, by torch alone.

def _norm64(x, w):
    x = x.double()
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, positions, theta):
    """NeoX rotation of x [rows][heads][hd]: pairs (j, j + hd/2) by positions * theta^j."""
    half = x.shape[-1] // 2
    angle = positions.double()[:, None] * torch.pow(torch.tensor(theta, dtype=torch.float64, device="cuda"),
                                                    torch.arange(half, dtype=torch.float64, device="cuda"))
    cos, sin = angle.cos()[:, None], angle.sin()[:, None]
    a, b = x[..., :half].double(), x[..., half:].double()
    return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)


def _attend64(q, kcache, vcache, pos0, group):
    """Causal attention of q [rows][heads][hd] at positions pos0.. over the caches."""
    rows, heads, hd = q.shape
    keys = pos0 + rows
    late = torch.arange(keys, device="cuda")[None, :] > torch.arange(pos0, keys, device="cuda")[:, None]
    out = torch.empty_like(q)
    for i in range(heads):
        scores = (q[:, i] @ kcache[i // group, :keys].double().t().contiguous()) / math.sqrt(hd)
        out[:, i] = torch.softmax(scores.masked_fill_(late, -math.inf), -1) @ vcache[i // group, :keys].double()
    return out


def _append64(c, qkv, kcache, vcache, pos0):
    """Ropes q and k, appends k and v (rounded to fp16) to the caches, and returns q."""
    rows, theta = qkv.shape[0], mh.theta_scale(ROPE_BASE, c["head_dim"])
    q, kv, hd = c["qdim"], c["kvdim"], c["head_dim"]
    positions = torch.arange(pos0, pos0 + rows, device="cuda")
    k = _rope64(qkv[:, q:q + kv].reshape(rows, -1, hd), positions, theta)
    kcache[:, pos0:pos0 + rows] = k.transpose(0, 1).half()
    vcache[:, pos0:pos0 + rows] = qkv[:, q + kv:].reshape(rows, -1, hd).transpose(0, 1).half()
    return _rope64(qkv[:, :q].reshape(rows, -1, hd), positions, theta)


def _linear64(x, w):
    return x @ w.double().t().contiguous()


def _mlp64(c, x, norm, gate, up, down):
    n = _norm64(x, norm)
    g = _linear64(n, gate)
    return x.double() + _linear64(g * torch.sigmoid(g) * _linear64(n, up), down)


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        # The token is a draw of the engine: no value in 64 bits.
        logits = _rand(seed, 1, (case["vocab"],), 3.0).double()
        history = _tokens(seed, case["history"], case["vocab"]).tolist()
        last = case["repeat_last_n"]
        penalty = float(np.float32(case["repeat_penalty"]))
        if penalty != 1.0:
            values = logits.cpu().numpy()
            for t in history if last < 0 else history[max(0, len(history) - last):]:
                values[t] = values[t] / penalty if values[t] > 0 else values[t] * penalty
            logits = torch.from_numpy(values).cuda()
        return {"logits": logits / float(np.float32(case["temperature"])), "token": None}
    c = _model(case)
    h, f, q, kv, hd = c["hidden"], c["ffn"], c["qdim"], c["kvdim"], c["head_dim"]
    if kind == "head":
        n = _norm64(_rand(seed, 1, (h,)), _weight(c, seed, "OUTPUT_NORM"))
        logits = _weight(c, seed, "TOKEN_EMBD").double() @ n
        return {"norm": n, "logits": logits, "token": None}
    if kind == "decode_attention":
        pos = case["position"]
        kcache, vcache = (_cache(c, seed, 0, i, pos) for i in (0, 1))
        qkv = torch.cat([_rand(seed, 1, (q,)), _rand(seed, 2, (kv,)), _rand(seed, 3, (kv,))])[None]
        roped = _append64(c, qkv, kcache, vcache, pos)
        return {"q_out": roped.reshape(-1), "out": _attend64(roped, kcache, vcache, pos, c["group"]).reshape(-1),
                "kcache": kcache.double(), "vcache": vcache.double()}
    if kind == "mlp":
        return _mlp64(c, _rand(seed, 1, (case["rows"], h)), *(_weight(c, seed, k) for k in (
            "FFN_NORM", "FFN_GATE", "FFN_UP", "FFN_DOWN")))
    if kind == "attention_block":
        rows, pos = case["rows"], case["position"]
        kcache, vcache = (_cache(c, seed, 0, i, pos) for i in (0, 1))
        roped = _append64(c, _rand(seed, 1, (rows, q + 2 * kv)), kcache, vcache, pos)
        attn = _attend64(roped, kcache, vcache, pos, c["group"]).reshape(rows, -1)
        return {"out": _rand(seed, 2, (rows, h)).double() + _linear64(attn, _weight(c, seed, "ATTN_OUTPUT")),
                "kcache": kcache.double(), "vcache": vcache.double()}
    if kind == "rows":
        rows, heads = case["rows"], c["heads"] + c["kv_heads"]
        x, b = _rand(seed, 0, (rows, h)), _rand(seed, 1, (rows, h))
        gate, up = _rand(seed, 2, (rows, f)).double(), _rand(seed, 3, (rows, f)).double()
        g = torch.Generator(device="cuda").manual_seed(seed + 77)
        positions = torch.randint(0, 2048, (rows,), dtype=torch.int32, device="cuda", generator=g)
        roped = _rope64(_rand(seed, 4, (rows, heads * hd)).reshape(rows, heads, hd), positions,
                        mh.theta_scale(ROPE_BASE, hd))
        return {"norm": _norm64(x, _rand(seed, 9, (h,), 0.1, 1.0, torch.float16)), "sum": x.double() + b.double(),
                "act": gate * torch.sigmoid(gate) * up, "roped": roped.reshape(rows, -1),
                "probs": torch.softmax(_rand(seed, 5, (rows * c["heads"], case["keys"]), 3.0).double(), -1)}
    # A whole model, layer by layer.
    rows, pos = case.get("count", 1), case["position"]
    embed = _weight(c, seed, "TOKEN_EMBD")
    x = embed[torch.from_numpy(_tokens(seed, rows, c["vocab"])).long().cuda()].double()
    out = {"k": [], "v": [], "token": None}
    for layer in range(c["layers"]):
        w = {k: _weight(c, seed, k, layer) for k in _KINDS}
        kcache, vcache = (_cache(c, seed, layer, i, pos) for i in (0, 1))
        qkv = _linear64(_norm64(x, w["ATTN_NORM"]), w["ATTN_QKV"]) + w["ATTN_QKV_B"].double()
        roped = _append64(c, qkv, kcache, vcache, pos)
        x = x + _linear64(_attend64(roped, kcache, vcache, pos, c["group"]).reshape(rows, -1), w["ATTN_OUTPUT"])
        x = _mlp64(c, x, w["FFN_NORM"], w["FFN_GATE"], w["FFN_UP"], w["FFN_DOWN"])
        out["k"].append(kcache)
        out["v"].append(vcache)
    n = _norm64(x[-1], _weight(c, seed, "OUTPUT_NORM"))
    out["logits"] = embed.double() @ n
    return out
