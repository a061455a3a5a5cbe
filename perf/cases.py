"""What a program built on this library has it do, as timed cases.

Two kinds of programs use it.  One holds an encoder of the BERT driver
(``BertEncoder``): weights are uploaded and the call list is captured once, then
every request hands in token ids and a padding mask on the host and takes hidden
states (or masked-LM logits) back on the host.  The other is a lowered module, or
a host program written against the C-ABI: its tensors stay on the GPU and it
calls the operator entry points one after the other.  ``listed()`` has both;
``draw()`` spreads the same families over their ranges.
"""
import ctypes
import importlib
import math

import torch

_rt = importlib.import_module("hands-on-mlir_amd.hom_runtime")
_bert = importlib.import_module("hands-on-mlir_amd.bert")

BASE = {"layers": 12, "hidden": 768, "heads": 12, "ffn": 3072}
LARGE = {"layers": 24, "hidden": 1024, "heads": 16, "ffn": 4096}
VOCAB = 30522
EPS = 1e-12


def listed():
    return [
        # One short text at a time: the smallest request of the reference's latency grid
        # ({base, large} x batch {1, 8, 16, 32} x seq {64, 128}), all launch and host latency.
        dict(name="bert_base_b1_s64", kind="encoder", batch=1, seq=64, lm=False, gelu="erf", **BASE),
        # The headline configuration: BERT-base, batch 8, sequence 128.
        dict(name="bert_base_b8_s128", kind="encoder", batch=8, seq=128, lm=False, gelu="erf", **BASE),
        # The largest configuration: BERT-large, batch 32, sequence 512.
        dict(name="bert_large_b32_s512", kind="encoder", batch=32, seq=512, lm=False, gelu="erf", **LARGE),
        # Masked-LM scoring of a couple of sentences padded to a length of their own (no
        # multiple of anything), tanh GELU as the nvte path has it, logits over the vocabulary.
        dict(name="masked_lm_base_b2_s57", kind="encoder", batch=2, seq=57, lm=True, gelu="tanh", **BASE),
        # A feed-forward layer with bias and GELU over a long batch of BERT-large tokens.
        dict(name="gemm_gelu_16384x4096x1024", kind="gemm", M=16384, N=4096, K=1024, layout="kn", act=1, source="bias"),
        # The fused QKV projection over a token count as it comes, weights stored [N, K].
        dict(name="gemm_nk_1531x2304x768", kind="gemm", M=1531, N=2304, K=768, layout="nk", act=0, source="none"),
        # Few rows against a wide weight (the skinny split-K shape) with a residual.
        dict(name="gemm_skinny_64x1024x4096", kind="gemm", M=64, N=1024, K=4096, layout="kn", act=0, source="full"),
        # A layer whose feature counts are odd: no row of A, B, C or D starts aligned.
        dict(name="gemm_odd_1000x1001x1003", kind="gemm", M=1000, N=1001, K=1003, layout="kn", act=0, source="bias"),
        # Residual GEMM -> layer norm -> GEMM as the fused pair: row statistics out of the first
        # GEMM, normalisation inside the second.
        dict(name="ln_gemm_pair_4096x1024_to_4096", kind="ln_pair", M=4096, H=1024, F=4096),
        # Attention on its own with the larger head size, ragged lengths.
        dict(name="attention_b8_s384_h16_d128", kind="attention", batch=8, seq=384, heads=16, d=128),
        # Residual add + affine layer norm over a batch of BERT-base tokens.
        dict(name="add_layernorm_8192x768", kind="layernorm", rows=8192, H=768, dtype="f16", residual=True),
        # The embedding front of a model: lengths from the mask, word rows gathered, positions
        # added, padding multiplied away by a [b, s, 1] mask (fp32, as an fp32 graph has it).
        dict(name="embed_f32_b16_s200", kind="embed", batch=16, seq=200, H=768, dtype="f32"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["encoder", "encoder", "encoder", "gemm", "gemm", "gemm", "gemm",
                       "ln_pair", "attention", "layernorm", "embed"])
    if kind == "encoder":
        size = rng.choice([BASE, BASE, LARGE])
        lm = rng.random() < 0.25
        # (logits are vocab wide: scoring is done for a few sentences at a time)
        return dict(kind=kind, batch=_log(rng, 1, 4 if lm else 32), seq=_log(rng, 16, 128 if lm else 512), lm=lm,
                    gelu=rng.choice(["erf", "erf", "tanh"]), **size)
    if kind == "gemm":
        layout = rng.choice(["kn", "kn", "nk"])
        M, N, K = _log(rng, 16, 16384), _log(rng, 256, 4096), _log(rng, 256, 4096)
        # feature counts: mostly multiples of 64 or 8, some as they come
        step = rng.choice([64, 64, 8, 1])
        N, K = max(step, N // step * step), max(step, K // step * step)
        return dict(kind=kind, M=M, N=N, K=K, layout=layout, act=rng.choice([0, 0, 1]),
                    source=rng.choice(["none", "bias", "full"]) if layout == "kn" else "none")
    if kind == "ln_pair":
        H = rng.choice([768, 1024])
        return dict(kind=kind, M=_log(rng, 64, 16384), H=H, F=rng.choice([H, 3 * H, 4 * H]))
    if kind == "attention":
        d = rng.choice([64, 64, 128, 192, 256])
        return dict(kind=kind, batch=_log(rng, 1, 32), seq=_log(rng, 16, 768), heads=rng.choice([8, 12, 16]), d=d)
    if kind == "layernorm":
        H = _log(rng, 64, 8192)
        step = rng.choice([64, 8, 1])
        return dict(kind=kind, rows=_log(rng, 64, 8192), H=max(step, H // step * step),
                    dtype=rng.choice(["f16", "f16", "f32"]), residual=rng.random() < 0.5)
    H = rng.choice([768, 1024, _log(rng, 64, 2048)])
    return dict(kind=kind, batch=_log(rng, 1, 64), seq=_log(rng, 16, 512), H=H, dtype=rng.choice(["f16", "f32"]))


class _Inputs:
    """Seeded device tensors."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, mean=0.0, dtype=torch.float16):
        t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=self.g)
        return t.to(dtype)

    def integers(self, lo, hi, *shape):
        return torch.randint(lo, hi, shape, generator=self.g, device="cuda", dtype=torch.int64)

    def lengths(self, batch, seq):
        return self.integers(max(1, seq // 4), seq + 1, batch)


def _empty(*shape, dtype=torch.float16):
    return torch.empty(shape, dtype=dtype, device="cuda")


def _mask(lens, seq):
    return (torch.arange(seq, device="cuda")[None, :] < lens[:, None]).to(torch.int64)


class _Call:
    """One entry point with its operands' descriptors laid out, as generated code keeps them."""

    def __init__(self, name, *args):
        self.keep, flat = [], []
        for a in args:
            if isinstance(a, torch.Tensor):
                m = _rt.MemRef.from_tensor(a)
                self.keep += [m, a]
                flat += [m.rank, ctypes.cast(m.descriptor, ctypes.c_void_p).value]
            elif a is None:  # an absent operand
                flat += [0, None]
            else:
                flat.append(a)
        self.args = flat
        self.fn = getattr(_rt.load_runtime(), name)

    def __call__(self):
        self.fn(*self.args)


class _EncoderState:
    def __init__(self, case, seed):
        x = _Inputs(seed)
        host = lambda t: t.cpu().numpy()  # noqa: E731
        H, F, L = case["hidden"], case["ffn"], case["layers"]
        b, s = case["batch"], case["seq"]
        weights = [{"wqkv": host(x.normal(H, 3 * H, std=0.02)), "wo": host(x.normal(H, H, std=0.02)),
                    "w1": host(x.normal(H, F, std=0.02)), "w2": host(x.normal(F, H, std=0.02))} for _ in range(L)]
        model = {"weights": weights, "word": host(x.normal(VOCAB, H, std=0.02)),
                 "pos_type": host(x.normal(s, H, std=0.02)), "w_transform": host(x.normal(H, H, std=0.02))}
        self.ids = host(x.integers(0, VOCAB, b, s))
        self.mask = host(_mask(x.lengths(b, s), s))
        self.lm = case["lm"]
        self.enc = _bert.BertEncoder(layers=L, hidden=H, heads=case["heads"], ffn=F, bs=b, seq=s, vocab=VOCAB,
                                     gelu_form=case["gelu"], lm_head=self.lm)
        self.enc.load(model)
        self.enc.set_inputs(ids=self.ids, mask=self.mask)
        self.enc.capture()

    def __del__(self):
        enc = getattr(self, "enc", None)
        if enc is not None:
            enc.close()

    def run(self):
        self.enc.set_inputs(ids=self.ids, mask=self.mask)
        self.enc.replay()
        return self.enc.logits() if self.lm else self.enc.output()


class _CallList:
    def __init__(self, calls, outputs):
        self.calls, self.outputs = calls, outputs

    def run(self):
        for c in self.calls:
            c()
        return self.outputs


def _prepare_gemm(case, x):
    M, N, K = case["M"], case["N"], case["K"]
    nk = case["layout"] == "nk"
    A = x.normal(1, M, K)
    B = x.normal(1, N, K, std=0.02) if nk else x.normal(1, K, N, std=0.02)
    D = _empty(1, M, N)
    C = {"none": D, "bias": x.normal(1, 1, N, std=0.02), "full": x.normal(1, M, N)}[case["source"]]
    beta = 0.0 if case["source"] == "none" else 1.0
    call = _Call("nvteGemmF16" if nk else "cutlassGemmF16", A, False, B, nk, C, D, case["act"], 1.0, beta, 0, 1)
    return _CallList([call], [D])


def _prepare_ln_pair(case, x):
    # x1 = attn . Wo + x  with the row statistics of x1;  y = LN(x1) . W1
    M, H, F = case["M"], case["H"], case["F"]
    A, Wo, R, W1 = x.normal(1, M, H), x.normal(1, H, H, std=0.02), x.normal(1, M, H), x.normal(1, H, F, std=0.02)
    X1, Y, var, mean = _empty(1, M, H), _empty(1, M, F), _empty(1, M, 1), _empty(1, M, 1)
    return _CallList([_Call("cutlassGemmWithVarMeanF16", A, Wo, R, X1, var, mean, 1.0, 1.0, 0, EPS),
                      _Call("cutlassLayernormGemmF16", X1, W1, Y, Y, var, mean, 1.0, 0.0, 0)], [X1, var, mean, Y])


def _prepare_attention(case, x):
    b, s, h, d = case["batch"], case["seq"], case["heads"], case["d"]
    qkv = x.normal(b, s, 3 * h * d)
    cu = torch.zeros(b + 1, dtype=torch.int32, device="cuda")
    cu[1:] = torch.cumsum(x.lengths(b, s), 0)
    out = _empty(b, s, h * d)
    return _CallList([_Call("nvteBertAttentionF16", qkv, cu, out, 1.0 / math.sqrt(d), h)], [out])


def _prepare_layernorm(case, x):
    rows, H = case["rows"], case["H"]
    if case["dtype"] == "f32":  # an fp32 graph's add (of a tensor or one bias row), then the in-place layer norm
        X, Y = x.normal(1, rows, H, std=2.0, mean=0.5, dtype=torch.float32), _empty(1, rows, H, dtype=torch.float32)
        R = x.normal(1, rows if case["residual"] else 1, H, dtype=torch.float32)
        return _CallList([_Call("thrustElementwiseAddF32", X, R, Y), _Call("nvteLayernormF32", Y, EPS)], [Y])
    X, Y = x.normal(1, rows, H, std=2.0, mean=0.5), _empty(1, rows, H)
    if not case["residual"]:
        return _CallList([_Call("homAddLayernormF16", X, None, None, None, Y, EPS)], [Y])
    R, gamma, beta = x.normal(1, rows, H), x.normal(H, std=0.02, mean=1.0), x.normal(H, std=0.02)
    return _CallList([_Call("homAddLayernormF16", X, R, gamma, beta, Y, EPS)], [Y])


def _prepare_embed(case, x):
    b, s, H = case["batch"], case["seq"], case["H"]
    sfx, dt = ("F16", torch.float16) if case["dtype"] == "f16" else ("F32", torch.float32)
    ids, mask = x.integers(0, VOCAB, b, s), _mask(x.lengths(b, s), s)
    word, pos = x.normal(1, VOCAB, H, std=0.02, dtype=dt), x.normal(1, s, H, std=0.02, dtype=dt)
    keep = mask.to(dt).reshape(b, s, 1)
    cu = _empty(b + 1, dtype=torch.int32)
    rows, summed, out = (_empty(b, s, H, dtype=dt) for _ in range(3))
    return _CallList([_Call("thrustCuSeqLenI64", mask, cu), _Call("thrustGather" + sfx, ids, word, rows),
                      _Call("thrustElementwiseAdd" + sfx, rows, pos, summed),
                      _Call("thrustElementwiseMul" + sfx, summed, keep, out)], [cu, out])


_PREPARE = {"gemm": _prepare_gemm, "ln_pair": _prepare_ln_pair, "attention": _prepare_attention,
            "layernorm": _prepare_layernorm, "embed": _prepare_embed}


def prepare(case, seed):
    if case["kind"] == "encoder":
        return _EncoderState(case, seed)
    return _PREPARE[case["kind"]](case, _Inputs(seed))


def run(state):
    return state.run()


def work(case):
    kind = case["kind"]
    if kind == "encoder":
        # Weights once, the request in and the answer out; activations need not leave the chip.
        L, H, F, b, s = (case[k] for k in ("layers", "hidden", "ffn", "batch", "seq"))
        M = b * s
        weights = L * (4 * H * H + 2 * H * F)
        flops = 2 * M * weights + L * 4 * b * s * s * H * 0.4375  # (as for attention below)
        nbytes = 2 * weights + 2 * s * H + min(M, VOCAB) * H * 2 + 16 * M + 2 * M * H
        if case["lm"]:
            flops += 2 * M * (H * H + H * VOCAB)
            nbytes += 2 * (H * H + H * VOCAB) + 2 * M * VOCAB - 2 * M * H
        return {"bytes": nbytes, "flops": flops}
    if kind == "gemm":
        M, N, K = case["M"], case["N"], case["K"]
        source = {"none": 0, "bias": N, "full": M * N}[case["source"]]
        return {"bytes": 2 * (M * K + K * N + M * N + source), "flops": 2 * M * N * K}
    if kind == "ln_pair":
        M, H, F = case["M"], case["H"], case["F"]
        return {"bytes": 2 * (3 * M * H + H * H + H * F + M * F + 2 * M), "flops": 2 * M * H * (H + F)}
    if kind == "attention":
        # lengths are uniform in [seq / 4, seq]: mean of len^2 is (1 + 1/4 + 1/16) / 3 of seq^2
        b, s, hd = case["batch"], case["seq"], case["heads"] * case["d"]
        return {"bytes": 2 * (3 * 0.625 * b * s * hd + b * s * hd), "flops": 4 * hd * b * s * s * 0.4375}
    size = 2 if case["dtype"] == "f16" else 4
    if kind == "layernorm":
        rows, H = case["rows"], case["H"]
        return {"bytes": size * rows * H * (3 if case["residual"] else 2), "flops": 8 * rows * H}
    b, s, H = case["batch"], case["seq"], case["H"]
    n = b * s
    return {"bytes": size * (2 * n * H + s * H) + 8 * 2 * n + size * n, "flops": 2 * n * H}


def tolerance(case):
    kind = case["kind"]
    if kind == "encoder":
        # fp16 activations through 12 or 24 layers: two pipelines that round in different places
        # come out 1e-3 to 3e-3 apart in norm, the LM head adds its own GEMMs
        return {"rel": 5e-3}
    if kind == "embed":
        return "exact"  # lengths, copied rows, one rounded sum, a product with 0 or 1
    if kind == "layernorm" and case["dtype"] == "f32":
        return {"rel": 1e-5}
    # fp32 accumulation, one rounding to fp16 (2^-11 relative at most)
    return {"rel": 1e-3}
