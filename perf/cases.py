"""The work that a user of this library has it do, as measurable cases.

The library serves the matmul path of the Whisper large-v3-turbo engine:
encoder layers over a window (or many windows), the decoder at one token, a
batch of tokens or a prompt, the logits, and the loading of weights.  Every
case goes through the operator wrappers of madi_amd.q8, as an engine calls
them.  Widths are the model's own (1280, 3840, 5120, vocabulary 51866); row
counts range over what those operators are called with.

Weights are random Q8 rows (int8 quants, one fp16 scale per 32) of about the
spread of trained projections (rms 0.04), activations N(0, 1) as after a
layer norm; both are made from the seed alone, on the GPU.
"""
from __future__ import annotations

import math

import torch

from madi_amd import lib, q8

D, MLP, VOCAB = q8.D, q8.MLP, q8.VOCAB
DEC_LAYERS = 4
CACHE_ROWS = 448  # the decoder's positions


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one decoder projection for one token: the smallest call there is
        dict(name="gemv_bias_1280", kind="gemv", n=D, k=D),
        # one token through the decoder's projections and logits (the inner
        # loop of transcription): embedding row, 4 layers of six GEMVs, logits
        dict(name="decode_token", kind="token", layers=DEC_LAYERS, pos=57),
        # the logits alone (67 MB of weights for one row)
        dict(name="logits_51866", kind="logits", vocab=VOCAB),
        # several segments decoded side by side: one layer's six projections
        dict(name="batched_layer_8", kind="rows", m=8),
        # and their logits, through the engine's dequantised tok_emb handle
        dict(name="batched_logits_16", kind="batched_logits", m=16, vocab=VOCAB),
        # a prompt's rows through one decoder layer's six projections
        dict(name="prefill_layer_320", kind="rows", m=320),
        # one encoder layer over a 30 s window, in the engine's call order:
        # q|k|v, attention, out, fc1 + GELU, fc2
        dict(name="encoder_layer_1500", kind="encoder", seq=1500),
        # the same over a short streaming window (7.5 s), an odd row count
        dict(name="encoder_layer_375", kind="encoder", seq=375),
        # encoder self-attention of one window
        dict(name="attention_1500", kind="attention", seq=1500, heads=20),
        # the MLP over a long recording's 16 windows at once
        dict(name="long_audio_mlp_24000", kind="mlp", m=24000),
        # the engine's F16-cache mode: one layer's GEMMs on F16 weights
        dict(name="f16_cache_layer_1500", kind="f16_layer", m=1500),
        # loading: F16 rows quantised to the Q8 layout on the GPU
        dict(name="quantize_fc1", kind="quantize", n=MLP, k=D),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "token", "logits", "rows", "rows", "batched_logits", "encoder", "encoder",
                       "attention", "mlp", "f16_layer", "quantize"])
    if kind == "gemv":
        return dict(kind=kind, n=_log(rng, 384, 3 * MLP), k=64 * _log(rng, 6, 80))
    if kind == "token":
        return dict(kind=kind, layers=rng.randint(1, DEC_LAYERS), pos=rng.randint(0, CACHE_ROWS - 1))
    if kind == "logits":
        return dict(kind=kind, vocab=rng.randint(20000, VOCAB))
    if kind == "rows":
        return dict(kind=kind, m=_log(rng, 2, CACHE_ROWS))
    if kind == "batched_logits":
        return dict(kind=kind, m=rng.randint(2, 32), vocab=rng.randint(20000, VOCAB))
    if kind == "encoder":
        return dict(kind=kind, seq=_log(rng, 100, 1500))
    if kind == "attention":
        return dict(kind=kind, seq=_log(rng, 64, 3000), heads=rng.randint(6, 20))
    if kind == "mlp":
        return dict(kind=kind, m=_log(rng, 1501, 24000))
    if kind == "f16_layer":
        return dict(kind=kind, m=_log(rng, 100, 1500))
    return dict(kind=kind, n=_log(rng, 384, VOCAB), k=64 * _log(rng, 6, 80))


# ---------------------------------------------------------------- inputs
class DeviceBuffer:
    """Device memory of the library's own (madi_alloc), as the engine's loader
    holds its weights' and scratch buffers."""

    def __init__(self, nbytes):
        self.p = lib().madi_alloc(nbytes)
        if not self.p:
            raise MemoryError("madi_alloc(%d)" % nbytes)

    def __del__(self):
        if getattr(self, "p", None):
            lib().madi_free(self.p)


class Source:
    """Everything drawn from one seed, in one order."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def weight(self, n, k):
        """Natural Q8 rows: int8 [n][k], fp16 [n][k/32]."""
        qs = torch.randint(-127, 128, (n, k), dtype=torch.int8, device="cuda", generator=self.g)
        sc = torch.rand((n, k // 32), device="cuda", generator=self.g) * 6e-4 + 2e-4
        return qs, sc.half()

    def normal(self, *shape, scale=1.0):
        return torch.randn(shape, device="cuda", generator=self.g) * scale

    def bias(self, n):
        return self.normal(n, scale=0.1)


def _load(w):
    return q8.upload_q8_device_repack(w[0].cpu().numpy(), w[1].cpu().numpy())


def _load_alloc(w):
    return q8.upload_q8_alloc(w[0].cpu().numpy(), w[1].cpu().numpy())


def _f32(*shape):
    return torch.empty(shape, dtype=torch.float32, device="cuda")


def _f16(*shape):
    return torch.empty(shape, dtype=torch.float16, device="cuda")


#: One decoder layer's projections, (n, k): self q|k|v, self out, cross q,
#: cross out, FFN up, FFN down.
DEC_SHAPES = ((3 * D, D), (D, D), (D, D), (D, D), (MLP, D), (D, MLP))


def _token_inputs(case, seed):
    s = Source(seed)
    emb = s.weight(VOCAB, D)
    layers = []
    for _ in range(case["layers"]):
        w = [s.weight(n, k) for n, k in DEC_SHAPES]
        b = [s.bias(n) for n, _ in DEC_SHAPES]
        # what the attention between the projections hands on
        mid = [s.normal(D) for _ in range(2)]
        caches = [s.normal(CACHE_ROWS, D) for _ in range(2)]
        layers.append((w, b, mid, caches))
    tok = torch.randint(0, VOCAB, (1,), dtype=torch.int32, device="cuda", generator=s.g)
    return emb, layers, tok


def _rows_inputs(case, seed):
    s = Source(seed)
    w = [s.weight(n, k) for n, k in DEC_SHAPES]
    return w, s.normal(case["m"], D), s.normal(case["m"], MLP)


def _encoder_inputs(case, seed):
    s = Source(seed)
    w = [s.weight(3 * D, D), s.weight(D, D), s.weight(MLP, D), s.weight(D, MLP)]
    b = [s.bias(3 * D), None, s.bias(MLP), None]
    return w, b, s.normal(case["seq"], D).half()


def _attention_inputs(case, seed):
    s = Source(seed)
    return [s.normal(case["seq"], case["heads"] * 64, scale=c).half() for c in (1.4, 1.4, 1.0)]


def _mlp_inputs(case, seed):
    s = Source(seed)
    return s.weight(MLP, D), s.weight(D, MLP), s.bias(MLP), s.bias(D), s.normal(case["m"], D).half()


#: The F16-cache layer: q, k, v and out, fc1, fc2 as [k][n] weights.
F16_SHAPES = ((D, D), (D, D), (D, D), (D, D), (MLP, D), (D, MLP))


def _f16_inputs(case, seed):
    s = Source(seed)
    w = [(s.normal(k, n) * 0.04).half() for n, k in F16_SHAPES]
    b = [s.bias(n) for n, _ in F16_SHAPES]
    return w, b, s.normal(case["m"], D).half(), s.normal(case["m"], MLP).half()


def prepare(case, seed):
    q8.init()
    kind = case["kind"]
    st = {"case": case}
    if kind == "gemv":
        s = Source(seed)
        w, x, b = s.weight(case["n"], case["k"]), s.normal(case["k"]), s.bias(case["n"])
        st.update(w=_load(w), x=x, b=b, out=_f32(case["n"]))
    elif kind == "token":
        emb, layers, tok = _token_inputs(case, seed)
        st.update(emb=_load(emb), tok=tok, x=_f32(D), h=_f32(MLP), logits=_f32(VOCAB),
                  pos=torch.tensor([case["pos"]], dtype=torch.int32, device="cuda"),
                  gelu=q8.getFunction("gemv_q8_bias_gelu"), res=q8.getFunction("gemv_q8_bias_res"))
        st["layers"] = [dict(w=[_load(x) for x in w], b=b, vb=b[0][2 * D:].clone(), mid=mid, kc=c[0],
                             vc=c[1], q=_f32(D), cq=_f32(D)) for w, b, mid, c in layers]
    elif kind == "logits":
        s = Source(seed)
        w, x = s.weight(case["vocab"], D), s.normal(D)
        st.update(w=_load(w), x=x, out=_f32(case["vocab"]))
    elif kind == "rows":
        w, x, h = _rows_inputs(case, seed)
        st.update(w=[_load(v) for v in w], x=x, h=h, out=[_f32(case["m"], n) for n, _ in DEC_SHAPES])
    elif kind == "batched_logits":
        s = Source(seed)
        w, x = s.weight(case["vocab"], D), s.normal(case["m"], D).half()
        # the F16 copy the engine makes once per decode (recorded, not written)
        st.update(w16=DeviceBuffer(2 * case["vocab"] * D), w=_load_alloc(w), x=x,
                  out=_f16(case["m"], case["vocab"]))
        q8.deqW16(st["w16"].p, st["w"], case["vocab"], D)
    elif kind == "encoder":
        w, b, x = _encoder_inputs(case, seed)
        m = case["seq"]
        st.update(wdq=DeviceBuffer(2 * MLP * D), w=[_load_alloc(v) for v in w], x=x,
                  b=[b[0][:D].clone(), b[0][D:2 * D].clone(), b[0][2 * D:].clone(), b[2]],
                  q=_f16(m, D), k=_f16(m, D), v=_f16(m, D), a=_f16(m, D), o=_f16(m, D), h=_f16(m, MLP),
                  y=_f16(m, D), m4=q8.getFunction("m4_gemm_nn"), m4b=q8.getFunction("m4_gemm_bias"),
                  m4g=q8.getFunction("m4_gemm_bias_gelu"), flash=q8.getFunction("m4_flash_enc"))
    elif kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        st.update(q=q, k=k, v=v, out=torch.empty_like(q), flash=q8.getFunction("m4_flash_enc"))
    elif kind == "mlp":
        w1, w2, b1, b2, x = _mlp_inputs(case, seed)
        st.update(w1=_load(w1), w2=_load(w2), b1=b1, b2=b2, x=x, h=_f16(case["m"], MLP), y=_f16(case["m"], D))
    elif kind == "f16_layer":
        w, b, x, h = _f16_inputs(case, seed)
        st.update(w=w, b=b, x=x, h=h, out=[_f16(case["m"], n) for n, _ in F16_SHAPES],
                  m4=q8.getFunction("m4_gemm_nn"), m4b=q8.getFunction("m4_gemm_bias"),
                  m4g=q8.getFunction("m4_gemm_bias_gelu"))
    elif kind == "quantize":
        st.update(w=(Source(seed).normal(case["n"], case["k"]) * 0.04).half())
    else:
        raise ValueError(kind)
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "gemv":
        q8.kGemvQ8Bias(st["out"], st["x"], st["w"], st["b"], case["n"], case["k"])
        return st["out"]
    if kind == "token":
        x, h, emb = st["x"], st["h"], st["emb"]
        q8.embLookup(x, emb.qs, emb.scales, st["tok"])
        for y in st["layers"]:
            w, b = y["w"], y["b"]
            q8.kQkv(y["q"], x, w[0], b[0], y["vb"], y["kc"], y["vc"], st["pos"])
            q8.kGemvQ8BiasEpi(st["res"], x, y["mid"][0], w[1], b[1], D, D)
            q8.kGemvQ8Bias(y["cq"], x, w[2], b[2], D, D)
            q8.kGemvQ8BiasEpi(st["res"], x, y["mid"][1], w[3], b[3], D, D)
            q8.kGemvQ8BiasEpi(st["gelu"], h, x, w[4], b[4], MLP, D)
            q8.kGemvQ8BiasEpi(st["res"], x, h, w[5], b[5], D, MLP)
        q8.kLogitGemv(st["logits"], emb.qs, emb.scales, x)
        return {"logits": st["logits"], "x": x,
                "layers": [{n: y[n] for n in ("q", "kc", "vc", "cq")} for y in st["layers"]]}
    if kind == "logits":
        q8.kLogitGemv(st["out"], st["w"].qs, st["w"].scales, st["x"], case["vocab"])
        return st["out"]
    if kind == "rows":
        for w, out, (n, k) in zip(st["w"], st["out"], DEC_SHAPES):
            q8.pproj(st["h"] if k == MLP else st["x"], w, out, case["m"], n, k)
        return st["out"]
    if kind == "batched_logits":
        q8.matmulF16Batched(st["x"], st["w16"].p, st["out"], case["m"], case["vocab"], D)
        return st["out"]
    if kind == "encoder":
        m, wdq, b = case["seq"], st["wdq"].p, st["b"]
        qkv, wo, w1, w2 = st["w"]
        for i, c in enumerate("qkv"):
            q8.kDeq(wdq, qkv.rows(i * D, D), D, D)
            q8.kM4Bias(st["m4b"], st["x"], wdq, st[c], b[i], m, D, D)
        q8.kFlash(st["flash"], st["a"], st["q"], st["k"], st["v"], m)
        q8.kDeq(wdq, wo, D, D)
        q8.kM4(st["m4"], st["a"], wdq, st["o"], m, D, D)
        q8.kDeq(wdq, w1, MLP, D)
        q8.kM4Bias(st["m4g"], st["o"], wdq, st["h"], b[3], m, MLP, D)
        q8.kDeq(wdq, w2, D, MLP)
        q8.kM4(st["m4"], st["h"], wdq, st["y"], m, D, MLP)
        return {c: st[c] for c in "qkvaohy"}
    if kind == "attention":
        q8.kFlash(st["flash"], st["out"], st["q"], st["k"], st["v"], case["seq"], case["heads"])
        return st["out"]
    if kind == "mlp":
        q8.kGemmQ8Bias(st["x"], st["w1"], st["h"], st["b1"], case["m"], MLP, D, gelu=True)
        q8.kGemmQ8Bias(st["h"], st["w2"], st["y"], st["b2"], case["m"], D, MLP)
        return st["h"], st["y"]
    if kind == "f16_layer":
        for i, (n, k) in enumerate(F16_SHAPES):
            a = st["h"] if k == MLP else st["x"]
            if i in (3, 5):
                q8.kM4(st["m4"], a, st["w"][i], st["out"][i], case["m"], n, k)
            else:
                q8.kM4Bias(st["m4g" if i == 4 else "m4b"], a, st["w"][i], st["out"][i], st["b"][i],
                           case["m"], n, k)
        return st["out"]
    w = q8.quantize(st["w"], case["n"], case["k"])
    return list(w._keep)


# ---------------------------------------------------------------- what it cannot do without
def _gemm(m, n, k, wbytes, abytes, cbytes):
    return m * k * abytes + n * k * wbytes + m * n * cbytes, 2 * m * n * k


Q8B = 1 + 2 / 32  # bytes of one Q8 weight


def work(case):
    kind = case["kind"]
    if kind == "gemv":
        parts = [_gemm(1, case["n"], case["k"], Q8B, 4, 4), (4 * case["n"], 0)]
    elif kind == "token":
        parts = [_gemm(1, n, k, Q8B, 4, 4) for n, k in DEC_SHAPES] * case["layers"]
        parts.append(_gemm(1, VOCAB, D, Q8B, 4, 4))
    elif kind == "logits":
        parts = [_gemm(1, case["vocab"], D, Q8B, 4, 4)]
    elif kind == "rows":
        parts = [_gemm(case["m"], n, k, Q8B, 4, 4) for n, k in DEC_SHAPES]
    elif kind == "batched_logits":
        parts = [_gemm(case["m"], case["vocab"], D, Q8B, 2, 2)]
    elif kind == "encoder":
        m = case["seq"]
        parts = [_gemm(m, n, k, Q8B, 2, 2) for n, k in ((3 * D, D), (D, D), (MLP, D), (D, MLP))]
        parts.append((4 * m * D * 2, 4 * m * m * D))
    elif kind == "attention":
        d = case["heads"] * 64
        parts = [(4 * case["seq"] * d * 2, 4 * case["seq"] ** 2 * d)]
    elif kind == "mlp":
        parts = [_gemm(case["m"], n, k, Q8B, 2, 2) for n, k in ((MLP, D), (D, MLP))]
    elif kind == "f16_layer":
        parts = [_gemm(case["m"], n, k, 2, 2, 2) for n, k in F16_SHAPES]
    else:
        # per weight: a maximum and a scale, a rounding and a clamp
        parts = [(case["n"] * case["k"] * (2 + Q8B), 4 * case["n"] * case["k"])]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


def tolerance(case):
    return TOLERANCE[case["kind"]]


TOLERANCE = {
    "gemv": {"rel": 2e-6}, "logits": {"rel": 2e-6}, "rows": {"rel": 2e-6}, "token": {"rel": 1e-5},
    "batched_logits": {"rel": 1e-3}, "encoder": {"rel": 2.5e-3}, "attention": {"rel": 1e-3},
    "mlp": {"rel": 1e-3}, "f16_layer": {"rel": 1e-3}, "quantize": "exact",
}


# ---------------------------------------------------------------- in 64 bits
def _deq(w):
    """The Q8 weight's value, q * s."""
    return w[0].double() * w[1].double().repeat_interleave(32, dim=1)


def _deq16(w):
    """The F16 weight that the engine's dequantisation defines: q * s rounded once to fp16."""
    return _deq(w).half().double()


def _gelu(x):
    return 0.5 * x * (1 + torch.erf(x * math.sqrt(0.5)))


def _attention(q, k, v, heads):
    seq = q.shape[0]
    q, k, v = (t.view(seq, heads, 64) for t in (q, k, v))
    out = torch.empty_like(q)
    for i in range(heads):
        out[:, i] = torch.softmax(q[:, i] @ k[:, i].t().contiguous() / 8, dim=1) @ v[:, i]
    return out.reshape(seq, heads * 64)


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemv":
        s = Source(seed)
        w, x, b = s.weight(case["n"], case["k"]), s.normal(case["k"]), s.bias(case["n"])
        return _deq(w) @ x.double() + b.double()
    if kind == "token":
        emb, layers, tok = _token_inputs(case, seed)
        x = _deq((emb[0][tok], emb[1][tok]))[0]
        outs = []
        for w, b, mid, (kc, vc) in layers:
            b, mid = [t.double() for t in b], [t.double() for t in mid]
            qkv = _deq(w[0]) @ x
            kc, vc = kc.double(), vc.double()
            kc[case["pos"]] = qkv[D:2 * D]
            vc[case["pos"]] = qkv[2 * D:] + b[0][2 * D:]
            y = dict(q=qkv[:D] + b[0][:D], kc=kc, vc=vc)
            x = x + _deq(w[1]) @ mid[0] + b[1]
            y["cq"] = _deq(w[2]) @ x + b[2]
            x = x + _deq(w[3]) @ mid[1] + b[3]
            x = x + _deq(w[5]) @ _gelu(_deq(w[4]) @ x + b[4]) + b[5]
            outs.append(y)
        return {"logits": _deq(emb) @ x, "x": x, "layers": outs}
    if kind == "logits":
        s = Source(seed)
        w, x = s.weight(case["vocab"], D), s.normal(D)
        return _deq(w) @ x.double()
    if kind == "rows":
        # the operator rounds its rows to fp16 and multiplies by the F16 weight
        w, x, h = _rows_inputs(case, seed)
        x, h = x.half().double(), h.half().double()
        return [(h if k == MLP else x) @ _deq16(v).t() for v, (n, k) in zip(w, DEC_SHAPES)]
    if kind == "batched_logits":
        s = Source(seed)
        w, x = s.weight(case["vocab"], D), s.normal(case["m"], D).half()
        return x.double() @ _deq16(w).t()
    if kind == "encoder":
        w, b, x = _encoder_inputs(case, seed)
        qkv = x.double() @ _deq16(w[0]).t() + b[0].double()
        y = {c: qkv[:, i * D:(i + 1) * D].contiguous() for i, c in enumerate("qkv")}
        y["a"] = _attention(y["q"], y["k"], y["v"], q8.NH)
        y["o"] = y["a"] @ _deq16(w[1]).t()
        y["h"] = _gelu(y["o"] @ _deq16(w[2]).t() + b[2].double())
        y["y"] = y["h"] @ _deq16(w[3]).t()
        return y
    if kind == "attention":
        return _attention(*(t.double() for t in _attention_inputs(case, seed)), case["heads"])
    if kind == "mlp":
        w1, w2, b1, b2, x = _mlp_inputs(case, seed)
        h = _gelu(x.double() @ _deq16(w1).t() + b1.double())
        return h, h @ _deq16(w2).t() + b2.double()
    if kind == "f16_layer":
        w, b, x, h = _f16_inputs(case, seed)
        x, h = x.double(), h.double()
        out = [(h if k == MLP else x) @ w[i].double() for i, (n, k) in enumerate(F16_SHAPES)]
        out = [y if i in (3, 5) else y + b[i].double() for i, y in enumerate(out)]
        out[4] = _gelu(out[4])
        return out
    return None  # quantised bytes: compared exactly
