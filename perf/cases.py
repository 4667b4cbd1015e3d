"""Cases whose speed is watched: the work a program has the quantized-linear path do.

A case is a dict of plain values.  `prepare(case, seed)` makes the inputs on the GPU and
what a program keeps between calls (weights, output buffers, built chains, captured
decode graphs); `run(state)` is one pass through the public entry points; `exact` is the
same result in 64 bits from plain torch; `work` the bytes and operations a pass cannot
do without; `tolerance` what another correct implementation may differ by.

Kinds of case:

* call     one eager engine-signature linear (gemm_i8 / gemm_w4), with or without a
           residual, any M and N (ragged N included);
* head     the vocabulary head with the final norm in its launch (pro_gemm_i8);
* decode   the engine's linears and producers of consecutive layers, 1-8 rows, as one
           engine chain per layer body or as a HIP graph of fused calls;
* prefill  one layer's producers and linears over a chunk of rows, as eager calls;
* a16      one fp16-activation linear (linear_w8 / linear_w4), decode to prefill rows;
* chain16  dependent fp16-activation linears of consecutive layers in one launch;
* requant  a loader turning float weights into the W8 and W4 layouts;
* repack   a loader turning GPTQ / AWQ / compressed-tensors int4 into the W4 layout.
"""
from __future__ import annotations

import importlib
import importlib.util
import pathlib
import sys

import torch

ALIAS = "qwen35_amd"
ROOT = pathlib.Path(__file__).resolve().parent.parent
EPS = 1e-6
HEAD_DIM = 256


def _kernels(name):
    """The package's kernels.<name>; its directory is no Python identifier, so it is
    loaded under an alias."""
    if ALIAS not in sys.modules:
        pkg = ROOT / "qwen_3.5_comfy_prompt_enhancer_amd"
        spec = importlib.util.spec_from_file_location(ALIAS, pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[ALIAS] = mod
        spec.loader.exec_module(mod)
    return importlib.import_module(f"{ALIAS}.kernels.{name}")


# ------------------------------------------------------------------ the cases

def listed():
    return [
        # the smallest call: a decode step's attention output projection, eager, one row
        dict(name="call-w8-m1", kind="call", wt="w8", group=0, zeros=False, M=1, K=2048, N=2048, residual=True),
        # a vocabulary extended by added tokens, so that N is odd: two candidates' logits
        dict(name="call-w8-ragged-m2", kind="call", wt="w8", group=0, zeros=False, M=2, K=2048, N=50021,
             residual=False),
        # the logits of four candidates, vocabulary 248320, with the final norm
        dict(name="head-w8-m4", kind="head", wt="w8", group=0, zeros=False, M=4, K=2048, N=248320),
        # token generation, INT8 model, one sequence: layer bodies as engine chains
        dict(name="decode-w8-m1", kind="decode", wt="w8", group=0, zeros=False, M=1, hidden=2048, inter=6144,
             layers=6, form="chain"),
        # token generation, W4 checkpoint with zeros, four candidates: a graph of fused calls
        dict(name="decode-w4-m4", kind="decode", wt="w4", group=128, zeros=True, M=4, hidden=2048, inter=6144,
             layers=6, form="fused"),
        # a full prefill chunk of the INT8 model, one layer
        dict(name="prefill-w8-m512", kind="prefill", wt="w8", group=0, zeros=False, M=512, hidden=2048,
             inter=6144),
        # a short prompt through one layer of a W4 model of the 9B class
        dict(name="prefill-w4-9b-m137", kind="prefill", wt="w4", group=128, zeros=False, M=137, hidden=4096,
             inter=12288),
        # a decode step of a W4 9B-class model on fp16 activations, four rows, one launch
        dict(name="chain16-w4-9b-m4", kind="chain16", wt="w4", group=128, zeros=False, M=4, hidden=4096,
             inter=12288, layers=3),
        # prefill on fp16 activations, the largest chunk
        dict(name="a16-w8-m2048", kind="a16", wt="w8", group=0, zeros=False, M=2048, K=2048, N=6144),
        # prefill on fp16 activations, a short prompt, W4
        dict(name="a16-w4-m128", kind="a16", wt="w4", group=128, zeros=False, M=128, K=6144, N=2048),
        # loading float weights: INT8 per column and symmetric int4 in groups of 32
        dict(name="requant-4096x12288", kind="requant", K=4096, N=12288, group=32),
        # loading external int4 checkpoints
        dict(name="repack-4096x12288", kind="repack", K=4096, N=12288, group=128),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def _weights_of(rng, w4_zeros=True):
    if rng.random() < 0.5:
        return dict(wt="w8", group=0, zeros=False)
    return dict(wt="w4", group=rng.choice([64, 128]), zeros=bool(w4_zeros and rng.random() < 0.4))


def draw(rng):
    kind = rng.choice(["call", "call", "decode", "decode", "prefill", "prefill", "a16", "a16", "head", "chain16",
                       "requant", "repack"])
    if kind == "call":
        c = dict(kind=kind, **_weights_of(rng), M=_log(rng, 1, 512), K=64 * _log(rng, 4, 128))
        if c["wt"] == "w4":
            c["K"] = -(-c["K"] // c["group"]) * c["group"]
        n = _log(rng, 256, 65536)
        if rng.random() < 0.7:
            n = -(-n // 16) * 16                                      # the engine's layouts
            n = max(16, min(n, 25_000_000_000 // (c["M"] * c["K"]) // 16 * 16))
        else:
            n = min(n, 4_000_000_000 // (c["M"] * c["K"])) | 1         # ragged
        return dict(c, N=n, residual=rng.random() < 0.5)
    if kind == "head":
        return dict(kind=kind, **_weights_of(rng), M=rng.randint(1, 8), K=rng.choice([1024, 2048]),
                    N=16 * _log(rng, 2000, 15520))
    if kind == "decode":
        h = rng.choice([1024, 2048, 2560, 4096])
        return dict(kind=kind, **_weights_of(rng), M=rng.randint(1, 8), hidden=h, inter=128 * _log(rng, h // 64, h // 40),
                    layers=max(1, min(rng.randint(2, 6), 400_000_000 // (15 * h * h))), form=rng.choice(["chain", "fused"]))
    if kind == "prefill":
        h = rng.choice([1024, 2048, 2560, 4096])
        f = 128 * _log(rng, h // 64, h // 40)
        most = min(700, 64_000_000_000 // (2 * (5 * h * h + 3 * h * f)))
        return dict(kind=kind, **_weights_of(rng), M=_log(rng, 9, most), hidden=h, inter=f)
    if kind == "a16":
        w = _weights_of(rng)
        m, k = _log(rng, 1, 2048), 128 * _log(rng, 8, 96)
        n = 16 * _log(rng, 32, 768)
        return dict(kind=kind, **dict(w, group=128 if w["wt"] == "w4" else 0), M=m, K=k,
                    N=max(512, min(n, 25_000_000_000 // (m * k) // 16 * 16)))
    if kind == "chain16":
        w = _weights_of(rng)
        h = rng.choice([1024, 2048, 4096])
        return dict(kind=kind, **dict(w, group=128 if w["wt"] == "w4" else 0), M=rng.randint(1, 8), hidden=h,
                    inter=3 * h, layers=max(1, min(rng.randint(1, 4), 400_000_000 // (12 * h * h))))
    return dict(kind=kind, K=128 * _log(rng, 4, 48), N=64 * _log(rng, 8, 192), group=rng.choice([32, 64]) if
                kind == "requant" else 128)


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(gen, *shape, dtype=torch.float32, std=1.0):
    return (torch.randn(*shape, generator=gen, device="cuda") * std).to(dtype)


def _linear(gen, case, K, N, sdt=None):
    """(w, scale, zero) of one [K, N] weight in the engine layout: normal codes, scales
    that keep a unit-variance input at about unit variance."""
    spread = 0.5 + torch.rand(N, generator=gen, device="cuda")
    if case["wt"] == "w8":
        w = _normal(gen, K, N, std=32.0).round_().clamp_(-127, 127).to(torch.int8)
        return w, (spread / (32.0 * K ** 0.5)).to(sdt or torch.float32), None
    G = K // case["group"]
    lo, hi = (_normal(gen, K // 2, N, std=2.5).round_().add_(8).clamp_(0, 15).to(torch.uint8) for _ in range(2))
    s = (0.75 + 0.5 * torch.rand(G, N, generator=gen, device="cuda")) * spread / (2.5 * K ** 0.5)
    z = torch.randint(6, 11, (G, N), generator=gen, device="cuda", dtype=torch.uint8) if case["zeros"] else None
    return lo | (hi << 4), s.to(sdt or torch.bfloat16), z


def _codes(gen, M, K):
    """int8 codes and per-64 scales of normal activations, as the producers make them."""
    x = _normal(gen, M, K // 64, 64)
    s = (x.abs().amax(-1) / 127).clamp_min(1e-8)
    q = x / s[..., None]
    q = torch.where(q >= 0, (q + 0.5).floor(), (q - 0.5).ceil()).clamp_(-127, 127)
    return q.to(torch.int8).reshape(M, K).contiguous(), s.contiguous()


def _out(M, N, dtype=torch.bfloat16):
    return torch.empty(M, N, dtype=dtype, device="cuda")


def _inputs(case, seed):
    """The tensors of a case that its seed determines (no library code)."""
    gen, kind = _gen(seed), case["kind"]
    s = dict(case=case)
    if kind == "call":
        s["a"] = _codes(gen, case["M"], case["K"])
        s["w"] = _linear(gen, case, case["K"], case["N"])
        s["res"] = _normal(gen, case["M"], case["N"], dtype=torch.bfloat16) if case["residual"] else None
    elif kind == "head":
        s["x"] = _normal(gen, case["M"], case["K"], dtype=torch.bfloat16, std=2.0)
        s["norm"] = _normal(gen, case["K"], dtype=torch.bfloat16, std=0.1)
        s["w"] = _linear(gen, case, case["K"], case["N"])
    elif kind in ("decode", "prefill"):
        M, h, f = case["M"], case["hidden"], case["inter"]
        s["layers"] = []
        for _ in range(case.get("layers", 1)):
            s["layers"].append(dict(
                x=_normal(gen, M, h, dtype=torch.bfloat16, std=2.0), gate=_normal(gen, M, 4 * h, dtype=torch.bfloat16),
                aout=_normal(gen, M, h, dtype=torch.bfloat16), post=_normal(gen, h, dtype=torch.bfloat16, std=0.1),
                inn=_normal(gen, h, dtype=torch.bfloat16, std=0.1), o=_linear(gen, case, h, h),
                g=_linear(gen, case, h, f), u=_linear(gen, case, h, f), d=_linear(gen, case, f, h),
                qkv=_linear(gen, case, h, 3 * h), z=_linear(gen, case, h, h)))
    elif kind == "a16":
        s["x"] = _normal(gen, case["M"], case["K"], dtype=torch.float16)
        s["w"] = _linear(gen, case, case["K"], case["N"], torch.float16)
    elif kind == "chain16":
        M, h, f = case["M"], case["hidden"], case["inter"]
        s["x"] = _normal(gen, M, h, dtype=torch.float16)
        s["layers"] = [{n: _linear(gen, case, k, m, torch.float16) for n, k, m in
                        (("q", h, h), ("k", h, h // 4), ("v", h, h // 4), ("o", h, h), ("g", h, f), ("u", h, f),
                         ("d", f, h))} for _ in range(case["layers"])]
    elif kind == "requant":
        s["w"] = _normal(gen, case["K"], case["N"], std=0.02)
    else:
        K, N, G = case["K"], case["N"], case["K"] // case["group"]

        def words(*shape):
            return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, generator=gen, device="cuda", dtype=torch.int32)
        s.update(gptq=words(K // 8, N), gptq_z=words(G, N // 8), awq=words(K, N // 8), awq_z=words(G, N // 8),
                 ct=words(N, K // 8), ct_s=_normal(gen, N, G, dtype=torch.bfloat16, std=0.01))
    return s


# ------------------------------------------------------------------ what a program keeps

def prepare(case, seed):
    s = _inputs(case, seed)
    kind, M = case["kind"], case.get("M")
    if kind == "call":
        s["out"] = _out(M, case["N"])
    elif kind == "head":
        s["pro"] = _kernels("fused").Producer.rmsnorm(s["x"], s["norm"], EPS)
        s["out"] = _out(M, case["N"])
    elif kind == "decode":
        _buffers(s)
        (_decode_chain if case["form"] == "chain" else _decode_graph)(s)
    elif kind == "prefill":
        _buffers(s)
    elif kind == "a16":
        s["out"] = _out(M, case["N"], torch.float16)
    elif kind == "chain16":
        s["chain"] = ch = _kernels("chain").DecodeChain(M)
        x, lvl, s["outs"] = s["x"], 0, []
        for L in s["layers"]:
            y = {n: _out(M, w[0].shape[1], torch.float16) for n, w in L.items()}
            for n, a, d in (("q", x, 0), ("k", x, 0), ("v", x, 0), ("o", y["q"], 1), ("g", y["o"], 2), ("u", y["o"], 2),
                            ("d", y["u"], 3)):
                ch.add(a, L[n][0], L[n][1], y[n], zero=L[n][2], residual=x if n == "d" else None, level=lvl + d)
            x, lvl = y["d"], lvl + 4
            s["outs"].append(y)
        ch.build()
    return s


def _buffers(s):
    """Each layer's outputs.  A layer body reads the hidden state, the attention output and
    the gates that the mixer before it left (inputs here: the mixer is not part of this
    path) and writes buffers of its own, so a pass can be made again from the same state."""
    c = s["case"]
    M, h, f = c["M"], c["hidden"], c["inter"]
    for L in s["layers"]:
        L["out"] = dict(h1=_out(M, h), h2=_out(M, h), proj=_out(M, 4 * h), fq=_out(M, f, torch.int8),
                        fs=_out(M, f // 64, torch.float32))
        if c["kind"] == "prefill":
            L["out"].update(xq=_out(M, h, torch.int8), xs=_out(M, h // 64, torch.float32))


def _decode_chain(s):
    """One engine chain per layer body, from the attention's output to the next layer's
    projections."""
    echain, P = _kernels("echain"), _kernels("fused").Producer
    s["chains"] = []
    for L in s["layers"]:
        o = L["out"]
        ch = echain.EngineChain(s["case"]["M"])
        ch.gemm_i8(None, None, L["o"][0], L["o"][1], o["h1"], residual=L["x"], b_z=L["o"][2],
                   pro=P.gate_mul(L["aout"], L["gate"], hd=HEAD_DIM), level=0)
        ch.mlp_gate_up_quant(None, None, L["g"][0], L["g"][1], L["u"][0], L["u"][1], o["fq"], o["fs"], zg=L["g"][2],
                             zu=L["u"][2], pro=P.rmsnorm(o["h1"], L["post"], EPS), level=1)
        ch.gemm_i8(o["fq"], o["fs"], L["d"][0], L["d"][1], o["h2"], residual=o["h1"], b_z=L["d"][2], level=2)
        ch.proj3(None, None, L["qkv"][0], L["qkv"][1], L["z"][0], L["z"][1], None, None, o["proj"], z1=L["qkv"][2],
                 z2=L["z"][2], pro=P.rmsnorm(o["h2"], L["inn"], EPS), level=3)
        s["chains"].append(ch.build())


def _decode_graph(s):
    """The same layer bodies as fused calls, captured once."""
    F = _kernels("fused")
    gemm = _kernels("gemm")

    def step():
        for L in s["layers"]:
            o = L["out"]
            F.pro_gemm_i8(F.Producer.gate_mul(L["aout"], L["gate"], hd=HEAD_DIM), L["o"][0], L["o"][1], o["h1"],
                          residual=L["x"], b_z=L["o"][2])
            F.pro_mlp_gate_up_quant(F.Producer.rmsnorm(o["h1"], L["post"], EPS), L["g"][0], L["g"][1], L["u"][0],
                                    L["u"][1], o["fq"], o["fs"], zg=L["g"][2], zu=L["u"][2])
            gemm.gemm_i8(o["fq"], o["fs"], L["d"][0], L["d"][1], o["h2"], residual=o["h1"], b_z=L["d"][2])
            F.pro_proj3(F.Producer.rmsnorm(o["h2"], L["inn"], EPS), L["qkv"][0], L["qkv"][1], L["z"][0], L["z"][1], None,
                        None, o["proj"], z1=L["qkv"][2], z2=L["z"][2])

    step()
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with _kernels("qlin").capture(s["graph"]):
        step()


# ------------------------------------------------------------------ one pass

def run(s):
    c = s["case"]
    kind = c["kind"]
    if kind == "call":
        w, ws, wz = s["w"]
        return _kernels("gemm").gemm_i8(*s["a"], w, ws, s["out"], residual=s["res"], b_z=wz)
    if kind == "head":
        w, ws, wz = s["w"]
        return _kernels("fused").pro_gemm_i8(s["pro"], w, ws, s["out"], b_z=wz)
    if kind == "decode":
        if c["form"] == "chain":
            for ch in s["chains"]:
                ch.run()
        else:
            s["graph"].replay()
        return [L["out"] for L in s["layers"]]
    if kind == "prefill":
        return _prefill(s)
    if kind == "a16":
        w, ws, wz = s["w"]
        lin = _kernels("linear")
        if c["wt"] == "w8":
            return lin.linear_w8(s["x"], w, ws, s["out"])
        return lin.linear_w4(s["x"], w, ws, s["out"], w_zero=wz)
    if kind == "chain16":
        s["chain"].run()
        return s["outs"]
    lay = _kernels("layout")
    if kind == "requant":
        return lay.requant_w8_row(s["w"]), lay.requant_w4_sym(s["w"], c["group"])
    return (lay.gptq_w4_to_engine(s["gptq"]), lay.gptq_zeros(s["gptq_z"]), lay.awq_w4_to_engine(s["awq"]),
            lay.awq_zeros(s["awq_z"]), lay.ct_w4_to_engine(s["ct"], c["K"], s["ct_s"]))


def _prefill(s):
    """A layer's calls over a chunk: in-norm and projections, gated attention output and
    its projection, post-norm and the MLP."""
    gemm, norm = _kernels("gemm"), _kernels("norm")
    L = s["layers"][0]
    o = L["out"]
    norm.rmsnorm_quant(L["x"], L["inn"], o["xq"], o["xs"], EPS)
    gemm.proj3(o["xq"], o["xs"], L["qkv"][0], L["qkv"][1], L["z"][0], L["z"][1], None, None, o["proj"], z1=L["qkv"][2],
               z2=L["z"][2])
    norm.gate_mul_quant(L["aout"], o["proj"], o["xq"], o["xs"], HEAD_DIM)
    gemm.gemm_i8(o["xq"], o["xs"], L["o"][0], L["o"][1], o["h1"], residual=L["x"], b_z=L["o"][2])
    norm.rmsnorm_quant(o["h1"], L["post"], o["xq"], o["xs"], EPS)
    gemm.mlp_gate_up_quant(o["xq"], o["xs"], L["g"][0], L["g"][1], L["u"][0], L["u"][1], o["fq"], o["fs"], zg=L["g"][2],
                           zu=L["u"][2])
    gemm.gemm_i8(o["fq"], o["fs"], L["d"][0], L["d"][1], o["h2"], residual=o["h1"], b_z=L["d"][2])
    return o


# ------------------------------------------------------------------ the same in 64 bits

def _dequant(wsz):
    w, s, z = wsz
    if w.dtype == torch.int8:
        return w.double() * s.double()
    K = 2 * w.shape[0]
    n = torch.empty(K, w.shape[1], dtype=torch.float64, device=w.device)
    n[0::2], n[1::2] = (w & 15).double(), (w >> 4).double()
    g = K // s.shape[0]
    n -= z.double().repeat_interleave(g, 0) if z is not None else 8.0
    return n.mul_(s.double().repeat_interleave(g, 0))


def _values(qs):
    q, s = qs
    return q.double() * s.double().repeat_interleave(64, 1)


def _quant(y):
    """Per-64 int8 codes (round half away from zero) and scales, the path's own format."""
    M, K = y.shape
    y = y.reshape(M, K // 64, 64)
    s = (y.abs().amax(-1) / 127).clamp_min(1e-8)
    q = y / s[..., None]
    q = torch.where(q >= 0, (q + 0.5).floor(), (q - 0.5).ceil()).clamp(-127, 127)
    return q.reshape(M, K), s


def _bf(x):
    return x.to(torch.bfloat16).double()


def _rms(x, w):
    x = x.double()
    return _quant(x * (x.square().mean(-1, keepdim=True) + EPS).rsqrt() * (w.double() + 1))


def _gated(a, proj):
    M, h = a.shape
    g = proj[:, : 2 * h].reshape(M, h // HEAD_DIM, 2, HEAD_DIM)[:, :, 1].reshape(M, h)
    return _quant(a.double() * torch.sigmoid(g.double()))


def _mm(qs, wsz):
    return _values(qs) @ _dequant(wsz)


def _mlp(h1, L, o):
    g, u = _mm(_rms(h1, L["post"]), L["g"]), _mm(_rms(h1, L["post"]), L["u"])
    o["fq"], o["fs"] = _quant(_bf(torch.nn.functional.silu(g) * u))
    return _mm((o["fq"], o["fs"]), L["d"]) + h1


def exact(case, seed):
    """64-bit results; what the path stores in 16 bits or in codes between two linears is
    rounded where it is stored, since the formats are part of the result."""
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind == "call":
        y = _mm(s["a"], s["w"])
        return y + s["res"].double() if s["res"] is not None else y
    if kind == "head":
        return _mm(_rms(s["x"], s["norm"]), s["w"])
    if kind == "a16":
        return s["x"].double() @ _dequant(s["w"])
    if kind == "decode":
        outs = []
        for L in s["layers"]:
            o = {}
            h1 = _mm(_gated(L["aout"], L["gate"]), L["o"]) + L["x"].double()
            h2 = _mlp(_bf(h1), L, o)
            xn = _rms(_bf(h2), L["inn"])
            p = torch.cat([_mm(xn, L["qkv"]), _mm(xn, L["z"])], 1)
            o.update(h1=h1, h2=h2, proj=p)
            outs.append(o)
        return outs
    if kind == "prefill":
        L, o = s["layers"][0], {}
        xn = _rms(L["x"], L["inn"])
        p = torch.cat([_mm(xn, L["qkv"]), _mm(xn, L["z"])], 1)
        h1 = _mm(_gated(L["aout"], _bf(p)), L["o"]) + L["x"].double()
        o["xq"], o["xs"] = _rms(_bf(h1), L["post"])
        o.update(h1=h1, h2=_mlp(_bf(h1), L, o), proj=p)
        return o
    if kind == "chain16":
        def half(t):
            return t.to(torch.float16).double()
        x, outs = s["x"].double(), []
        for L in s["layers"]:
            y = {n: x @ _dequant(L[n]) for n in ("q", "k", "v")}
            y["o"] = half(y["q"]) @ _dequant(L["o"])
            y["g"], y["u"] = (half(y["o"]) @ _dequant(L[n]) for n in ("g", "u"))
            y["d"] = half(y["u"]) @ _dequant(L["d"]) + x
            x = half(y["d"])
            outs.append(y)
        return outs
    if kind == "requant":
        w = s["w"].double()
        s8 = (w.abs().amax(0) / 127).clamp_min(1e-8)
        s4 = (w.reshape(-1, case["group"], case["N"]).abs().amax(1) / 7).clamp_min(1e-8)
        return (None, s8), (None, s4)
    return None


# ------------------------------------------------------------------ work and tolerance

def _wbytes(case, K, N, sbytes):
    if case["wt"] == "w8":
        return K * N + N * sbytes[0]
    G = K // case["group"]
    return K * N // 2 + G * N * (sbytes[1] + (1 if case["zeros"] else 0))


def work(case):
    kind = case["kind"]
    if kind in ("requant", "repack"):
        K, N, G = case["K"], case["N"], case["K"] // case["group"]
        if kind == "requant":
            return {"bytes": 4 * K * N + K * N + 4 * N + K * N // 2 + 2 * G * N, "flops": 4 * K * N}
        return {"bytes": 3 * K * N + 2 * (G * N // 2 + G * N) + 4 * G * N, "flops": 0}
    M, eng = case["M"], (4, 2)
    if kind in ("call", "head", "a16"):
        K, N = case["K"], case["N"]
        x = M * K + M * K // 16 if kind == "call" else 2 * M * K + (2 * K if kind == "head" else 0)
        b = _wbytes(case, K, N, (2, 2) if kind == "a16" else eng) + x + 2 * M * N
        return {"bytes": b + (2 * M * N if case.get("residual") else 0), "flops": 2 * M * K * N}
    h, f, n = case["hidden"], case["inter"], case.get("layers", 1)
    if kind == "chain16":
        shapes = [(h, h)] * 2 + [(h, h // 4)] * 2 + [(h, f)] * 2 + [(f, h)]
        b = sum(_wbytes(case, k, m, (2, 2)) + 2 * M * m for k, m in shapes)
        return {"bytes": n * b + 2 * M * h, "flops": n * sum(2 * M * k * m for k, m in shapes)}
    shapes = [(h, h), (h, f), (h, f), (f, h), (h, 3 * h), (h, h)]
    b = sum(_wbytes(case, k, m, eng) for k, m in shapes) + 4 * h            # weights, the two norms' weights
    b += M * (3 * 2 * h + 2 * 2 * h + 2 * 4 * h + f + f // 16)    # x, aout, gates; h1, h2, proj, codes
    if kind == "prefill":
        b += M * (h + h // 16)
    return {"bytes": n * b, "flops": n * sum(2 * M * k * m for k, m in shapes)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("requant", "repack"):
        return "exact"                 # bytes, and scales that are one correctly rounded division
    # four times what the kernels differ by from the 64-bit result rounded to the output type
    if kind == "a16":
        return {"rel": 5e-4, "max": 5e-3}      # fp16 outputs of fp32 sums
    if kind == "chain16":
        return {"rel": 3e-3, "max": 1.6e-2}    # the same, each level reading the last one's fp16
    if kind in ("call", "head"):
        return {"rel": 2e-3, "max": 3e-2}      # a bf16 rounding that falls the other way: one ulp
    # through a layer such a rounding also moves an int8 code by one
    return {"rel": 1.1e-2, "max": 8e-2, "differ": 1e-2}
