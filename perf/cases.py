"""Performance cases of the gfx950 backend: what its users run, and over which sizes.

Each case is one pass through a public entry point (`vibe_compiler_amd.backend.Context`
or `vibe_compiler_amd.decoder_layer.DecoderLayer`) on tensors that are already on the
GPU.  The paths and their declared ranges:

layer    DecoderLayer.forward, the two configurations the repository names (hidden 4096,
         32/8 heads, FFN 14336; and 32/32 heads, FFN 11008), 1 .. 1024 tokens, BF16 or F16
prefill  attention_prefill, head_dim 128 or 64, MHA and GQA, causal or not, 33 .. 4096
         tokens, BF16 or F16
masked   attention_prefill_masked, head_dim 128 or 64: a boolean padding mask, an additive
         mask, or a sliding window; 33 .. 2048 tokens
decode   attention_decode, or attention_decode_append (one token with the KV append),
         1 .. 32 sequences over 128 .. 8192 cached tokens, MHA and GQA
gemm_i8  gemm_i8, any m and n up to 4096, k a multiple of 64, rhs [K,N] or [N,K]
gemm     gemm_mfma on BF16 / F16, any m and n up to 4096, rhs [K,N] or [N,K], output in
         the input format or F32
mlp_f32  the fp32 MLP block: two gemm_f32_mfma calls with the fused bias / GELU epilogues
formal   gemm, the per-command lane's bit-exact GEMM (F32, BF16 or F16 operands)
"""
from __future__ import annotations

import math

import torch

from vibe_compiler_amd import backend as B
from vibe_compiler_amd import decoder_layer as DL

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
FMT = {"bf16": B.BF16, "f16": B.F16, "f32": B.F32}

# hidden, q heads, kv heads, ffn of the two decoder layers the repository names
LAYERS = {"gqa14336": (4096, 32, 8, 14336), "mha11008": (4096, 32, 32, 11008)}

_context = None


def context():
    """The handle a program keeps for its whole life."""
    global _context
    if _context is None:
        _context = B.Context(0)
    return _context


def listed():
    return [
        # A whole decoder layer over a prompt of 1024 tokens: the layer benchmark.
        dict(name="layer_1024_bf16", path="layer", config="gqa14336", tokens=1024, dtype="bf16"),
        # The llama-2-7b-block case: a short prompt, where the weights are most of the traffic.
        dict(name="layer_16_f16", path="layer", config="mha11008", tokens=16, dtype="f16"),
        # The headline FA prefill.
        dict(name="prefill_2048_bf16", path="prefill", batch=1, heads=16, kv_heads=16, q_len=2048, kv_len=2048,
             head_dim=128, causal=True, dtype="bf16"),
        # GQA prefill of a prompt that no tile divides.
        dict(name="prefill_gqa_1025_f16", path="prefill", batch=1, heads=32, kv_heads=8, q_len=1025, kv_len=1025,
             head_dim=128, causal=True, dtype="f16"),
        # A padded batch with head_dim 64 and a boolean key mask (encoder attention).
        dict(name="masked_pad_1031_f16", path="masked", kind="padding", batch=4, heads=8, kv_heads=8, q_len=1031,
             kv_len=1031, head_dim=64, dtype="f16"),
        # The FD benchmark: 32 sequences over full 8192-token caches.
        dict(name="decode_32x8192_bf16", path="decode", append=False, batch=32, heads=32, kv_heads=8, kv_len=8192,
             dtype="bf16"),
        # One sequence's decode step with the KV append (the decode-kv-cache case), where latency counts.
        dict(name="decode_append_1x4095_f16", path="decode", append=True, batch=1, heads=32, kv_heads=32, kv_len=4095,
             dtype="f16"),
        # The int8 GEMM benchmark, rhs as stored [K, N].
        dict(name="i8_4096", path="gemm_i8", m=4096, k=4096, n=4096, rhs_t=False),
        # A ragged int8 projection of a few hundred rows.
        dict(name="i8_300x4096x1000", path="gemm_i8", m=300, k=4096, n=1000, rhs_t=True),
        # The 16-bit GEMM of the board timings, weight in the [N, K] orientation.
        dict(name="gemm_4096_bf16", path="gemm", m=4096, k=4096, n=4096, rhs_t=True, out="same", dtype="bf16"),
        # The fp32 MLP block of the benchmark.
        dict(name="mlp_f32_128x512x2048", path="mlp_f32", rows=128, width=512, hidden=2048),
        # One GEMM command of the per-command (bit-exact) lane.
        dict(name="formal_128x512x2048_f32", path="formal", m=128, k=512, n=2048, dtype="f32", psum=False),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    path = rng.choice(["layer", "prefill", "masked", "decode", "gemm_i8", "gemm", "mlp_f32", "formal"])
    half = rng.choice(["bf16", "f16"])
    if path == "layer":
        return dict(path=path, config=rng.choice(sorted(LAYERS)), tokens=_log(rng, 1, 1024), dtype=half)
    if path in ("prefill", "masked"):
        heads, kv_heads = rng.choice([(1, 1), (8, 8), (16, 16), (28, 28), (32, 8)])
        top = 4096 if path == "prefill" else 2048
        q_len = _log(rng, 33, top)
        case = dict(path=path, batch=rng.choice([1, 1, 2, 4]), heads=heads, kv_heads=kv_heads, q_len=q_len,
                    kv_len=q_len if rng.random() < 0.7 else _log(rng, 33, top), head_dim=rng.choice([64, 128]),
                    dtype=half)
        if path == "prefill":
            case["causal"] = case["kv_len"] == q_len and rng.random() < 0.8
        else:
            case["kind"] = rng.choice(["padding", "additive", "window"])
        # no more work than the largest listed case
        while 4 * case["head_dim"] * heads * case["batch"] * q_len * case["kv_len"] > 4e11:
            case["batch"] -= 1
        return case
    if path == "decode":
        heads, kv_heads = rng.choice([(32, 8), (32, 32), (16, 16), (8, 4)])
        case = dict(path=path, append=rng.random() < 0.5, batch=_log(rng, 1, 32), heads=heads, kv_heads=kv_heads,
                    kv_len=_log(rng, 128, 8192), dtype=half)
        case["batch"] = min(case["batch"], 32 * 8 * 8192 // (kv_heads * case["kv_len"]))
        return case
    if path == "gemm_i8":
        return dict(path=path, m=_log(rng, 1, 4096), k=64 * _log(rng, 4, 64), n=_log(rng, 64, 4096),
                    rhs_t=rng.random() < 0.5)
    if path == "gemm":
        return dict(path=path, m=_log(rng, 1, 4096), k=32 * _log(rng, 8, 128), n=_log(rng, 64, 4096),
                    rhs_t=rng.random() < 0.7, out=rng.choice(["same", "same", "f32"]), dtype=half)
    if path == "mlp_f32":
        width = 64 * _log(rng, 2, 16)
        return dict(path=path, rows=_log(rng, 1, 1024), width=width, hidden=4 * width)
    return dict(path=path, m=_log(rng, 1, 256), k=_log(rng, 32, 1024), n=_log(rng, 16, 2048),
                dtype=rng.choice(["f32", "f32", "bf16", "f16"]), psum=rng.random() < 0.3)


def _visible(case):
    """(q, kv) pairs one head of one sequence has to evaluate."""
    q, kv = case["q_len"], case["kv_len"]
    if case["path"] == "prefill":
        return sum(min(i + 1, kv) for i in range(q)) if case["causal"] else q * kv
    if case["kind"] == "window":
        return sum(max(0, min(i + 1, kv) - max(0, i + 1 - _window(case))) for i in range(q))
    if case["kind"] == "padding":
        return q * sum(_lengths(case)) / case["batch"]
    return q * kv


def _window(case):
    return max(16, case["kv_len"] // 4)


def _lengths(case):
    """Valid keys of each sequence of a padded batch."""
    return [max(1, case["kv_len"] * (case["batch"] - b) // case["batch"]) for b in range(case["batch"])]


# ------------------------------------------------------------------ inputs
def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rnd(*shape, std=1.0, dtype=None):
        return (torch.randn(*shape, generator=g, device="cuda") * std).to(DT[dtype or case["dtype"]])

    path = case["path"]
    if path == "layer":
        hidden, hq, hkv, ffn = LAYERS[case["config"]]
        w = DL.random_weights(torch, g, hidden=hidden, q_heads=hq, kv_heads=hkv, head_dim=128, ffn=ffn,
                              dtype=DT[case["dtype"]])
        for name in ("input_norm", "post_norm"):
            w[name] = (1 + 0.1 * torch.randn(hidden, generator=g, device="cuda")).to(DT[case["dtype"]])
        return dict(weights=w, x=rnd(case["tokens"], hidden))
    if path in ("prefill", "masked"):
        b, hq, hkv, s, t, d = (case[k] for k in ("batch", "heads", "kv_heads", "q_len", "kv_len", "head_dim"))
        inp = dict(q=rnd(b, hq, s, d), k=rnd(b, hkv, t, d), v=rnd(b, hkv, t, d))
        if case.get("kind") == "padding":
            n = torch.tensor(_lengths(case), device="cuda")
            inp["keep"] = (torch.arange(t, device="cuda")[None] < n[:, None]).view(b, 1, 1, t)
        elif case.get("kind") == "additive":
            inp["bias"] = torch.randn(1, 1, s, t, generator=g, device="cuda")
        return inp
    if path == "decode":
        b, hq, hkv, t = (case[k] for k in ("batch", "heads", "kv_heads", "kv_len"))
        cap = t if not case["append"] else (t + 63) // 64 * 64
        inp = dict(q=rnd(b, hq, 1, 128), k=rnd(b, hkv, cap, 128), v=rnd(b, hkv, cap, 128))
        if case["append"]:
            inp.update(k_new=rnd(b, hkv, 1, 128), v_new=rnd(b, hkv, 1, 128))
        return inp
    if path == "gemm_i8":
        m, k, n = case["m"], case["k"], case["n"]
        i8 = lambda *s: torch.randint(-127, 128, s, generator=g, device="cuda", dtype=torch.int8)  # noqa: E731
        return dict(a=i8(m, k), b=i8(n, k) if case["rhs_t"] else i8(k, n),
                    scale=torch.rand(n, generator=g, device="cuda") * 0.009 + 0.001)
    if path == "gemm":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(a=rnd(m, k), b=rnd(*((n, k) if case["rhs_t"] else (k, n)), std=0.02))
    if path == "mlp_f32":
        r, w, h = case["rows"], case["width"], case["hidden"]
        return dict(x=rnd(r, w, dtype="f32"), w1=rnd(w, h, std=w ** -0.5, dtype="f32"), b1=rnd(h, std=0.02, dtype="f32"),
                    w2=rnd(h, w, std=h ** -0.5, dtype="f32"), b2=rnd(w, std=0.02, dtype="f32"))
    m, k, n = case["m"], case["k"], case["n"]
    inp = dict(a=rnd(m, k), b=rnd(k, n, std=k ** -0.5))
    if case["psum"]:
        inp["psum"] = rnd(m, n, dtype="f32")
    return inp


def prepare(case, seed):
    st = dict(_inputs(case, seed), case=case, hip=context())
    path = case["path"]

    def empty(*shape, dtype=None):
        return torch.empty(*shape, dtype=DT[dtype or case["dtype"]], device="cuda")

    if path == "layer":
        hidden, hq, hkv, ffn = LAYERS[case["config"]]
        st["layer"] = DL.DecoderLayer(st["hip"], st.pop("weights"), case["tokens"], hidden=hidden, q_heads=hq,
                                      kv_heads=hkv, head_dim=128, ffn=ffn, dtype=DT[case["dtype"]])
        st["y"] = empty(case["tokens"], hidden)
    elif path in ("prefill", "masked", "decode"):
        st["o"] = torch.empty_like(st["q"])
    elif path == "gemm_i8":
        st["y"] = empty(case["m"], case["n"], dtype="bf16")
    elif path == "gemm":
        st["y"] = empty(case["m"], case["n"], dtype=None if case["out"] == "same" else "f32")
    elif path == "mlp_f32":
        st["h"] = empty(case["rows"], case["hidden"], dtype="f32")
        st["y"] = empty(case["rows"], case["width"], dtype="f32")
    else:
        st["y"] = empty(case["m"], case["n"])
    return st


def run(st):
    case, hip = st["case"], st["hip"]
    path = case["path"]
    if path == "layer":
        return st["layer"].forward(st["x"], st["y"])
    if path == "prefill":
        hip.attention_prefill(st["q"], st["k"], st["v"], st["o"], case["head_dim"] ** -0.5, causal=case["causal"],
                              fmt=FMT[case["dtype"]])
        return st["o"]
    if path == "masked":
        window = case["kind"] == "window"
        hip.attention_prefill_masked(st["q"], st["k"], st["v"], st["o"], case["head_dim"] ** -0.5, causal=window,
                                     window=_window(case) if window else 0, bias=st.get("bias"), keep=st.get("keep"),
                                     fmt=FMT[case["dtype"]])
        return st["o"]
    if path == "decode":
        if case["append"]:
            hip.attention_decode_append(st["q"], st["k_new"], st["v_new"], st["k"], st["v"], st["o"], 128 ** -0.5,
                                        case["kv_len"] - 1, chunks=16, fmt=FMT[case["dtype"]])
            return st["o"], st["k"], st["v"]
        hip.attention_decode(st["q"], st["k"], st["v"], st["o"], 128 ** -0.5, chunks=16, fmt=FMT[case["dtype"]])
        return st["o"]
    if path == "gemm_i8":
        hip.gemm_i8(st["a"], st["b"], st["scale"], st["y"], case["m"], case["k"], case["n"], rhs_t=case["rhs_t"])
        return st["y"]
    if path == "gemm":
        fmt = FMT[case["dtype"]]
        hip.gemm_mfma(st["a"], st["b"], st["y"], case["m"], case["k"], case["n"], in_fmt=fmt,
                      out_fmt=fmt if case["out"] == "same" else B.F32, rhs_t=case["rhs_t"])
        return st["y"]
    if path == "mlp_f32":
        r, w, h = case["rows"], case["width"], case["hidden"]
        hip.gemm_f32_mfma(st["x"], st["w1"], st["h"], r, w, h, bias=st["b1"], epilogue=B.EPILOGUE_BIAS_GELU_TANH)
        hip.gemm_f32_mfma(st["h"], st["w2"], st["y"], r, h, w, bias=st["b2"], epilogue=B.EPILOGUE_BIAS)
        return st["y"]
    fmt = FMT[case["dtype"]]
    hip.gemm(st["a"], st["b"], st["y"], case["m"], case["k"], case["n"], in_fmt=fmt, out_fmt=fmt,
             psum=st.get("psum"))
    return st["y"]


# ------------------------------------------------------------------ what a pass has to move and compute
def work(case):
    path = case["path"]
    if path == "layer":
        hidden, hq, hkv, ffn = LAYERS[case["config"]]
        weights = hidden * (hq + 2 * hkv) * 128 + hidden * hidden + 3 * hidden * ffn + 2 * hidden
        return dict(bytes=2 * (weights + 2 * case["tokens"] * hidden),
                    flops=DL.flops(case["tokens"], hidden, hq, hkv, 128, ffn))
    if path in ("prefill", "masked"):
        b, hq, hkv, s, t, d = (case[k] for k in ("batch", "heads", "kv_heads", "q_len", "kv_len", "head_dim"))
        mask = {"padding": b * t, "additive": 4 * s * t}.get(case.get("kind"), 0)
        return dict(bytes=2 * b * d * (2 * hq * s + 2 * hkv * t) + mask, flops=4 * d * b * hq * _visible(case))
    if path == "decode":
        b, hq, hkv, t = (case[k] for k in ("batch", "heads", "kv_heads", "kv_len"))
        return dict(bytes=2 * 128 * b * (2 * hq + 2 * hkv * t), flops=4 * 128 * b * hq * t)
    if path == "mlp_f32":
        r, w, h = case["rows"], case["width"], case["hidden"]
        return dict(bytes=4 * (2 * r * w + 2 * w * h + h + w), flops=4 * r * w * h)
    m, k, n = case["m"], case["k"], case["n"]
    if path == "gemm_i8":
        return dict(bytes=m * k + k * n + 4 * n + 2 * m * n, flops=2 * m * n * k)
    e = 4 if case["dtype"] == "f32" else 2
    out = 4 if case.get("out") == "f32" else e
    return dict(bytes=e * (m * k + k * n) + out * m * n + (4 * m * n if case.get("psum") else 0), flops=2 * m * n * k)


def tolerance(case):
    """About four times the relative error against float64 that was measured
    over the ranges above: attention 2.3e-3 (BF16) and 2.7e-4 (F16), GEMMs
    1.7e-3 and 2.1e-4 (the output's rounding), a whole layer 6.5e-3 and 8e-4,
    f32 sums 5e-7."""
    path, half = case["path"], case.get("dtype")
    if path in ("gemm_i8", "formal"):
        return "exact"  # exact int32 sums; the formal lane's fixed order of operations
    if path == "mlp_f32":
        return {"rel": 2e-6}
    if path == "layer":
        return {"rel": 0.02 if half == "bf16" else 0.004}
    if path == "gemm":
        return {"rel": 2e-6 if case["out"] == "f32" else 0.007 if half == "bf16" else 0.001}
    return {"rel": 0.009 if half == "bf16" else 0.0012}


# ------------------------------------------------------------------ the same in 64 bits
def _attention64(q, k, v, scale, mask=None, bias=None):
    """softmax(q k^T scale + bias) v in float64, head by head; `mask`
    [b|1, 1, s, t] is true where a key is visible."""
    b, hq, s, _ = q.shape
    group = hq // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for i in range(b):
        for h in range(hq):
            x = q[i, h].double() @ k[i, h // group].double().t() * scale
            if bias is not None:
                x += bias[0, 0].double()
            if mask is not None:
                x.masked_fill_(~mask[i if mask.shape[0] > 1 else 0, 0], float("-inf"))
            out[i, h] = torch.softmax(x, dim=-1).nan_to_num(0.0) @ v[i, h // group].double()
    return out


def _layer64(case, inp):
    hidden, hq, hkv, ffn = LAYERS[case["config"]]
    t = case["tokens"]
    w = inp["weights"]

    def norm(x, g):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * g.double()

    def linear(x, m):  # in slices: a whole weight in 64 bits would be large
        return torch.cat([x @ p.double().t() for p in m.split(4096)], dim=1)

    freq = 1.0 / 1e4 ** (torch.arange(0, 128, 2, device="cuda", dtype=torch.float64) / 128)
    angle = torch.arange(t, device="cuda", dtype=torch.float64)[:, None] * freq[None]
    cos, sin = angle.cos().repeat(1, 2), angle.sin().repeat(1, 2)

    def rope(x):  # [heads, t, 128]
        return x * cos + torch.cat([-x[..., 64:], x[..., :64]], dim=-1) * sin

    x = inp["x"].double()
    qkv = linear(norm(x, w["input_norm"]), w["wqkv"]).view(t, hq + 2 * hkv, 128).transpose(0, 1)
    q, k, v = rope(qkv[:hq]), rope(qkv[hq:hq + hkv]), qkv[hq + hkv:]
    causal = torch.ones(t, t, dtype=torch.bool, device="cuda").tril().view(1, 1, t, t)
    a = _attention64(q[None], k[None], v[None], 128 ** -0.5, causal)[0].transpose(0, 1).reshape(t, hidden)
    x1 = x + linear(a, w["wo"])
    h2 = norm(x1, w["post_norm"])
    act = torch.nn.functional.silu(linear(h2, w["wgate"])) * linear(h2, w["wup"])
    return x1 + linear(act, w["wdown"])


def exact(case, seed):
    inp = _inputs(case, seed)
    path = case["path"]
    if path == "layer":
        return _layer64(case, inp)
    if path in ("prefill", "masked"):
        s, t = case["q_len"], case["kv_len"]
        i, j = torch.arange(s, device="cuda")[:, None], torch.arange(t, device="cuda")[None]
        mask = inp.get("keep")
        if mask is not None:
            mask = mask.expand(-1, 1, s, t)
        elif case.get("kind") == "window":
            mask = ((j <= i) & (j > i - _window(case))).view(1, 1, s, t)
        elif case.get("causal"):
            mask = (j <= i).view(1, 1, s, t)
        return _attention64(inp["q"], inp["k"], inp["v"], case["head_dim"] ** -0.5, mask, inp.get("bias"))
    if path == "decode":
        t = case["kv_len"]
        if case["append"]:
            for c in ("k", "v"):
                inp[c][:, :, t - 1:t] = inp[c + "_new"]
        o = _attention64(inp["q"], inp["k"][:, :, :t], inp["v"][:, :, :t], 128 ** -0.5)
        return (o, inp["k"].double(), inp["v"].double()) if case["append"] else o
    if path == "gemm_i8":
        b = inp["b"].double()
        return (inp["a"].double() @ (b.t() if case["rhs_t"] else b)) * inp["scale"].double()
    if path == "gemm":
        b = inp["b"].double()
        return inp["a"].double() @ (b.t() if case["rhs_t"] else b)
    if path == "mlp_f32":
        h = inp["x"].double() @ inp["w1"].double() + inp["b1"].double()
        h = torch.nn.functional.gelu(h, approximate="tanh")
        return h @ inp["w2"].double() + inp["b2"].double()
    y = inp["a"].double() @ inp["b"].double()
    return y + inp["psum"].double() if case["psum"] else y
