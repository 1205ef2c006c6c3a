"""The work that a user of this library has it do, as timed cases.

Every case is one call (or the one pair of calls that always go together)
through the public binding, gemma_hip.GemmaHip: the projections of a decode
step and of a prompt pass, the attention blocks of the prompt pass and of the
vision tower, and whole decode steps, prompt passes and images.  Shapes are
those of the configurations in model_bin (gemma-3-270m, -1b, -4b and SigLIP),
whole and ragged.

    gemv              quantize + W8A8 projections of one row (decode)
    gemm              quantize + W8A8 projections of a block of rows (prompt)
    gemm_f32          the same of an unquantized model file, fp32 weights
    attention         the prompt pass's attention over the key/value cache
    vision_attention  the tower's attention over all patches
    decode            greedy steps of a whole model behind a filled cache
    prefill           the prompt pass of a whole model
    tower             one image through the vision tower
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

# the package's folder has a dot in its name, so its modules go by path
sys.path.insert(0, os.path.join(os.getcwd(), "gemma.c_amd"))

import gemma_hip  # noqa: E402
import model_bin  # noqa: E402


def listed():
    return [
        # the smallest call of a decode step: q, k and v of gemma-3-270m, all latency
        dict(name="gemv_qkv_270m", op="gemv", n1=1024, n2=256, n3=256, k=640),
        # the largest: the LM head of gemma-3-1b, a 302 MB weight stream per token
        dict(name="gemv_lm_head_1b", op="gemv", n1=262144, n2=0, n3=0, k=1152),
        # a prompt of odd length through gemma-3-1b's down projection: few tiles, long rows
        dict(name="gemm_1b_down_471", op="gemm", m=471, n1=1152, n2=0, k=6912),
        # gate and up of gemma-3-4b over a 2048-token prompt, the largest product there is
        dict(name="gemm_4b_gate_up_2048", op="gemm", m=2048, n1=10240, n2=10240, k=2560),
        # gate and up of an unquantized gemma-3-1b over a 512-token prompt
        dict(name="gemm_f32_1b_gate_up", op="gemm_f32", m=512, n1=6912, n2=6912, k=1152),
        # a sliding-window layer of gemma-3-4b over a 2048-token prompt
        dict(name="attention_4b_sliding", op="attention", rows=2048, pos=0, heads=8, kv=4,
             hdim=256, slide=1024),
        # a global layer of gemma-3-1b, an odd chunk of a long prompt behind a filled cache
        dict(name="attention_1b_global_613", op="attention", rows=613, pos=1387, heads=4, kv=1,
             hdim=256, slide=0),
        # one SigLIP layer's attention: an 896-pixel image is 4096 patches
        dict(name="vision_attention_siglip", op="vision_attention", rows=4096, heads=16, dim=1152),
        # 16 greedy tokens of gemma-3-1b behind a 512-token prompt
        dict(name="decode_1b", op="decode", model="gemma-3-1b", layers=26, context=512, steps=16),
        # a short prompt through a third of gemma-3-270m, where launches count
        dict(name="prefill_270m_32", op="prefill", model="gemma-3-270m", layers=6, tokens=32),
        # a 2048-token prompt through a sliding and a global layer of gemma-3-4b
        dict(name="prefill_4b_2048", op="prefill", model="gemma-3-4b", layers=2, tokens=2048),
        # an 896-pixel image through a third of SigLIP's layers
        dict(name="tower_siglip", op="tower", px=896, layers=9),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, v, unit=1):
    """A multiple of 16, as every model's widths are, or now and then of `unit`."""
    unit = 16 if rng.random() < 0.8 else unit
    return v // unit * unit


def draw(rng):
    op = rng.choice(["gemv", "gemv", "gemm", "gemm", "gemm", "gemm_f32", "gemm_f32", "attention",
                     "attention", "attention", "vision_attention", "vision_attention", "decode",
                     "prefill", "prefill", "tower"])
    if op == "gemv":
        k = _width(rng, _log(rng, 640, 10240))
        top = min(262144, 300_000_000 // k)
        n1 = _log(rng, 256, top)
        return dict(op=op, n1=n1, n2=n1 if rng.random() < 0.5 and 2 * n1 <= top else 0, n3=0, k=k)
    if op in ("gemm", "gemm_f32"):
        k = _width(rng, _log(rng, 640, 10240), 4 if op == "gemm_f32" else 1)
        m = _log(rng, 17, 4096)
        # fp32 products cost about ten times the int8 ones
        most = 2048 * 20480 * 2560 // (12 if op == "gemm_f32" else 1)
        n1 = _width(rng, _log(rng, 256, max(512, min(10240, most // (m * k)))))
        pair = rng.random() < 0.5 and 2 * n1 * m * k <= most
        return dict(op=op, m=m, n1=n1, n2=n1 if pair else 0, k=k)
    if op == "attention":
        heads, kv, hdim = rng.choice([(4, 1, 256), (8, 4, 256), (8, 4, 256), (4, 2, 128)])
        rows = _log(rng, 16, 2048)
        return dict(op=op, rows=rows, pos=rng.choice([0, 0, rng.randint(1, 2048)]) if rows < 1400
                    else 0, heads=heads, kv=kv, hdim=hdim, slide=rng.choice([0, 512, 1024]))
    if op == "vision_attention":
        side = rng.randint(14, 64)  # images of 196 to 896 pixels in patches of 14
        heads, hdim = rng.choice([(16, 72), (16, 72), (12, 64)])
        return dict(op=op, rows=side * side, heads=heads, dim=heads * hdim)
    model = rng.choice(["gemma-3-270m", "gemma-3-1b"])
    if op == "decode":
        return dict(op=op, model=model, layers=rng.randint(2, 8), context=_log(rng, 16, 2000),
                    steps=rng.randint(2, 16))
    if op == "prefill":
        return dict(op=op, model=model, layers=rng.randint(1, 4), tokens=_log(rng, 16, 1500))
    return dict(op=op, px=14 * 4 * rng.randint(4, 16), layers=rng.randint(1, 6))


# ---- inputs ------------------------------------------------------------------

_gh = None


def _lib():
    """The library's handle: one per process, on the first GPU."""
    global _gh
    if _gh is None:
        torch.cuda.init()
        _gh = gemma_hip.GemmaHip(0)
    return _gh


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _weights_i8(g, n, k):
    """Int8 rows and scales of N(0, 0.02) weights quantized per row."""
    q = torch.empty((n, k), dtype=torch.int8, device="cuda")
    for i in range(0, n, 65536):
        j = min(n, i + 65536)
        q[i:j] = (_randn(g, j - i, k) * 31.75).round_().clamp_(-127, 127).to(torch.int8)
    s = torch.rand(n, generator=g, device="cuda") * 2e-4 + 5e-4
    return q, s


def _activations(g, m, k):
    """Rows as a norm leaves them, with a few channels far larger than the rest."""
    x = _randn(g, m, k)
    x[:, :: 97] *= 8.0
    return x


def _host(t):
    return t.cpu().numpy()


def _parts(case):
    return [n for n in (case["n1"], case["n2"], case.get("n3", 0)) if n]


def _norms(g, *names_sizes):
    return {name: _host(_randn(g, n) * 0.1) for name, n in names_sizes}


def _quantized(g, rows, cols):
    q, s = _weights_i8(g, rows, cols)
    return _host(q), _host(s)


def _global(i, layers):
    """Every sixth layer attends to all positions, here the last one too."""
    return (i + 1) % 6 == 0 or i + 1 == layers


def _text_model(g, name, layers):
    """A random W8A8 model in the layout that model_bin.read_bin() returns."""
    c = model_bin.CONFIGS[name]
    dim, hdim, mlp = c["dim"], c["hdim"], c["mlp"]
    q_sz, kv_sz = c["n_heads"] * hdim, c["nkv"] * hdim
    cfg = dict(nl=layers, n_heads=c["n_heads"], nkv=c["nkv"], hdim=hdim, dim=dim, mlp_dim=mlp,
               q_scale=hdim, slide=c["slide"], nvocab=model_bin.NVOCAB, theta_l=10000.0,
               theta_g=1000000.0, eps=1e-6, sc_att=0.0, sc_log=0.0, qk_norm=True, mlp_pre=True,
               mlp_pst=True, swa=[int(not _global(i, layers)) for i in range(layers)], quant=True)
    shapes = dict(wq=(q_sz, dim), wk=(kv_sz, dim), wv=(kv_sz, dim), wo=(dim, q_sz),
                  w1=(mlp, dim), w2=(mlp, dim), w3=(dim, mlp))
    out = []
    for _ in range(layers):
        ly = {w: _quantized(g, *s) for w, s in shapes.items()}
        ly.update(_norms(g, ("nq", hdim), ("nk", hdim), ("n1", dim), ("n2", dim), ("n3", dim),
                         ("n4", dim)))
        out.append(ly)
    return {"config": cfg, "emb": _quantized(g, model_bin.NVOCAB, dim), "layers": out,
            "fnorm": _host(_randn(g, dim) * 0.1)}


def _vision_model(g, px, layers):
    """A random W8A8 SigLIP tower of `layers` layers in model_bin's layout."""
    c = dict(model_bin.VISION_CONFIGS["siglip"], nl=layers, img_px=px)
    dim, mlp, p = c["dim"], c["mlp_dim"], c["psize"]
    c["img_tok"] = (px // p // 4) ** 2
    text_dim = model_bin.CONFIGS["gemma-3-4b"]["dim"]

    def vec(n, mean, std):
        return _host(_randn(g, n) * std + mean)

    out = []
    for _ in range(layers):
        ly = {w: _quantized(g, *s) for w, s in dict(
            wq=(dim, dim), wk=(dim, dim), wv=(dim, dim), wo=(dim, dim), w1=(mlp, dim),
            w2=(dim, mlp)).items()}
        ly.update({b: vec(n, 0.0, 0.02) for b, n in (("bq", dim), ("bk", dim), ("bv", dim),
                                                     ("bo", dim), ("b1", mlp), ("b2", dim))})
        ly.update(n1=vec(dim, 1.0, 0.05), n1_b=vec(dim, 0.0, 0.05), n2=vec(dim, 1.0, 0.05),
                  n2_b=vec(dim, 0.0, 0.05))
        out.append(ly)
    return {"config": dict(c, eps=1e-6, text_dim=text_dim, quant=True),
            "pe": _host(_randn(g, dim, 3 * p * p) * 0.02), "pe_b": vec(dim, 0.0, 0.02),
            "pos": _quantized(g, (px // p) ** 2, dim), "layers": out,
            "post_n": vec(dim, 1.0, 0.05), "post_nb": vec(dim, 0.0, 0.05),
            "norm": vec(dim, 0.0, 0.1), "proj": _quantized(g, text_dim, dim)}


class _Owned:
    """A decoder or a tower that goes when the state that holds it goes."""

    def __init__(self, obj):
        self.obj = obj

    def __del__(self):
        if not sys.is_finalizing():
            self.obj.close()


def prepare(case, seed):
    gh, g, op = _lib(), _gen(seed), case["op"]
    if op == "gemv":
        k = case["k"]
        w = [_weights_i8(g, n, k) for n in _parts(case)]
        return dict(op=op, k=k, x=_activations(g, 1, k)[0].contiguous(), w=w,
                    y=[torch.empty(n, device="cuda") for n in _parts(case)],
                    xq=torch.empty(k, dtype=torch.int8, device="cuda"),
                    xs=torch.empty(1, device="cuda"))
    if op == "gemm":
        m, k = case["m"], case["k"]
        w = [_weights_i8(g, n, k) for n in _parts(case)]
        return dict(op=op, m=m, k=k, x=_activations(g, m, k), w=w,
                    q=torch.empty((m, k), dtype=torch.int8, device="cuda"),
                    s=torch.empty(m, device="cuda"),
                    y=torch.empty((m, sum(_parts(case))), device="cuda"))
    if op == "gemm_f32":
        m, k = case["m"], case["k"]
        w = [_randn(g, n, k) * 0.02 for n in _parts(case)]
        return dict(op=op, m=m, k=k, x=_activations(g, m, k), w=w,
                    y=torch.empty((m, sum(_parts(case))), device="cuda"))
    if op == "attention":
        # q and k as the q/k norms leave them: every head row of unit mean square
        n, h, kv, d, p = (case[f] for f in ("rows", "heads", "kv", "hdim", "pos"))
        unit = lambda t: t / t.square().mean(-1, keepdim=True).sqrt()  # noqa: E731
        return dict(op=op, case=dict(case), q=unit(_randn(g, n, h, d)).reshape(n, h * d),
                    kc=unit(_randn(g, kv, p + n, d)), vc=_randn(g, kv, p + n, d),
                    out=torch.empty((n, h * d), device="cuda"))
    if op == "vision_attention":
        n, dim = case["rows"], case["dim"]
        return dict(op=op, case=dict(case), qkv=_randn(g, n, 3 * dim),
                    bias=_randn(g, 3 * dim) * 0.02, out=torch.empty((n, dim), device="cuda"))
    if op in ("decode", "prefill"):
        model = _text_model(g, case["model"], case["layers"])
        ids = np.random.default_rng(seed).integers(6, model_bin.NVOCAB, 4096).astype(np.int32)
        logits = np.empty(model_bin.NVOCAB, np.float32)
        if op == "prefill":
            n = case["tokens"]
            return dict(op=op, own=_Owned(gh.decoder(model, n + 64)), ids=ids[:n], logits=logits)
        n, steps = case["context"], case["steps"]
        dec = gh.decoder(model, n + steps)
        # the cache is filled in the verification arithmetic, so that what the
        # steps return depends on the steps alone
        dec.set_attention(gemma_hip.ATTN_F64)
        first = dec.prefill(ids[:n], 0)
        dec.set_attention(gemma_hip.ATTN_F32)
        return dict(op=op, own=_Owned(dec), first=first, pos=n, steps=steps, logits=logits)
    vis = gh.vision(_vision_model(g, case["px"], case["layers"]))
    return dict(op=op, own=_Owned(vis), img=model_bin.synth_image(case["px"], seed))


# ---- one pass ----------------------------------------------------------------


def run(st):
    gh, op = _lib(), st["op"]
    if op == "decode":
        # all but the last token without leaving the GPU, the last with its logits
        dec, pos, n = st["own"].obj, st["pos"], st["steps"]
        toks = dec.generate(st["first"], pos, n - 1)
        last = dec.step(int(toks[-1]), pos + n - 1, st["logits"])
        return dict(logits=st["logits"], tokens=toks, last=last)
    if op == "prefill":
        st["own"].obj.prefill(st["ids"], 0, st["logits"])
        return st["logits"]
    if op == "tower":
        return st["own"].obj.forward(st["img"])
    s = torch.cuda.current_stream().cuda_stream
    if op == "gemv":
        gh.quantize_matmul([(q, sc, y, y.numel()) for (q, sc), y in zip(st["w"], st["y"])],
                           st["x"], st["k"], st["xq"], st["xs"], s)
        return dict(y=st["y"], xq=st["xq"], xs=st["xs"])
    if op == "gemm":
        m, k = st["m"], st["k"]
        gh.quantize(st["q"], st["s"], st["x"], k, m, k, s)
        gh.matmul_cols(st["y"], 0, [(q, sc, q.shape[0]) for q, sc in st["w"]], st["q"], k,
                       st["s"], m, k, s)
        return dict(y=st["y"], q=st["q"], s=st["s"])
    if op == "gemm_f32":
        m, k = st["m"], st["k"]
        gh.matmul_f32_cols(st["y"], 0, [(w, w.shape[0]) for w in st["w"]], st["x"], k, m, k, s)
        return st["y"]
    c = st["case"]
    if op == "attention":
        n, h, d = c["rows"], c["heads"], c["hdim"]
        gh.prefill_attention(st["out"], st["q"], h * d, st["kc"], st["vc"], n, c["pos"], h,
                             c["kv"], d, c["pos"] + n, c["slide"], 1.0 / math.sqrt(d), 0.0, False,
                             gemma_hip.ATTN_F32, s)
        return st["out"]
    gh.vision_attention(st["out"], st["qkv"], st["bias"], c["rows"], c["heads"], c["dim"],
                        gemma_hip.ATTN_F32, s)
    return st["out"]


# ---- what a pass cannot do without ---------------------------------------------


def _pairs(rows, pos, slide):
    """(query, key) pairs of causal rows at pos .. pos + rows - 1."""
    return sum(min(p + 1, slide) if slide else p + 1 for p in range(pos, pos + rows))


def _text_sizes(name):
    c = model_bin.CONFIGS[name]
    q, kv = c["n_heads"] * c["hdim"], c["nkv"] * c["hdim"]
    return c, q, kv, c["dim"] * (2 * q + 2 * kv + 3 * c["mlp"])  # weights of a layer


def work(case):
    op = case["op"]
    if op == "gemv":
        n, k = sum(_parts(case)), case["k"]
        return dict(bytes=n * k + 8 * n + 5 * k + 4, flops=2 * n * k)
    if op == "gemm":
        m, n, k = case["m"], sum(_parts(case)), case["k"]
        return dict(bytes=5 * m * k + 4 * m + n * k + 4 * n + 4 * m * n, flops=2 * m * n * k)
    if op == "gemm_f32":
        m, n, k = case["m"], sum(_parts(case)), case["k"]
        return dict(bytes=4 * (m * k + n * k + m * n), flops=2 * m * n * k)
    if op == "attention":
        n, h, d = case["rows"], case["heads"], case["hdim"]
        return dict(bytes=4 * (2 * n * h * d + 2 * case["kv"] * (case["pos"] + n) * d),
                    flops=4 * h * d * _pairs(n, case["pos"], case["slide"]))
    if op == "vision_attention":
        n, dim = case["rows"], case["dim"]
        return dict(bytes=4 * (4 * n * dim + 3 * dim), flops=4 * n * n * dim)
    if op == "tower":
        v = model_bin.VISION_CONFIGS["siglip"]
        n, d = (case["px"] // v["psize"]) ** 2, v["dim"]
        layer = 4 * d * d + 2 * d * v["mlp_dim"]
        patch, out = 3 * v["psize"] ** 2, model_bin.CONFIGS["gemma-3-4b"]["dim"]
        tok = n // 16
        return dict(bytes=case["layers"] * layer + 4 * d * patch + n * d + out * d + 4 * tok * out
                    + 12 * case["px"] ** 2,
                    flops=2 * n * d * patch + 2 * tok * out * d
                    + case["layers"] * (2 * n * layer + 4 * n * n * d))
    c, q, kv, layer = _text_sizes(case["model"])
    nl, head = case["layers"], model_bin.NVOCAB * c["dim"]
    swa = sum(not _global(i, nl) for i in range(nl))
    if op == "decode":
        pos = range(case["context"], case["context"] + case["steps"])
        keys = sum(swa * min(p + 1, c["slide"]) + (nl - swa) * (p + 1) for p in pos)
        n = case["steps"]
        return dict(bytes=n * (nl * layer + head) + 8 * kv * keys + 4 * model_bin.NVOCAB,
                    flops=2 * n * (nl * layer + head) + 4 * q * keys)
    n = case["tokens"]
    pairs = swa * _pairs(n, 0, c["slide"]) + (nl - swa) * _pairs(n, 0, 0)
    return dict(bytes=nl * (layer + 8 * n * kv) + head + 4 * model_bin.NVOCAB,
                flops=2 * n * nl * layer + 2 * head + 4 * q * pairs)


# ---- how far a correct result may be off ------------------------------------------


def tolerance(case):
    op = case["op"]
    if op in ("gemv", "gemm", "decode"):
        # quantize, integer sums and the rescale are a contract to the bit, and the
        # decode step's norms, attention and GELU are 64-bit, rounded once
        return "exact" if op != "decode" else {"rel": 1e-5}
    if op in ("gemm_f32", "attention", "vision_attention"):
        return {"rel": 4e-6, "max": 1e-4}
    # a whole W8A8 pass: one fp32 rounding that moves an activation over a
    # quantizer's .5 boundary travels through every later layer (two correct
    # attention kernels: up to 0.027 over these prompts, 0.014 over the tower)
    return {"rel": 0.03, "max": 0.3}


# ---- the same in 64 bits ------------------------------------------------------------


def _quantize64(x):
    amax = x.abs().amax(-1, keepdim=True)
    return torch.trunc(x * (127.0 / amax) + 0.5 * torch.sign(x)), amax / 127.0


def exact(case, seed):
    """In plain torch at 64 bits; None for whole W8A8 models, where a tie at a
    quantizer's boundary decides each later layer's integers, and for integers."""
    op = case["op"]
    if op in ("decode", "prefill", "tower"):
        return None
    st = prepare(case, seed)
    if op in ("gemv", "gemm"):
        q, s = _quantize64(st["x"].double().reshape(-1, case["k"]))
        y = []
        for w, ws in st["w"]:
            y.append(torch.cat([(q @ w[i:i + 16384].double().t()) * ws[i:i + 16384].double() * s
                                for i in range(0, w.shape[0], 16384)], 1))
        if op == "gemv":
            return dict(y=[v[0] for v in y], xq=None, xs=s[0])
        return dict(y=torch.cat(y, 1), q=None, s=s[:, 0])
    if op == "gemm_f32":
        x = st["x"].double()
        return torch.cat([x @ w.double().t() for w in st["w"]], 1)
    if op == "attention":
        n, h, kv, d, p = (case[f] for f in ("rows", "heads", "kv", "hdim", "pos"))
        at = torch.arange(p, p + n, device="cuda")[:, None]
        key = torch.arange(p + n, device="cuda")[None, :]
        off = (key > at) | ((key <= at - case["slide"]) if case["slide"] else key < 0)
        q, out = st["q"].double().reshape(n, h, d), []
        for i in range(h):
            j = i // (h // kv)
            sc = (q[:, i] @ st["kc"][j].double().t()) / math.sqrt(d)
            out.append(torch.softmax(sc.masked_fill(off, -math.inf), 1) @ st["vc"][j].double())
        return torch.cat(out, 1)
    n, h, dim = case["rows"], case["heads"], case["dim"]
    x = (st["qkv"] + st["bias"]).double().reshape(n, 3, h, dim // h)
    out = []
    for i in range(h):
        sc = (x[:, 0, i] @ x[:, 1, i].t()) / math.sqrt(dim // h)
        out.append(torch.softmax(sc, 1) @ x[:, 2, i])
    return torch.cat(out, 1)
