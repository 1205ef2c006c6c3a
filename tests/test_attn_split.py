"""The split-f16 attention (attn_split.h) where it can go wrong: counts of
queries and keys around its 32-key tiles and its 128- and 256-query
workgroups, every head dim with and without a partial 32-dim block, tiles
whose magnitudes differ by far more than f16's range, and calls that can't
have a workspace.

Bars, relative to the largest output.  A product of two 22-bit operands keeps
all but 2^-21 of itself, so a score s = sum q k is off by at most
2^-21 sum |q k| (5e-7 * 16 at the inputs here, whose scaled |q||k| sums stay
below 16), a weight by that much relatively, and an output, a weighted mean, by
the same of the largest value: 8e-6; the fp32 sums over up to a thousand keys
add the 1e-5 that the other fp32 kernels are held to."""

from __future__ import annotations

import numpy as np
import pytest

TOL = 2e-5
F64 = np.float64


def _softmax_av(s, v):
    p = np.exp(s - s.max(axis=1, keepdims=True))
    return (p @ v) / p.sum(axis=1, keepdims=True)


def _vision_want(qkv, bias, heads, dim):
    x = (qkv + bias).astype(F64)
    hd = dim // heads
    out = []
    for h in range(heads):
        c = slice(h * hd, (h + 1) * hd)
        q, k, v = x[:, :dim][:, c], x[:, dim:2 * dim][:, c], x[:, 2 * dim:][:, c]
        out.append(_softmax_av(q @ k.T * F64(np.float32(1) / np.sqrt(np.float32(hd))), v))
    return np.concatenate(out, axis=1)


def _vision(gh, qkv, bias, heads, dim, stream=None):
    import torch

    n = qkv.shape[0]
    dq, db = torch.from_numpy(qkv).cuda(), torch.from_numpy(bias).cuda()
    out = torch.full((n + 1, dim), float("nan"), device="cuda")
    gh.vision_attention(out, dq, db, n, heads, dim, 1,
                        stream or torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.isnan(got[n]).all()  # nothing past the last row
    return got[:n]


def _close(got, want, tol=TOL):
    rel = float(np.abs(got - want).max()) / float(np.abs(want).max())
    print(f"|d|/max = {rel:.3g}", flush=True)
    assert rel <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("n,heads,hd", [
    (1, 2, 72), (31, 2, 72), (32, 1, 16), (33, 3, 64), (64, 2, 32), (65, 2, 128), (127, 2, 72),
    (128, 2, 64), (129, 1, 72), (257, 1, 32), (257, 130, 16), (300, 100, 72)])
def test_vision_tile_edges(gh, n, heads, hd):
    rng = np.random.default_rng(n + hd)
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim)).astype(np.float32)
    bias = (0.5 * rng.standard_normal(3 * dim)).astype(np.float32)
    _close(_vision(gh, qkv, bias, heads, dim), _vision_want(qkv, bias, heads, dim))


def _tile_scales(n, exps):
    """2^e per 32-row tile, cycling through exps."""
    return np.exp2(np.asarray(exps, F64)[(np.arange(n) // 32) % len(exps)])[:, None]


@pytest.mark.gpu
@pytest.mark.parametrize("exps", [(0, 20, -20), (60, 0), (0, 3, -30, 30), (100, -90, 0),
                                  (-140, -140, -120)],
                         ids=lambda e: "v2^" + "_".join(map(str, e)))
def test_vision_tiles_of_any_magnitude(gh, exps):
    """Each 32-key tile of V at its own magnitude, the output of every query
    that of the largest it sees; q and k rows at magnitudes whose products are
    ordinary."""
    rng = np.random.default_rng(7)
    n, heads, hd = 300, 2, 72
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim))
    qs = np.exp2(rng.integers(-30, 30, n))[:, None]
    qkv[:, :dim] *= qs
    qkv[:, dim:2 * dim] *= 2.0 ** -30
    qkv[:, 2 * dim:] *= _tile_scales(n, exps)
    qkv = qkv.astype(np.float32)
    bias = np.zeros(3 * dim, np.float32)
    _close(_vision(gh, qkv, bias, heads, dim), _vision_want(qkv, bias, heads, dim))


@pytest.mark.gpu
def test_vision_small_tiles_keep_their_precision(gh):
    """A tile of huge values whose weights vanish leaves the others' precision
    alone, whether it comes first, last or between them."""
    rng = np.random.default_rng(8)
    n, heads, hd = 320, 1, 72
    q = rng.standard_normal((n, hd))
    q[:, 0] = 40.0  # the huge tile's keys score -40 * 40 / sqrt(72) below the rest
    k = rng.standard_normal((n, hd))
    k[:, 0] = 0.0
    for first in (0, 128, 288):
        kk, v = k.copy(), rng.standard_normal((n, hd))
        kk[first:first + 32, 0] = -40.0
        v[first:first + 32] *= 2.0 ** 60
        qkv = np.concatenate([q, kk, v], axis=1).astype(np.float32)
        bias = np.zeros(3 * hd, np.float32)
        _close(_vision(gh, qkv, bias, heads, hd), _vision_want(qkv, bias, heads, hd))


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [16, 32, 64, 72, 128])
@pytest.mark.parametrize("exps", [(55, 0, -55), (None, -62, -62), (-62, None, -62), (0, None, 0),
                                  (30, 60, 90), (100, 50, 0, -50, -100), (-9, 0, 0)],
                         ids=lambda e: "v2^" + "_".join(map(str, e)))
def test_vision_value_tiles_far_apart(gh, exps, hd):
    """Tiles of V that fall or rise time and again, and tiles of zeros (None):
    every query's output is that of all of them."""
    rng = np.random.default_rng(hd)
    n, heads = 32 * len(exps) + 5, 2
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim))
    e = np.array([-np.inf if x is None else x for x in exps])[(np.arange(n) // 32) % len(exps)]
    qkv[:, 2 * dim:] *= np.exp2(e)[:, None]
    qkv = qkv.astype(np.float32)
    bias = np.zeros(3 * dim, np.float32)
    _close(_vision(gh, qkv, bias, heads, dim), _vision_want(qkv, bias, heads, dim))


def _close_each(got, want, axis, tol=TOL):
    """Every row (axis 1) or column (axis 0) held to its own largest value: TOL is
    that of the weights, which all of a row's or a column's outputs share."""
    rel = float((np.abs(got - want).max(axis=axis) / np.abs(want).max(axis=axis)).max())
    print(f"largest |d|/max of one = {rel:.3g}", flush=True)
    assert rel <= tol


@pytest.mark.gpu
@pytest.mark.parametrize("n,exp", [(96, -6), (96, -10), (300, -18), (96, -24), (33, -24),
                                   (5, -24), (96, -60)])
@pytest.mark.parametrize("hd", [64, 72])
def test_vision_small_dims(gh, n, exp, hd):
    """Dims of V far below the rest of their tiles keep their own precision."""
    rng = np.random.default_rng(n - exp)
    qkv = rng.standard_normal((n, 3 * hd))
    small = [2 * hd + 5, 3 * hd - 1]
    qkv[:, small] *= 2.0 ** exp
    qkv = qkv.astype(np.float32)
    bias = np.zeros(3 * hd, np.float32)
    _close_each(_vision(gh, qkv, bias, 1, hd), _vision_want(qkv, bias, 1, hd), 0)


@pytest.mark.gpu
@pytest.mark.parametrize("exp", [-4, -12, -20, -40, None])
@pytest.mark.parametrize("hd", [16, 72, 128])
def test_vision_small_keys(gh, exp, hd):
    """Queries whose weight is all but wholly on keys with values far below the
    others', which are in their tile, or zero: the others' share of them, about
    e^-14, is as precise as the rest."""
    rng = np.random.default_rng(hd)
    n = 200
    q, k, v = (rng.standard_normal((n, hd)) for _ in range(3))
    q *= 0.3
    k *= 0.3
    q[:, 0] = 2.0
    k[:, 0] = 0.0
    k[[3, 77, 78, 150], 0] = 7.0 * np.sqrt(hd)
    v[[3, 77, 78, 150]] *= 0.0 if exp is None else 2.0 ** exp
    qkv = np.concatenate([q, k, v], axis=1).astype(np.float32)
    bias = np.zeros(3 * hd, np.float32)
    _close_each(_vision(gh, qkv, bias, 1, hd), _vision_want(qkv, bias, 1, hd), 1)


@pytest.mark.gpu
@pytest.mark.parametrize("exp", [4, 12, 20, 40])
def test_vision_query_outliers(gh, exp):
    """A dim of the queries far above the others, met by zeros in the keys, and
    one of the keys met by zeros in the queries: scores come from the others."""
    rng = np.random.default_rng(exp)
    n, hd = 160, 72
    qkv = rng.standard_normal((n, 3 * hd))
    qkv[:, 7] *= 2.0 ** exp
    qkv[:, hd + 7] = 0
    qkv[:, 9] = 0
    qkv[:, hd + 9] *= 2.0 ** exp
    qkv = qkv.astype(np.float32)
    bias = np.zeros(3 * hd, np.float32)
    _close_each(_vision(gh, qkv, bias, 1, hd), _vision_want(qkv, bias, 1, hd), 1)


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["dims", "keys", "outlier"])
@pytest.mark.parametrize("hd,n,pos0,slide", [(256, 150, 90, 0), (128, 260, 0, 100)])
def test_prefill_small_values(gh, monkeypatch, what, hd, n, pos0, slide):
    """The same of the prompt pass, whole and in chunks of its keys."""
    monkeypatch.setenv("GEMMA_HIP_PF_ATTN", "bf3")
    nh, nkv = 4, 2
    q, kc, vc = _prefill_inputs(n, pos0, nh, nkv, hd, seed=hd)
    ctx = pos0 + n
    q *= np.float32(0.5)
    if what == "dims":
        vc[:, :ctx, [5, hd - 1]] *= np.float32(2.0 ** -24)
    elif what == "keys":
        kc[:, :ctx, 0] = 0
        q[:, 0:nh * hd:hd] = 2
        kc[:, 3:ctx:40, 0] = 7.0 * np.sqrt(hd)
        vc[:, 3:ctx:40] *= np.float32(2.0 ** -16)
    else:
        q[:, 1:nh * hd:hd] *= np.float32(2.0 ** 20)
        kc[:, :ctx, 1] = 0
    args = (n, pos0, nh, nkv, hd, slide, 0.0, False)
    got, want = _prefill(gh, q, kc, vc, *args), _prefill_want(q, kc, vc, *args)
    for h in range(nh):
        c = slice(h * hd, (h + 1) * hd)
        _close_each(got[:, c], want[:, c], 0 if what == "dims" else 1)


@pytest.mark.gpu
@pytest.mark.parametrize("first", [0, 128, 288])
@pytest.mark.parametrize("exp", [70, 110])
def test_vision_huge_tile_of_no_weight(gh, exp, first):
    """A tile of V further above the rest than any running unit could follow,
    whose weights are zero: the others' values stay whole."""
    rng = np.random.default_rng(exp + first)
    n, hd = 320, 72
    q, k, v = (rng.standard_normal((n, hd)) for _ in range(3))
    q[:, 0] = 40.0  # the huge tile's keys score -40 * 40 / sqrt(72) below the rest: e^-188
    k[:, 0] = 0.0
    k[first:first + 32, 0] = -40.0
    v[first:first + 32] *= 2.0 ** exp
    qkv = np.concatenate([q, k, v], axis=1).astype(np.float32)
    bias = np.zeros(3 * hd, np.float32)
    _close(_vision(gh, qkv, bias, 1, hd), _vision_want(qkv, bias, 1, hd))


@pytest.mark.gpu
def test_vision_zero_and_peaked(gh):
    """All-zero q, k or v tiles, and scores so far apart that one key takes
    all the weight (the reference maximum moves with nearly every tile)."""
    rng = np.random.default_rng(9)
    n, heads, hd = 200, 2, 64
    dim = heads * hd
    bias = np.zeros(3 * dim, np.float32)
    qkv = rng.standard_normal((n, 3 * dim)).astype(np.float32)
    qkv[40:80, :dim] = 0
    qkv[64:96, dim:] = 0
    _close(_vision(gh, qkv, bias, heads, dim), _vision_want(qkv, bias, heads, dim))
    # key j scores about 4 j for every query: whole numbers, exact in every form
    qkv = np.zeros((n, 3 * dim), np.float32)
    qkv[:, 0:dim:hd] = 8.0
    qkv[:, dim:2 * dim:hd] = 4.0 * np.arange(n)[:, None]
    qkv[:, 2 * dim:] = rng.standard_normal((n, dim))
    _close(_vision(gh, qkv, bias, heads, dim), _vision_want(qkv, bias, heads, dim))


@pytest.mark.gpu
def test_vision_attention_under_capture(gh):
    """A captured call can't allocate a workspace: it takes the kernel that
    needs none, and each replay gives that kernel's result."""
    import torch

    rng = np.random.default_rng(10)
    n, heads, hd = 300, 2, 72
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim)).astype(np.float32)
    bias = (0.5 * rng.standard_normal(3 * dim)).astype(np.float32)
    want = _vision_want(qkv, bias, heads, dim)
    dq, db = torch.from_numpy(qkv).cuda(), torch.from_numpy(bias).cuda()
    out = torch.zeros((n, dim), device="cuda")
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        gh.vision_attention(out, dq, db, n, heads, dim, 1, side.cuda_stream)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        _close(out.cpu().numpy(), want)
        _close(_vision(gh, qkv, bias, heads, dim), want)


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [16, 32, 64, 72, 128])
@pytest.mark.parametrize("n,heads", [(1, 1), (33, 2), (129, 1), (257, 3), (300, 8)])
def test_vision_workspace_free_kernel(gh, n, heads, hd):
    """The kernel of captured calls at every head dim and around its 16-query
    waves, 128- and 256-query workgroups and 32-key tiles, V's tiles at
    magnitudes far apart."""
    import torch

    rng = np.random.default_rng(n + hd)
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim))
    qkv[:, 2 * dim:] *= _tile_scales(n, (0, 40, -40))
    qkv = qkv.astype(np.float32)
    bias = (0.5 * rng.standard_normal(3 * dim)).astype(np.float32)
    want = _vision_want(qkv, bias, heads, dim)
    dq, db = torch.from_numpy(qkv).cuda(), torch.from_numpy(bias).cuda()
    out = torch.full((n + 1, dim), float("nan"), device="cuda")
    side = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        gh.vision_attention(out, dq, db, n, heads, dim, 1, side.cuda_stream)
    for _ in range(2):
        out[:n] = 0
        graph.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        assert np.isnan(got[n]).all()
        _close(got[:n], want)


def _prefill_want(q, kc, vc, n, pos0, nh, nkv, hd, slide, cap, dense, asc=None):
    ctx = pos0 + n
    pos = pos0 + np.arange(n)
    j = np.arange(ctx)[None, :]
    live = np.ones((n, ctx), bool) if dense else j <= pos[:, None]
    if slide and not dense:
        live = live & (j > pos[:, None] - slide)
    out = []
    for h in range(nh):
        s = q[:, h * hd:(h + 1) * hd].astype(F64) @ kc[h // (nh // nkv), :ctx].astype(F64).T
        s = s / np.sqrt(F64(hd)) if asc is None else s * F64(np.float32(asc))
        if cap:
            s = np.tanh(s / cap) * cap
        out.append(_softmax_av(np.where(live, s, -np.inf), vc[h // (nh // nkv), :ctx].astype(F64)))
    return np.concatenate(out, axis=1)


def _prefill(gh, q, kc, vc, n, pos0, nh, nkv, hd, slide, cap, dense, asc=None):
    import torch

    dq, dk, dv = (torch.from_numpy(a).cuda() for a in (q, kc, vc))
    out = torch.full((n + 1, nh * hd), float("nan"), device="cuda")
    gh.prefill_attention(out, dq, q.shape[1], dk, dv, n, pos0, nh, nkv, hd, kc.shape[1], slide,
                         np.float32(1.0) / np.sqrt(np.float32(hd)) if asc is None else asc, cap,
                         dense, 1, stream=torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    assert np.isnan(got[n]).all()
    return got[:n]


def _prefill_inputs(n, pos0, nh, nkv, hd, seed):
    rng = np.random.default_rng(seed)
    q = rng.standard_normal((n, nh * hd + 8)).astype(np.float32)  # a padded row stride
    kc = rng.standard_normal((nkv, pos0 + n + 5, hd)).astype(np.float32)
    vc = rng.standard_normal((nkv, pos0 + n + 5, hd)).astype(np.float32)
    kc[:, pos0 + n:] = np.nan  # never read
    vc[:, pos0 + n:] = np.nan
    return q, kc, vc


@pytest.mark.gpu
@pytest.mark.parametrize("n,pos0,nh,nkv,hd,slide,cap,dense", [
    (1, 0, 4, 1, 256, 0, 0.0, False), (33, 0, 4, 1, 256, 0, 0.0, False),
    (32, 31, 2, 1, 256, 0, 0.0, False), (65, 127, 8, 4, 256, 40, 0.0, False),
    (129, 0, 4, 2, 128, 33, 0.0, False), (64, 1, 4, 1, 128, 1, 0.0, False),
    (97, 300, 32, 1, 128, 64, 0.0, False), (40, 500, 4, 1, 256, 100, 30.0, False),
    (70, 26, 2, 2, 128, 16, 5.0, True), (257, 11, 8, 4, 256, 0, 0.0, True)])
def test_prefill_tile_edges(gh, monkeypatch, n, pos0, nh, nkv, hd, slide, cap, dense):
    monkeypatch.setenv("GEMMA_HIP_PF_ATTN", "bf3")  # the split kernel at every size
    q, kc, vc = _prefill_inputs(n, pos0, nh, nkv, hd, seed=n + hd)
    args = (n, pos0, nh, nkv, hd, slide, cap, dense)
    _close(_prefill(gh, q, kc, vc, *args), _prefill_want(q, kc, vc, *args))


@pytest.mark.gpu
@pytest.mark.parametrize("hd", [128, 256])
def test_prefill_tiles_of_any_magnitude(gh, monkeypatch, hd):
    """Tiles of V at magnitudes far apart, a window that hides the largest
    from some rows (held to their own largest output)."""
    monkeypatch.setenv("GEMMA_HIP_PF_ATTN", "bf3")
    n, pos0, nh, nkv, slide = 150, 200, 4, 2, 90
    q, kc, vc = _prefill_inputs(n, pos0, nh, nkv, hd, seed=3)
    ctx = pos0 + n
    vc[:, :ctx] *= _tile_scales(ctx, (0, 12, -12, 30)).astype(np.float32)
    q *= np.exp2(np.random.default_rng(4).integers(-20, 20, n))[:, None].astype(np.float32)
    kc[:, :ctx] *= np.float32(2.0 ** -20)
    args = (n, pos0, nh, nkv, hd, slide, 0.0, False)
    got, want = _prefill(gh, q, kc, vc, *args), _prefill_want(q, kc, vc, *args)
    for i in range(n):
        _close(got[i], want[i])


@pytest.mark.gpu
@pytest.mark.parametrize("what", ["v2^70", "v2^110", "vinf", "vnan", "kinf"])
@pytest.mark.parametrize("hd", [128, 256])
def test_prefill_unseen_tiles(gh, monkeypatch, hd, what):
    """Rows 0 .. 95 of a causal pass, 16 to a wave, against keys 96 .. 127 that
    none of them sees but that their workgroup walks: huge, infinite or no
    numbers, they leave those rows what they are; and the same of the first 32
    keys for rows 64 .. 127 behind a 16-key window."""
    monkeypatch.setenv("GEMMA_HIP_PF_ATTN", "bf3")
    n, nh, nkv = 128, 2, 2
    for slide, hidden, rows in ((0, slice(96, 128), slice(0, 96)),
                                (16, slice(0, 32), slice(64, 128))):
        q, kc, vc = _prefill_inputs(n, 0, nh, nkv, hd, seed=hd)
        to = kc if what[0] == "k" else vc
        if what[1:] in ("inf", "nan"):
            to[:, hidden] = np.float32(what[1:])
        else:
            to[:, hidden] *= np.float32(2.0 ** int(what[3:]))
        got = _prefill(gh, q, kc, vc, n, 0, nh, nkv, hd, slide, 0.0, False)
        kc[:, hidden] = vc[:, hidden] = 0  # nothing of them reaches those rows
        want = _prefill_want(q, kc, vc, n, 0, nh, nkv, hd, slide, 0.0, False)
        _close(got[rows], want[rows])


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["", "bf3", "f32"])
@pytest.mark.parametrize("n,hd,asc,cap", [(750, 256, -0.0625, 0.0), (90, 256, -0.25, 20.0),
                                          (90, 128, -0.5, 0.0), (90, 256, 0.0, 0.0)])
def test_prefill_scale_sign(gh, monkeypatch, kind, n, hd, asc, cap):
    """Scores are q.k * asc for any asc, whichever kernel runs: negative, and
    zero (every visible key weighs the same)."""
    monkeypatch.setenv("GEMMA_HIP_PF_ATTN", kind)
    q, kc, vc = _prefill_inputs(n, 7, 4, 1, hd, seed=n)
    q *= np.float32(0.5)  # |q.k| asc stays below 16, as TOL assumes
    args = (n, 7, 4, 1, hd, 0, cap, False, asc)
    _close(_prefill(gh, q, kc, vc, *args), _prefill_want(q, kc, vc, *args))


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["gemma-3-4b", "test-hd128"])
def test_prefill_kernel_choice_agrees(gh, monkeypatch, model):
    """Either side of the size where the split kernel takes over, the default
    is one of the two forced kernels' results, and both agree."""
    import model_bin

    c = model_bin.CONFIGS[model]
    nh, nkv, hd = c["n_heads"], c["nkv"], c["hdim"]
    least = 1.1e9 * hd / 256  # flops: 4 hd nh pairs
    edge = int((least / (2 * hd * nh)) ** 0.5)
    for n in (edge - 8, edge + 8):
        q, kc, vc = _prefill_inputs(n, 0, nh, nkv, hd, seed=5)
        args = (n, 0, nh, nkv, hd, 0, 0.0, False)
        outs = {}
        for kind in ("f32", "bf3", ""):
            monkeypatch.setenv("GEMMA_HIP_PF_ATTN", kind)
            outs[kind] = _prefill(gh, q, kc, vc, *args)
        _close(outs["bf3"], outs["f32"])
        assert np.array_equal(outs[""], outs["bf3" if n > edge else "f32"]), n


@pytest.mark.gpu
def test_attention_workspaces_by_stream(gh):
    """The kept workspaces: calls of different sizes and both entry points in
    turn on two streams at once, no call waited for, each with its own inputs;
    and a captured call of the prompt's entry point, refused."""
    import torch

    from gemma_hip import GemmaHipError

    streams = [torch.cuda.Stream() for _ in range(2)]
    hd, nh, nkv, jobs = 128, 4, 2, []
    for i, n in enumerate((40, 300, 90, 500, 64, 400)):
        q, kc, vc = _prefill_inputs(n, 0, nh, nkv, hd, seed=20 + i)
        qkv = np.random.default_rng(i).standard_normal((n, 3 * 72)).astype(np.float32)
        jobs.append((n, q, kc, vc, qkv, *(torch.from_numpy(a).cuda() for a in (q, kc, vc, qkv)),
                     torch.zeros((n, nh * hd), device="cuda"), torch.zeros((n, 72), device="cuda")))
    bias = torch.zeros(3 * 72, device="cuda")
    torch.cuda.synchronize()
    asc = np.float32(1.0) / np.sqrt(np.float32(hd))
    for i, (n, q, kc, vc, qkv, dq, dk, dv, dqkv, out, vout) in enumerate(jobs):
        s = streams[i % 2].cuda_stream
        gh.prefill_attention(out, dq, q.shape[1], dk, dv, n, 0, nh, nkv, hd, kc.shape[1], 0, asc,
                             0.0, False, 1, stream=s)
        gh.vision_attention(vout, dqkv, bias, n, 1, 72, 1, stream=s)
    torch.cuda.synchronize()
    for n, q, kc, vc, qkv, dq, dk, dv, dqkv, out, vout in jobs:
        _close(out.cpu().numpy(), _prefill_want(q, kc, vc, n, 0, nh, nkv, hd, 0, 0.0, False))
        _close(vout.cpu().numpy(), _vision_want(qkv, np.zeros(216, np.float32), 1, 72))
    n, q, kc, dq, dk, dv, out = (jobs[0][i] for i in (0, 1, 2, 5, 6, 7, 9))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=streams[0]):
        with pytest.raises(GemmaHipError, match="captured"):
            gh.prefill_attention(out, dq, q.shape[1], dk, dv, n, 0, nh, nkv, hd, kc.shape[1], 0,
                                 asc, 0.0, False, 1, stream=streams[0].cuda_stream)


@pytest.mark.gpu
def test_attention_workspace_grows_seldom(gh):
    """A prompt in 48 chunks, each behind the ones before: the workspace doubles
    a few times, where one that grew to each call's size would wait for the
    stream and allocate with nearly every chunk (2 MiB more each)."""
    import torch

    nh, nkv, hd, rows, chunks = 4, 4, 256, 256, 48
    q = torch.randn(rows, nh * hd, device="cuda")
    kc = torch.randn(nkv, rows * chunks, hd, device="cuda")
    out = torch.empty_like(q)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    sizes = []
    for i in range(chunks):
        gh.prefill_attention(out, q, nh * hd, kc, kc, rows, rows * i, nh, nkv, hd, rows * chunks, 0,
                             1 / 16, 0.0, False, 1, stream=stream.cuda_stream)
        sizes.append(torch.cuda.mem_get_info()[0])
    torch.cuda.synchronize()
    changes = sum(a != b for a, b in zip(sizes, sizes[1:]))
    print(f"{changes} allocations", flush=True)
    assert changes <= 8


@pytest.mark.gpu
@pytest.mark.parametrize("entry", ["vision", "prefill"])
def test_attention_beside_a_capture(gh, entry):
    """Eager attention on one stream while another is being captured (in the
    global mode): it may need its first workspace, gets it, and leaves the
    capture whole."""
    import torch

    rng = np.random.default_rng(11)
    n, heads, hd, nh, nkv = 300, 2, 72, 4, 2
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim)).astype(np.float32)
    bias = np.zeros(3 * dim, np.float32)
    q, kc, vc = _prefill_inputs(n, 0, nh, nkv, 128, seed=12)
    dqkv, db, dq, dk, dv = (torch.from_numpy(a).cuda() for a in (qkv, bias, q, kc, vc))
    x = torch.zeros(1000, device="cuda")
    out = torch.empty((n, dim if entry == "vision" else nh * 128), device="cuda")
    streams = [torch.cuda.Stream() for _ in range(2)]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=streams[0], capture_error_mode="global"):
        x += 1
        s = streams[1].cuda_stream
        if entry == "vision":
            gh.vision_attention(out, dqkv, db, n, heads, dim, 1, s)
        else:
            gh.prefill_attention(out, dq, q.shape[1], dk, dv, n, 0, nh, nkv, 128, kc.shape[1], 0,
                                 np.float32(1) / np.sqrt(np.float32(128)), 0.0, False, 1, stream=s)
        x += 2
    torch.cuda.synchronize()
    for i in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert (x == 3 * (i + 1)).all()
    _close(out.cpu().numpy(), _vision_want(qkv, bias, heads, dim) if entry == "vision" else
           _prefill_want(q, kc, vc, n, 0, nh, nkv, 128, 0, 0.0, False))


@pytest.mark.gpu
def test_per_thread_streams(gh):
    """hipStreamPerThread, one handle for a stream of each thread's own: calls
    that need workspaces (both attentions, int8 and fp32 split-K products) from
    four threads at once give what they give one after another."""
    import threading

    import torch

    per_thread = 2  # hipStreamPerThread
    nh, nkv, hd, m, n8, k8 = 4, 2, 128, 300, 640, 2064
    asc = np.float32(1) / np.sqrt(np.float32(hd))
    gen = torch.Generator(device="cuda").manual_seed(1)

    def inputs():
        r = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
        i8 = lambda *s: torch.randint(-127, 128, s, generator=gen, device="cuda",  # noqa: E731
                                      dtype=torch.int8)
        d = dict(q=r(400, nh * hd), kc=r(nkv, 400, hd), vc=r(nkv, 400, hd), qkv=r(400, 3 * 144),
                 a=r(64, 2048), b=r(512, 2048), a8=i8(m, k8), b8=i8(n8, k8), sa=r(m).abs(),
                 sb=r(n8).abs())
        d["out"] = [torch.zeros(s, device="cuda")
                    for s in ((400, nh * hd), (400, 144), (64, 512), (m, n8))]
        return d

    bias = torch.zeros(3 * 144, device="cuda")

    def calls(d):
        o = d["out"]
        gh.prefill_attention(o[0], d["q"], nh * hd, d["kc"], d["vc"], 400, 0, nh, nkv, hd, 400, 0,
                             asc, 0.0, False, 1, stream=per_thread)
        gh.vision_attention(o[1], d["qkv"], bias, 400, 2, 144, 1, per_thread)
        gh.matmul_f32(o[2], 512, d["b"], 2048, d["a"], 2048, 64, 512, 2048, per_thread)
        gh.matmul(o[3], n8, d["b8"], k8, d["sb"], d["a8"], k8, d["sa"], m, n8, k8, per_thread)

    jobs = [inputs() for _ in range(4)]
    torch.cuda.synchronize()
    want = []
    for d in jobs:
        calls(d)
        torch.cuda.synchronize()
        want.append([t.clone() for t in d["out"]])
        for t in d["out"]:
            t.zero_()
    torch.cuda.synchronize()
    errors = []

    def work(d):
        try:
            for _ in range(20):
                calls(d)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(d,)) for d in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for d, w in zip(jobs, want):
        assert all(torch.equal(a, b) for a, b in zip(d["out"], w))
    # and what they give is right
    d = jobs[0]
    _close(d["out"][0].cpu().numpy(),
           _prefill_want(d["q"].cpu().numpy(), d["kc"].cpu().numpy(), d["vc"].cpu().numpy(), 400, 0,
                         nh, nkv, hd, 0, 0.0, False))
    _close(d["out"][2].cpu().numpy(), (d["a"].double() @ d["b"].double().T).cpu().numpy())


def _rms(got, want):
    return float(np.linalg.norm(got - want) / np.linalg.norm(want))


# Where the errors of the two forms stand, as a guard against growth that the
# bars of single values would let through: two f16 pieces round each sum half as
# often as three bf16 pieces with six products, and stay below them (measured,
# split against three pieces: 4.3e-7 / 5.4e-7 over 1024 patches, 2.7e-7 / 3.3e-7 in
# a 300-row prompt).
@pytest.mark.gpu
@pytest.mark.parametrize("n,heads,hd", [(300, 2, 72), (1024, 2, 72), (1000, 2, 128), (600, 4, 64)])
def test_vision_error_level(gh, n, heads, hd):
    import torch

    rng = np.random.default_rng(n)
    dim = heads * hd
    qkv = rng.standard_normal((n, 3 * dim)).astype(np.float32)
    bias = (0.02 * rng.standard_normal(3 * dim)).astype(np.float32)
    want = _vision_want(qkv, bias, heads, dim)
    split = _rms(_vision(gh, qkv, bias, heads, dim), want)
    dq, db = torch.from_numpy(qkv).cuda(), torch.from_numpy(bias).cuda()
    out = torch.zeros((n, dim), device="cuda")
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        gh.vision_attention(out, dq, db, n, heads, dim, 1, side.cuda_stream)
    graph.replay()
    torch.cuda.synchronize()
    three = _rms(out.cpu().numpy(), want)
    print(f"split {split:.3g}, three pieces {three:.3g}", flush=True)
    assert split <= three


@pytest.mark.gpu
@pytest.mark.parametrize("n,pos0,nh,nkv,hd", [(300, 0, 4, 1, 256), (257, 500, 4, 1, 256),
                                              (500, 0, 4, 2, 128)])
def test_prefill_error_level(gh, monkeypatch, n, pos0, nh, nkv, hd):
    monkeypatch.setenv("GEMMA_HIP_PF_ATTN", "split")
    q, kc, vc = _prefill_inputs(n, pos0, nh, nkv, hd, seed=n)
    args = (n, pos0, nh, nkv, hd, 0, 0.0, False)
    split = _rms(_prefill(gh, q, kc, vc, *args), _prefill_want(q, kc, vc, *args))
    vc[:, 0:pos0 + n:32] = 0  # a zero key in every tile: three pieces
    three = _rms(_prefill(gh, q, kc, vc, *args), _prefill_want(q, kc, vc, *args))
    print(f"split {split:.3g}, three pieces {three:.3g}", flush=True)
    assert split <= three
