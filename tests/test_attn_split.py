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
