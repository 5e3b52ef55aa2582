"""Decode-batch projections (skv_decode_linear, its partials, skv_reduce_add_layernorm) against float64.

Sizes sit at the edges of the kernel's tiles (16 to 64 rows, 16 or 32 columns), of its 128-byte chunks and of its
split (4 KiB rows). The bar is the output's rounding plus the fp32 accumulation bound k * 2^-24 * sum |x w|.
"""
import copy

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from speech_serving import models, native

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _data(m, n, k, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k, generator=g, device="cuda").to(dt)
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dt)
    b = torch.randn(n, generator=g, device="cuda").to(dt)
    ref = x.double() @ w.double().t() + b.double()
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t() + b.double().abs())
    return x, w, b, ref, bound


def _check(y, ref, bound, what):
    err = (y.double() - ref).abs()
    tol = EPS[y.dtype] * ref.abs() + bound + 1e-30
    assert bool((err <= tol).all()), f"{what}: max excess {float((err - tol).max()):.3g}"


# (m, n) around the row and column tiles and the one-workgroup-per-unit rule; k in elements of a 16-bit dtype:
# 256 (one chunk per wave), 264 and 776 (partial last chunks), 1280 (8 waves, 3 rounds, a partial round), 2048 (4 rounds)
MN = [(1, 4), (1, 1284), (9, 20), (16, 16), (17, 36), (33, 132), (64, 1280), (65, 3840), (128, 1056), (300, 260)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k16", [256, 264, 776, 1280, 2048])
def test_decode_linear_against_float64(cuda, dt, k16):
    k = k16 if dt != torch.float32 else k16 // 2
    for m, n in MN:
        x, w, b, ref, bound = _data(m, n, k, dt, m * 7 + n)
        _check(native.decode_linear(x, w, b), ref, bound, f"m={m} n={n} k={k}")
        y = native.decode_linear(x, w, b, gelu=True)
        # |GELU'| < 1.13; erf and the products add a few fp32 roundings of |pre|
        _check(y, F.gelu(ref), 1.13 * bound + 2.0 ** -20 * ref.abs(), f"gelu m={m} n={n} k={k}")


@pytest.mark.parametrize("dt,k", [(torch.bfloat16, 2056), (torch.float16, 5120), (torch.float32, 1536)])
def test_partials_and_reduce_add_layernorm(cuda, dt, k):
    for m, n in [(1, 256), (17, 384), (64, 1280), (128, 4096 if dt != torch.float32 else 2048)]:
        x, w, b, ref, bound = _data(m, n, k, dt, m + n)
        assert native.decode_linear(x, w, b) is None  # a split contraction
        p = native.decode_partials(x, w, b)
        assert p.part.shape[0] > 1
        _check(p.tensor(), ref, bound, f"sum m={m} n={n}")
        r, gm, bt = (torch.randn(s, device="cuda").to(dt) for s in ((m, n), (n,), (n,)))
        s, h = native.reduce_add_layernorm(p, r, gm, bt, 1e-5)
        _check(s, ref + r.double(), bound + 2.0 ** -23 * (ref.abs() + r.double().abs()), f"residual m={m} n={n}")
        want = F.layer_norm(s.double(), (n,), gm.double(), bt.double(), 1e-5)
        # the bar of the plain residual add + LayerNorm
        err = (h.double() - want).abs()
        assert bool((err <= 1e-5 + 2 * EPS[dt] * want.abs() + (1e-3 if dt != torch.float32 else 1e-5)).all())


def test_rows_do_not_depend_on_the_batch(cuda):
    for n, k in [(3840, 1280), (768, 768), (256, 256)]:
        x, w, b, _, _ = _data(128, n, k, torch.bfloat16, n)
        full = native.decode_linear(x, w, b)
        for m in (1, 8, 17, 64):
            assert torch.equal(native.decode_linear(x[:m], w, b), full[:m]), f"n={n} k={k} m={m}"
    x, w, b, _, _ = _data(128, 1280, 5120, torch.bfloat16, 5)
    full = native.decode_partials(x, w, b).tensor()
    assert torch.equal(native.decode_partials(x[:9], w, b).tensor(), full[:9])


def test_strided_rows_batch_dims_and_refused_calls(cuda):
    x, w, b, ref, bound = _data(24, 256, 512, torch.bfloat16, 3)
    big = torch.full((24, 640), float("nan"), device="cuda", dtype=torch.bfloat16)
    big[:, 64:576] = x
    xs = big[:, 64:576]  # rows 640 elements apart, NaN around them
    _check(native.decode_linear(xs, w, b), ref, bound, "strided")
    assert native.decode_linear(x.view(4, 6, 512), w, b).shape == (4, 6, 256)
    assert native.decode_linear(x[:0], w, b).shape == (0, 256)
    for bad in ((x[:, :500], w[:, :500], None), (x[:, 1:505], w[:, :504], None), (x, w[:255], None),
                (x[:, :128], w[:, :128], None), (x[:1].expand(24, 512), w, b), (x, w.float(), None),
                (x.expand(64, 24, 512), w, b)):
        assert native.decode_linear(*bad) is None
        y = models._linear(*bad) if bad[1].dtype == bad[0].dtype else None  # served by the library GEMM
        assert y is None or y.shape[-1] == bad[1].shape[0]


def test_mlp_in_a_graph_replays(cuda):
    torch.manual_seed(1)
    dt = torch.bfloat16
    seq = nn.Sequential(nn.Linear(768, 3072), nn.GELU(), nn.Linear(3072, 768)).to("cuda", dt)
    x = torch.randn(20, 768, device="cuda").to(dt)
    seq64 = copy.deepcopy(seq).double()
    with torch.no_grad():
        models.mlp(seq, x)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = models.mlp(seq, x)
        for seed in range(3):
            x.copy_(torch.randn(20, 768, generator=torch.Generator().manual_seed(seed)).to(dt))
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, models.mlp(seq, x))
            want = seq64(x.double())
            assert float((y.double() - want).norm() / want.norm()) < 2 * EPS[dt]
