"""Decode-batch projections (skv_decode_linear, its partials, skv_reduce_add_layernorm) against float64.

Sizes sit at the edges of the kernel's tiles (16 to 64 rows, 16 or 32 columns), of its 128-byte chunks and of its
split (6 KiB rows). The bar is the output's rounding plus the fp32 accumulation bound k * 2^-24 * sum |x w|.
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
# 256 (one chunk per wave), 264 and 776 (partial last chunks), 1280 (8 waves, 3 rounds, a partial round), 2048 (4 rounds),
# 2056 and 3072 (5 and 6 rounds, tiles of at most 32 rows)
MN = [(1, 4), (1, 1284), (9, 20), (16, 16), (17, 36), (33, 132), (64, 1280), (65, 3840), (128, 1056), (300, 260)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k16", [256, 264, 776, 1280, 2048, 2056, 3072])
def test_decode_linear_against_float64(cuda, dt, k16):
    k = k16 if dt != torch.float32 else k16 // 2
    for m, n in MN:
        if m > 128 and k16 > 2048:
            continue  # a longer row takes a decode batch only
        x, w, b, ref, bound = _data(m, n, k, dt, m * 7 + n)
        _check(native.decode_linear(x, w, b), ref, bound, f"m={m} n={n} k={k}")
        y = native.decode_linear(x, w, b, gelu=True)
        # |GELU'| < 1.13; erf and the products add a few fp32 roundings of |pre|
        _check(y, F.gelu(ref), 1.13 * bound + 2.0 ** -20 * ref.abs(), f"gelu m={m} n={n} k={k}")


@pytest.mark.parametrize("dt,k", [(torch.bfloat16, 3080), (torch.float16, 5120), (torch.float32, 1540)])
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


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d", [256, 384, 768, 1280])
def test_residual_and_normed_projection(cuda, dt, d):
    """A residual projection, then a projection of its LayerNorm, in one launch each."""
    if dt == torch.float32 and d == 1280:
        d = 1024  # the longest unsplit fp32 row
    for m, n in [(1, 256), (4, 3 * d), (17, 512), (33, 1040), (64, 4 * d), (128, 4)]:
        a, w, b, ref, bound = _data(m, d, d, dt, m + n)
        g = torch.Generator(device="cuda").manual_seed(m)
        res = (3 * torch.randn(m, d, generator=g, device="cuda") + 5).to(dt)  # a mean well off zero
        s, stats = native.decode_linear_residual(a, w, b, res)
        _check(s, ref + res.double(), bound + 2.0 ** -23 * (ref.abs() + res.double().abs()), f"residual m={m} d={d}")
        grp = s.double().view(m, d // 16, 16)
        assert torch.allclose(stats[..., 0].double(), grp.sum(-1), rtol=1e-5, atol=1e-4)
        dev = (grp - grp.mean(-1, keepdim=True)).square().sum(-1)
        assert torch.allclose(stats[..., 1].double(), dev, rtol=1e-5, atol=1e-4)
        gm, bt = (torch.randn(d, generator=g, device="cuda").to(dt) for _ in range(2))
        w2 = (torch.randn(n, d, generator=g, device="cuda") * d ** -0.5).to(dt)
        b2 = torch.randn(n, generator=g, device="cuda").to(dt)
        want = F.layer_norm(s.double(), (d,), gm.double(), bt.double(), 1e-5)
        for gelu in (False, True):
            y = native.decode_linear_normed(s, stats, gm, bt, 1e-5, w2, b2, gelu)
            if y is None:  # a tile of 64 rows, or more workgroups than units
                assert m * n > 16 * 256 * 16 * 4
                break
            ref2 = want @ w2.double().t() + b2.double()
            # each normalised element rounded to dtype (and a few fp32 roundings), then the product's own bound
            slack = (2 * EPS[dt] + (d + 8) * 2.0 ** -24) * (want.abs() + 1e-2) @ w2.double().abs().t() + 1e-6
            _check(y, F.gelu(ref2) if gelu else ref2, 1.13 * slack + 2.0 ** -20 * ref2.abs(), f"normed m={m} n={n} d={d}")
        full = native.decode_linear_normed(s, stats, gm, bt, 1e-5, w2, b2)
        if full is None:
            continue
        assert torch.equal(native.decode_linear_normed(s[:1], stats[:1].contiguous(), gm, bt, 1e-5, w2, b2), full[:1])


def test_fused_projection_refuses_what_it_does_not_take(cuda):
    a, w, b, _, _ = _data(8, 512, 512, torch.bfloat16, 1)
    res = torch.zeros(8, 512, device="cuda", dtype=torch.bfloat16)
    assert native.decode_linear_residual(a, w[:500], None, res[:, :500]) is None  # columns not whole groups of 16
    assert native.decode_linear_residual(a, w, None, res.float()) is None
    assert native.decode_linear_residual(a, w, None, res[:4]) is None
    big = torch.zeros(129, 512, device="cuda", dtype=torch.bfloat16)
    s, st = native.decode_linear_residual(big, w, None, big)
    assert native.decode_linear_normed(s, st, b, b, 1e-5, w) is None  # past the decode batch
    assert native.decode_linear_normed(s[:8], st[:8], b[1:], b, 1e-5, w) is None
    assert native.decode_linear_normed(s[:8], st[:7], b, b, 1e-5, w) is None
    nan = a.clone()
    nan[3, 7] = float("nan")  # reaches its own row only
    s, st = native.decode_linear_residual(nan, w, b, res)
    y = native.decode_linear_normed(s, st, b, b, 1e-5, w)
    bad = torch.isnan(y).any(dim=1)
    assert bool(bad[3]) and int(bad.sum()) == 1


def test_fp32_gelu_is_as_exact_as_torch(cuda):
    """Over identity weights the products are x itself, so the GELU's own error shows: on every interval at most torch's
    (x / 2 (1 + erff), to a percent for another erff), which is the smallest near zero."""
    g = torch.Generator(device="cuda").manual_seed(1)
    w = torch.eye(128, device="cuda")
    for lo, hi in ((0.0, 0.1), (0.1, 0.3), (0.3, 1.0), (1.0, 2.0), (2.0, 4.0), (4.0, 9.0)):
        for sign in (-1.0, 1.0):
            x = sign * (lo + (hi - lo) * torch.rand(128, 128, generator=g, device="cuda"))
            want = F.gelu(x.double())
            err, ref = ((y.double() - want) / want.abs().clamp_min(1e-30) for y in (native.decode_linear(x, w, gelu=True), F.gelu(x)))
            assert float(err.norm()) <= 1.01 * float(ref.norm()), (sign * lo, sign * hi)
            assert float(err.abs().max()) <= 1.01 * float(ref.abs().max()), (sign * lo, sign * hi)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
def test_normed_projection_is_as_exact_as_the_layernorm_launch(cuda, dt):
    """Over identity weights, for rows whose mean is up to 400 times their spread: the error against float64 is at most a
    percent above that of the LayerNorm launch (in fp32, where the mean's rounding is all there is, a tenth)."""
    for mean, d in ((0, 512), (8, 512), (64, 256), (64, 1024), (400, 1024)):
        g = torch.Generator(device="cuda").manual_seed(mean + d)
        res = (torch.randn(64, d, generator=g, device="cuda") + mean).to(dt)
        zeros, one, eye = (t.to("cuda", dt) for t in (torch.zeros(64, 256), torch.ones(d), torch.eye(d)))
        s, stats = native.decode_linear_residual(zeros, zeros.new_zeros(d, 256), None, res)
        assert torch.equal(s, res)
        want = F.layer_norm(s.double(), (d,), eps=1e-5)
        y = native.decode_linear_normed(s, stats, one, zeros.new_zeros(d), 1e-5, eye)
        n = native.add_layernorm(s, None, one, zeros.new_zeros(d), 1e-5)[1]
        err, ref = (float((t.double() - want).norm()) for t in (y, n))
        assert err <= (1.1 if dt == torch.float32 else 1.01) * ref, (mean, d, err, ref)


# 31 x 2052 and 31 x 4100 outputs take tiles of 32 x 16 and 32 x 32, 64 x 4100 of 64 x 32; k (16-bit) one length for each of the
# kernel's wave and round counts, with a partial last chunk or round where there is room for one
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("k16", [256, 480, 768, 992, 1280, 2048])
def test_every_tile_plain_and_normed(cuda, dt, k16):
    k = k16 if dt != torch.float32 else k16 // 2
    g = torch.Generator(device="cuda").manual_seed(k16)
    zeros = torch.zeros(64, 256, device="cuda", dtype=dt)
    gm, bt = (torch.randn(k, generator=g, device="cuda").to(dt) for _ in range(2))
    for m, n in ((16, 20), (31, 2052), (31, 4100), (64, 4100)):
        x, w, b, ref, bound = _data(m, n, k, dt, m + n)
        _check(native.decode_linear(x, w, b), ref, bound, f"m={m} n={n} k={k}")
        s, stats = native.decode_linear_residual(zeros[:m], zeros.new_zeros(k, 256), None, x)
        assert torch.equal(s, x)
        y = native.decode_linear_normed(s, stats, gm, bt, 1e-5, w, b)
        assert (y is None) == (m == 64)  # tiles of 64 rows leave the LayerNorm to a launch
        if y is not None:
            want = F.layer_norm(s.double(), (k,), gm.double(), bt.double(), 1e-5)
            # each normalised element rounded to dtype (and a few fp32 roundings), then the product's own bound
            slack = (2 * EPS[dt] + (k + 8) * 2.0 ** -24) * (want.abs() + 1e-2) @ w.double().abs().t() + 1e-6
            ref = want @ w.double().t() + b.double()
            _check(y, ref, slack + 2.0 ** -20 * ref.abs(), f"normed m={m} n={n} k={k}")
