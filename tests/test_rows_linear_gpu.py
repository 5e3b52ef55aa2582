"""Projections of many rows (skv_rows_linear) against float64: bias, GELU, residual, and q/k/v columns by head.

Sizes sit at the edges of the kernel's 64- to 192-row tiles and 128-byte steps; the last four of SIZES and the two of
MORE_TILES take its larger tiles. The bar is the output's rounding plus the fp32 accumulation bound k * 2^-24 * sum |x w|.
"""
import pytest
import torch
import torch.nn.functional as F

from speech_serving import models, native

pytestmark = pytest.mark.gpu

EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}
SIZES = [(1, 8, 8), (63, 64, 64), (64, 72, 72), (65, 128, 136), (129, 200, 1288), (300, 1288, 200), (1000, 136, 2056),
         (1500, 1280, 1280), (1500, 3840, 1288), (1500, 5120, 1280), (1300, 8200, 640)]

MORE_TILES = [(1801, 1072, 328), (1751, 3272, 328)]  # 128 x 64 and 128 x 192 outputs, the last tiles nearly empty


def _data(m, n, k, dt):
    g = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
    x, r = (torch.randn(m, c, generator=g, device="cuda").to(dt) for c in (k, n))
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dt)
    b = torch.randn(n, generator=g, device="cuda").to(dt)
    ref = x.double() @ w.double().t()
    bound = k * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    return x, w, b, r, ref, bound


def _check(y, ref, bound, what):
    err = (y.double() - ref).abs()
    tol = EPS[y.dtype] * ref.abs() + bound + 1e-6
    assert bool((err <= tol).all()), f"{what}: max excess {float((err - tol).max()):.3g}"


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("size", SIZES)
def test_rows_linear_against_float64(cuda, dt, size):
    x, w, b, r, ref, bound = _data(*size, dt)
    few = 2.0 ** -21 * (ref.abs() + b.double().abs() + r.double().abs())
    _check(native.rows_linear(x, w), ref, bound, "plain")
    _check(native.rows_linear(x, w, b, res=r), ref + b.double() + r.double(), bound + few, "bias, residual")
    pre = ref + b.double()
    y = native.rows_linear(x, w, b, gelu=True)
    if y is None:  # the library and a GELU launch are the faster way
        assert size[0] > 1000
        y = models._linear(x, w, b, gelu=True)
        bound = 2 * bound + 2 * EPS[dt] * pre.abs()  # it rounds before the GELU too
    _check(y, F.gelu(pre), 1.13 * bound + few, "gelu")


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,s,heads,k", [(1, 130, 6, 384), (3, 67, 4, 256), (1, 1500, 20, 1280), (2, 1, 1, 64)])
def test_qkv_columns_by_head(cuda, dt, b, s, heads, k):
    x, w, _, _, ref, bound = _data(b * s, 3 * heads * 64, k, dt)
    q, kk, v = native.rows_qkv(x.view(b, s, k), w, heads)
    ref, bound = (t.view(b, s, 3, heads, 64) for t in (ref, bound))
    _check(q, ref[:, :, 0], bound[:, :, 0], "q")
    for got, i in ((kk, 1), (v, 2)):
        assert got.shape == (b, heads, s, 64) and got.is_contiguous()
        _check(got.transpose(1, 2), ref[:, :, i], bound[:, :, i], "kv"[i - 1])


def test_strides_and_refused_calls(cuda):
    x, w, b, r, ref, bound = _data(140, 256, 512, torch.bfloat16)
    big = torch.full((140, 640), float("nan"), device="cuda", dtype=torch.bfloat16)
    big[:, 64:576] = x
    _check(native.rows_linear(big[:, 64:576], w), ref, bound, "strided")
    wide = torch.full((256, 520), float("nan"), device="cuda", dtype=torch.bfloat16)
    wide[:, :512] = w
    _check(native.rows_linear(x, wide[:, :512]), ref, bound, "strided weight")
    assert native.rows_linear(x.view(4, 35, 512), w).shape == (4, 35, 256)
    for bad in ((x[:, :500], w[:, :500], None), (x[:, 1:505], w[:, :504], None), (x, w[:252], None), (x, w, b.float()),
                (x.float(), w.float(), None), (x[:1].expand(140, 512), w, b)):
        assert native.rows_linear(*bad) is None
    assert native.rows_linear(x, w, b, res=r[:, :128]) is None
    y = models._linear(x.float(), w.float(), b.float(), gelu=True)  # served by the library GEMM
    assert torch.allclose(y.double(), F.gelu(ref + b.double()), rtol=1e-3, atol=1e-3)
    x[77, 3] = float("nan")  # reaches its own row only
    assert torch.isnan(native.rows_linear(x, w)).any(dim=1).nonzero().flatten().tolist() == [77]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("size", MORE_TILES)
def test_rows_linear_over_the_other_tiles(cuda, dt, size):
    x, w, b, r, ref, bound = _data(*size, dt)
    few = 2.0 ** -21 * (ref.abs() + b.double().abs() + r.double().abs())
    _check(native.rows_linear(x, w), ref, bound, "plain")
    _check(native.rows_linear(x, w, b, res=r), ref + b.double() + r.double(), bound + few, "bias, residual")
