"""fp32 attention of several queries over contiguous K/V (encoder layers, a prompt's cross-attention) against float64.

Sizes sit at the edges of the kernel's 16-query tiles, 16-key steps and of the wave counts it picks by grid size. The bar is the
fp32 bound of the scores (64 products, |s| up to about 30 here) carried through the softmax, and of the sum over keys.
"""
import math

import pytest
import torch

from speech_serving import native

pytestmark = pytest.mark.gpu


def _reference(q, k, v, lens, scale):
    out = torch.zeros_like(q, dtype=torch.float64)
    group = q.shape[2] // k.shape[1]
    for b, n in enumerate(lens):
        if n:
            kk, vv = (t[b, :, :n].double().repeat_interleave(group, 0) for t in (k, v))
            s = torch.matmul(q[b].double().transpose(0, 1), kk.transpose(1, 2).contiguous()) * scale
            out[b] = torch.matmul(torch.softmax(s, -1), vv).transpose(0, 1)
    return out


# (batch, queries, heads, kv heads, keys)
# From 200 Ki query-key pairs on the matrix-core kernel runs (4, 8 or 16 waves by the number of tiles); the first two stay below.
@pytest.mark.parametrize("b,nq,h,hkv,t", [(1, 2, 1, 1, 1), (1, 17, 6, 6, 300), (400, 16, 33, 33, 1), (64, 17, 12, 4, 16),
                                          (70, 15, 12, 12, 17), (16, 16, 13, 13, 65), (40, 2, 20, 20, 129),
                                          (2, 40, 20, 4, 129), (1, 300, 6, 6, 300), (1, 600, 12, 12, 600)])
@pytest.mark.parametrize("scale", [0.125, -0.3])
def test_against_float64(cuda, b, nq, h, hkv, t, scale):
    g = torch.Generator(device="cuda").manual_seed(b + nq + t)
    q = torch.randn(b, nq, 3 * h * 64, generator=g, device="cuda")[..., h * 64:2 * h * 64].view(b, nq, h, 64)  # strided rows
    k, v = (torch.randn(b, hkv, t, 64, generator=g, device="cuda") for _ in range(2))
    lens = [t] + [max(0, t - 7 * i) if i % 5 else 0 for i in range(1, b)]
    for i, n in enumerate(lens):  # what lies past a row's length is never used
        k[i, :, n:], v[i, :, n:] = float("nan"), float("inf")
    out = native.dense_attention(q, k, v, torch.tensor(lens, dtype=torch.int32, device="cuda"), t, scale)
    err = (out.double() - _reference(q, k, v, lens, scale)).abs()
    smax = abs(scale) * 64 * 1.5
    assert float(err.max()) < (2 * smax + math.sqrt(t) + 16) * 2.0 ** -24 * float(v[torch.isfinite(v)].abs().max())


def test_slots_nan_rows_and_token_major_keys(cuda):
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(2, 130, 16, 64, generator=g, device="cuda")
    kv = torch.randn(2, 5, 50, 16, 64, generator=g, device="cuda")  # [k/v, slots, tokens, heads, 64]
    k, v = (x.transpose(1, 2) for x in kv)
    slots = torch.tensor([4, 1], dtype=torch.int32, device="cuda")
    lens = torch.tensor([50, 33], dtype=torch.int32, device="cuda")
    ref = _reference(q, k[[4, 1]], v[[4, 1]], [50, 33], 0.125)
    out = native.dense_attention(q, k, v, lens, 50, 0.125, slot_ids=slots)
    assert float((out.double() - ref).abs().max()) < 1e-5
    q[1, 7, 2, 5] = float("nan")  # reaches its own query and head only
    bad = torch.isnan(native.dense_attention(q, k, v, lens, 50, 0.125, slot_ids=slots)).any(-1).nonzero().tolist()
    assert bad == [[1, 7, 2]]
