"""Causal prompts (with and without a fused append) on the matrix-core kernels against float64.

The sizes are those that leave the one-workgroup-per-query kernel: tiles of 16 and of 64 queries, one wave and four per
tile, pool keys and new keys in the same row, rows shorter than their queries, split rows with partials, grouped KV
heads, invalid block ids, and K/V values that are not finite.
"""
import math

import pytest
import torch

from speech_serving import native

pytestmark = pytest.mark.gpu

D = 64
EPS = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _reference(q, ctx, keys, causal, scale):
    """Float64 output [B, Q, H, D]; keys(b, kvh) -> (K [T, D], V [T, D], valid [T]) over the row's ctx keys."""
    b, nq, h, _ = q.shape
    out = torch.zeros(q.shape, dtype=torch.float64)
    for r in range(b):
        for i in range(h):
            k, v, ok = keys(r, i)
            for qi in range(nq):
                seen = max(0, ctx[r] - (nq - 1 - qi)) if causal else ctx[r]
                sel = torch.nonzero(ok[:seen])[:, 0]
                if len(sel) == 0:
                    continue
                p = torch.softmax(k[sel] @ q[r, qi, i] * scale, 0)
                out[r, qi, i] = p @ v[sel]
    return out


def _paged(cuda, dt, q_len, past, heads, kv_heads, bs, bad_blocks=0, chunk=0, causal=True, fused=True, poison=None,
           short=()):
    g = torch.Generator().manual_seed(q_len * 131 + heads)
    b = len(past)
    ctx = [p + q_len for p in past]
    for r, c in short:  # rows with fewer keys than queries
        ctx[r] = c
    width = -(-max(max(ctx), 1) // bs)
    nb = b * width + 2
    kp, vp = (torch.randn(nb, bs, kv_heads, D, generator=g).to(dt) for _ in range(2))
    tables = torch.randperm(nb, generator=g)[: b * width].view(b, width).to(torch.int32)
    for i in range(bad_blocks):
        tables[i % b, (3 * i) % width] = [-1, nb, 2 ** 30][i % 3]
    q, kn, vn = (torch.randn(b, q_len, n, D, generator=g).to(dt) for n in (heads, kv_heads, kv_heads))
    if poison is not None:
        row, tok, value = poison
        vn[row, tok, :, 5] = value
    dev = [t.to(cuda) for t in (q, kp, vp, tables, kn, vn)]
    lens = torch.tensor(ctx, dtype=torch.int32, device=cuda)
    new = dict(k_new=dev[4], v_new=dev[5]) if fused else {}
    out = native.paged_attention(dev[0], dev[1], dev[2], dev[3], lens, width * bs, D ** -0.5, causal=causal,
                                 chunk_tokens=chunk, **new).cpu()
    torch.cuda.synchronize()
    want_k, want_v = kp.clone(), vp.clone()

    def keys(r, i):
        kvh = i // (heads // kv_heads)
        n = ctx[r]
        k, v, ok = torch.zeros(n, D, dtype=torch.float64), torch.zeros(n, D, dtype=torch.float64), torch.ones(n, dtype=bool)
        for t in range(n):
            blk = int(tables[r, t // bs])
            src = t - (n - q_len)
            if fused and src >= 0:
                k[t], v[t] = kn[r, src, kvh].double(), vn[r, src, kvh].double()
            elif 0 <= blk < nb:
                k[t], v[t] = kp[blk, t % bs, kvh].double(), vp[blk, t % bs, kvh].double()
            else:
                ok[t] = False
        return k, v, ok

    if fused:
        for r in range(b):
            for i in range(q_len):
                t = ctx[r] - q_len + i
                blk = int(tables[r, t // bs]) if t >= 0 else -1
                if 0 <= blk < nb:
                    want_k[blk, t % bs], want_v[blk, t % bs] = kn[r, i], vn[r, i]
        assert torch.equal(dev[1].cpu().view(torch.int16), want_k.view(torch.int16))
        assert torch.equal(dev[2].cpu().view(torch.int16), want_v.view(torch.int16))
    want = _reference(q.double(), ctx, keys, causal, D ** -0.5)
    return out.double(), want, EPS[dt]


def _close(out, want, eps):
    # one rounding of the output; scores and weights in fp32
    err = (out - want).abs()
    assert bool((err <= 2 * eps * want.abs() + 1e-4).all()), f"max err {float(err.max()):.2e}"


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("q_len,past,heads,kv_heads,bs", [
    (4, [0] * 32, 8, 8, 16),                    # one wave per tile: the start prompt
    (17, [0, 3, 15, 0], 20, 4, 8),              # two tiles, grouped KV heads, keys past one step
    (32, [0, 0, 0, 0], 8, 8, 16),               # the longest one-wave prompt
    (33, [7, 0, 64, 31], 8, 2, 32),             # four waves; pool keys and new keys
    (64, [0, 1, 63, 64, 200], 48, 12, 16),      # one 64-query tile
    (130, [0, 37, 190], 24, 8, 16),             # three 64-query tiles, the last nearly empty
])
def test_causal_prompt_with_fused_append(cuda, dt, q_len, past, heads, kv_heads, bs):
    _close(*_paged(cuda, dt, q_len, past, heads, kv_heads, bs))


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
def test_prompt_forms(cuda, dt):
    past = [40, 9, 0, 100]
    _close(*_paged(cuda, dt, 20, past, 16, 4, 16, short=[(1, 0), (2, 7)]))           # fewer keys than queries
    _close(*_paged(cuda, dt, 70, past, 32, 16, 16, short=[(1, 0), (2, 33)]))
    _close(*_paged(cuda, dt, 20, past, 16, 4, 16, bad_blocks=5))                     # old and new blocks invalid
    _close(*_paged(cuda, dt, 70, past, 32, 16, 16, bad_blocks=7))
    _close(*_paged(cuda, dt, 20, [300, 290, 17], 20, 20, 16, chunk=64))              # split rows, partials merged
    _close(*_paged(cuda, dt, 20, past, 16, 4, 16, fused=False))                      # causal, keys all in the pool
    _close(*_paged(cuda, dt, 70, past, 32, 16, 16, fused=False))
    _close(*_paged(cuda, dt, 20, past, 16, 4, 16, causal=False))                     # every query sees the new keys
    _close(*_paged(cuda, dt, 70, past, 32, 16, 16, causal=False))


@pytest.mark.parametrize("value", [math.inf, -math.inf, math.nan])
@pytest.mark.parametrize("q_len,heads,chunk", [(4, 128, 0), (20, 20, 0), (20, 20, 64), (70, 40, 0)])
def test_a_value_that_is_not_finite_reaches_only_the_queries_that_see_it(cuda, value, q_len, heads, chunk):
    tok = q_len - 2
    past = [0, 0] if q_len == 4 else [30, 0, 50] if chunk == 0 else [230, 0, 150]
    out, want, eps = _paged(cuda, torch.bfloat16, q_len, past, heads, heads, 16, chunk=chunk, poison=(0, tok, value))
    fine = torch.isfinite(want)
    assert not bool(fine[0, tok:, :, 5].any()) and bool(fine[0, :tok].all()) and bool(fine[1:].all())
    assert torch.equal(torch.isfinite(out), fine)
    _close(out[fine], want[fine], eps)


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("q_len,t,b,heads", [(20, 20, 4, 16), (20, 90, 4, 16), (65, 65, 4, 32), (128, 200, 3, 32)])
def test_causal_prompt_over_contiguous_rows(cuda, dt, q_len, t, b, heads):
    g = torch.Generator().manual_seed(t)
    q = torch.randn(b, q_len, heads, D, generator=g).to(dt)
    k, v = (torch.randn(b, heads, t, D, generator=g).to(dt) for _ in range(2))
    lens = [t, max(1, t - 13), q_len, 0][:b]
    out = native.dense_attention(q.to(cuda), k.to(cuda), v.to(cuda), torch.tensor(lens, dtype=torch.int32, device=cuda),
                                 t, D ** -0.5, causal=True).cpu()
    want = _reference(q.double(), lens, lambda r, i: (k[r, i].double(), v[r, i].double(), torch.ones(t, dtype=bool)),
                      True, D ** -0.5)
    _close(out.double(), want, EPS[dt])


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("b,n,h", [(128, 4, 20), (16, 33, 20), (8, 201, 20)])
def test_weights_of_prompts_have_fp32s_bits(cuda, dt, b, n, h):
    """Sums that cancel show the weights' own error: key 0 (V = 0) holds the maximum, the others weigh about 0.7 of it, V is
    +-1 in pairs, and only outputs below 2^-13 of sum p |v| count (their rounding is 2^-22 of it or less). Each weight
    carries the errors of its score and exponent (about 2^-24) and averages with the other 4 to 201; weights of 16 bits
    gave 1.5 to 2 times the bar, of 22 bits 1.2 times."""
    g = torch.Generator(device="cuda").manual_seed(n)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    q = torch.cat([torch.ones(b, n, h, 1, device="cuda"), rn(b, n, h, D - 1) * 0.002], -1).to(dt)
    k = torch.cat([torch.zeros(b, n, h, 1, device="cuda"), rn(b, n, h, D - 1) * 0.05], -1).to(dt)
    k[:, 0, :, 0] = 2.9
    v = rn(b, (n + 1) // 2, h, D).sign().repeat_interleave(2, 1)[:, :n]
    v[:, 1::2] *= -1
    v = v.roll(1, 1)
    v[:, 0] = 0
    v = v.to(dt)
    width = -(-n // 16)
    kp, vp = (torch.zeros(b * width, 16, h, D, device="cuda", dtype=dt) for _ in range(2))
    tables = torch.arange(b * width, device="cuda", dtype=torch.int32).view(b, width)
    lens = torch.full((b,), n, dtype=torch.int32, device="cuda")
    out = native.paged_attention(q, kp, vp, tables, lens, width * 16, D ** -0.5, causal=True, k_new=k, v_new=v).double()
    s = torch.matmul(q.double().transpose(1, 2), k.double().permute(0, 2, 3, 1).contiguous()) * D ** -0.5
    p = torch.softmax(s.masked_fill(torch.ones(n, n, device="cuda").triu(1) > 0, -math.inf), -1)
    want, size = (torch.matmul(p, t.double().transpose(1, 2)).transpose(1, 2) for t in (v, v.abs()))
    sel = (want.abs() < 2.0 ** -13 * size) & (size > 0)
    err = ((out - want).abs() / size)[sel]
    assert err.numel() > 100000
    bar = {torch.float16: {4: 3.9e-8, 33: 2.45e-8, 201: 1.93e-8}, torch.bfloat16: {4: 1.3e-7, 33: 7e-8, 201: 3.6e-8}}[dt][n]
    assert float(err.square().mean().sqrt()) < bar
