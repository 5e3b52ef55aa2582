"""Decoder layers outside the usual form (replaced or wrapped modules, unusual operands) against float64 torch.

The layers serve their usual modules and operands in fused native launches. Everything else has to reach the module a
user put there, with the tensors that it would see in plain torch.
"""
import copy
import types

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from speech_serving import models, native
from speech_serving.models import CrossKV, DecoderLayer, PagedKV

pytestmark = pytest.mark.gpu

D, HEADS = 128, 2
EPS = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 2.0 ** -24}


def _attend(q, k, v, causal, keep=None):
    """softmax(q k^T / 8) v of q [B, S, H, 64] over k, v [B, H, T, 64], in float64; keep [B, T]."""
    s = torch.matmul(q.transpose(1, 2), k.transpose(2, 3).contiguous()) / 8.0
    if causal:
        s = s.masked_fill(torch.ones(s.shape[-2:], device=s.device).triu(1 + s.shape[-1] - s.shape[-2]) > 0, -torch.inf)
    if keep is not None:
        s = s.masked_fill(~keep[:, None, None, :], -torch.inf)
    return torch.matmul(torch.softmax(s, -1), v).transpose(1, 2)


@torch.no_grad()
def _reference(layer, x, cross=None, keep=None, cross_keep=None):
    """(output, k, v) of the layer in float64, its modules called as they stand; cross: encoder states [B, T, D]."""
    m = copy.deepcopy(layer).double()
    x = x.double()
    b, s, _ = x.shape
    split = lambda t: t.view(t.shape[0], t.shape[1], m.num_heads, 64)  # noqa: E731
    h = m.norm1(x)
    q, k, v = (split(mod(h)) for mod in (m.self_attn_q, m.self_attn_k, m.self_attn_v))
    k, v = k.transpose(1, 2), v.transpose(1, 2)
    x = x + m.self_attn_out(_attend(q, k, v, m.is_decoder, keep).reshape(b, s, -1))
    h = m.norm2(x)
    if cross is not None:
        ck, cv = (split(mod(cross.double())).transpose(1, 2) for mod in (m.cross_attn_k, m.cross_attn_v))
        x = x + m.cross_attn_out(_attend(split(m.cross_attn_q(h)), ck, cv, False, cross_keep).reshape(b, s, -1))
        h = m.norm3(x)
    return x + m.mlp(h), k, v


def _layer(dt=torch.float32, d=D, heads=HEADS, is_decoder=False, seed=0):
    torch.manual_seed(seed)
    layer = DecoderLayer(d, heads, 64, is_decoder=is_decoder)
    with torch.no_grad():
        for p in layer.parameters():
            p.copy_(torch.randn_like(p) * (0.2 if p.dim() == 1 else p.shape[-1] ** -0.5) + (1.0 if p.dim() == 1 else 0.0))
    return layer.to("cuda", dt)


def _paged(layer, b, s, dt=torch.float32):
    """An empty paged cache for b rows of s tokens."""
    blocks = -(-s // 16)
    pools = [torch.zeros(b * blocks, 16, layer.num_heads, 64, device="cuda", dtype=dt) for _ in range(2)]
    tables = torch.arange(b * blocks, dtype=torch.int32, device="cuda").view(b, blocks)
    return PagedKV([pools[0]], [pools[1]], tables, torch.full((b,), s, dtype=torch.int32, device="cuda"), blocks * 16)


def _forms(layer, x):
    """The layer's output over x by forward, and (causal layers) by forward_paged."""
    with torch.no_grad():
        out = [layer(x)[0]]
        if layer.is_decoder:
            y = layer.forward_paged(x, 0, _paged(layer, x.shape[0], x.shape[1], x.dtype), None)
            out.append(y[0] + y[1])
    return out


def _close(got, want, what, rel=2e-6):
    err = float((got.double() - want).norm() / want.norm())
    assert got.shape == want.shape and err < rel, f"{what}: relative error {err:.2e}"


class Doubled(nn.LayerNorm):
    def forward(self, x):
        return 2.0 * super().forward(x)


class Renamed(nn.LayerNorm):
    """LayerNorm under another name, its forward its own."""


def _patched(norm):
    norm.forward = types.MethodType(lambda self, x: 3.0 * F.layer_norm(x, (D,), self.weight, self.bias), norm)
    return norm


NORMS = {"subclass with its own forward": lambda: Doubled(D), "Identity": nn.Identity, "RMSNorm": lambda: nn.RMSNorm(D),
         "no affine": lambda: nn.LayerNorm(D, elementwise_affine=False), "no bias": lambda: nn.LayerNorm(D, bias=False),
         "subclass": lambda: Renamed(D), "forward set on the instance": lambda: _patched(nn.LayerNorm(D))}


@pytest.mark.parametrize("kind", NORMS)
@pytest.mark.parametrize("is_decoder", [False, True])
def test_replaced_norm_is_the_one_that_runs(cuda, kind, is_decoder):
    layer = _layer(is_decoder=is_decoder)
    x = torch.randn(2, 20, D, device="cuda")
    for name in ("norm1", "norm2", "norm3"):
        setattr(layer, name, NORMS[kind]().to("cuda"))
    want = _reference(layer, x)[0]
    for got in _forms(layer, x):
        _close(got, want, kind)
    seen = []
    for norm in (layer.norm1, layer.norm2):
        norm.register_forward_hook(lambda mod, args, out: seen.append(mod))
    _forms(layer, x)
    assert seen == [layer.norm1, layer.norm2] * (1 + is_decoder)


def _offset(p, elements):
    """The parameter's values at an address `elements` past a 16-byte line (a view into a flat buffer)."""
    flat = torch.empty(p.numel() + 8, device=p.device, dtype=p.dtype)
    view = flat[elements:elements + p.numel()].view(p.shape)
    return nn.Parameter(view.copy_(p.detach()))


@pytest.mark.parametrize("name", ["weight", "bias"])
@pytest.mark.parametrize("is_decoder", [False, True])
def test_norm_parameters_inside_a_flat_buffer(cuda, name, is_decoder):
    layer = _layer(is_decoder=is_decoder)
    x = torch.randn(2, 20, D, device="cuda")
    want = _reference(layer, x)[0]
    for norm in (layer.norm1, layer.norm2, layer.norm3):
        setattr(norm, name, _offset(getattr(norm, name), 1))
        assert getattr(norm, name).data_ptr() % 16 == 4
    for got in _forms(layer, x):
        _close(got, want, name)


class Through(nn.Module):
    """A projection whose result passes through f."""

    def __init__(self, inner, f):
        super().__init__()
        self.inner, self.f = inner, f

    def forward(self, x):
        return self.f(self.inner(x))


RESULTS = {"another dtype": lambda y: y.to(torch.bfloat16),
           "broadcast over positions": lambda y: y.mean(1, keepdim=True),
           "rows between 16-byte lines": lambda y: F.pad(y, (1, 0))[..., 1:],
           "channels apart": lambda y: torch.stack((y, y), -1)[..., 0]}


@pytest.mark.parametrize("kind", RESULTS)
def test_projection_results_as_torch_would_add_them(cuda, kind):
    layer = _layer()
    layer.self_attn_out = Through(layer.self_attn_out, RESULTS[kind])
    x = torch.randn(2, 20, D, device="cuda")
    want = _reference(layer, x)[0]
    # bfloat16 rounds the attention output once: 2^-9 of a term of the sum
    _close(_forms(layer, x)[0], want, kind, 2.0 ** -9 if kind == "another dtype" else 2e-6)


def test_norm_operands_on_another_device_are_refused(cuda):
    x, w = torch.randn(8, D, device="cuda"), torch.ones(D, device="cuda")
    for bad in ((x, None, w.cpu(), w), (x, None, w, w.cpu()), (x, x.cpu(), w, w)):
        assert native.add_layernorm(*bad, 1e-5, fallback=True) is None
        with pytest.raises(RuntimeError, match="unsupported"):
            native.add_layernorm(*bad, 1e-5)
    part = native.Partials(torch.zeros(2, 8, D, device="cuda"), None, torch.Size((8, D)), torch.float32)
    for bad in ((x, w.cpu(), w), (x, w, w.cpu())):
        assert native.reduce_add_layernorm(part, *bad, 1e-5) is None
    layer = _layer()
    layer.norm2.weight = nn.Parameter(layer.norm2.weight.detach().cpu())
    with torch.no_grad(), pytest.raises(RuntimeError):
        layer(x.view(2, 4, D))


@pytest.mark.parametrize("is_decoder", [False, True])
def test_input_of_permuted_rows(cuda, is_decoder):
    layer = _layer(is_decoder=is_decoder)
    x = torch.randn(20, 3, D, device="cuda").transpose(0, 1)  # dense, positions outermost
    want = _reference(layer, x)[0]
    for got in _forms(layer, x):
        _close(got, want, "permuted")
    y, w, b = torch.randn(3, 20, D, device="cuda"), torch.randn(D, device="cuda"), torch.randn(D, device="cuda")
    s, n = native.add_layernorm(x, y, w, b, 1e-5)
    assert torch.equal(s, x + y)
    _close(n, F.layer_norm((x + y).double(), (D,), w.double(), b.double(), 1e-5), "permuted norm")


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
def test_residual_rows_broadcast_from_one(cuda, dt):
    layer = _layer(dt, 256, 4, is_decoder=True)
    x = torch.randn(1, 1, 256, device="cuda").to(dt).expand(8, 1, 256)  # row stride 0
    want = _reference(layer, x)[0]
    y = layer.forward_paged(x, 0, _paged(layer, 8, 1, dt), None)
    _close(y[0].double() + y[1].double(), want, "expanded residual", 2e-6 if dt == torch.float32 else 2 * EPS[dt])
    a, w = torch.randn(8, 256, device="cuda").to(dt), layer.self_attn_out.weight
    assert native.decode_linear_residual(a, w, None, x[:, 0]) is None
    assert native.decode_linear_residual(a[:1], w, None, x[:1, 0]) is not None


@pytest.mark.parametrize("d,heads", [(128, 2), (512, 8), (1024, 16)])  # fc2 by torch's library, unsplit, and in partials
@pytest.mark.parametrize("s", [1, 5])
def test_final_norm_is_called_with_the_last_position(cuda, d, heads, s):
    """decode_step_paged calls the final norm and the LM head on [B, D] rows, and logits agree with every position's."""
    torch.manual_seed(3)
    m = models.WhisperClassSpeechEncoderDecoderModel(0, 2, heads, d, 80, 264, 64).to("cuda")
    ids = torch.randint(0, 264, (3, s), device="cuda")
    pools = [_paged(m.decoder_layers[0], 3, s) for _ in range(2)]
    kv = PagedKV([p.k_pools[0] for p in pools], [p.v_pools[0] for p in pools], pools[0].block_tables,
                 pools[0].ctx_lens, pools[0].max_ctx)
    shapes = []
    with torch.no_grad():
        every = m.decode_step_paged(ids, kv, last_only=False)
        plain = m.decode_step_paged(ids, kv)
        for mod in (m.decoder_norm, m.lm_head):
            mod.register_forward_hook(lambda mod, args, out: shapes.append(tuple(args[0].shape)))
        hooked = m.decode_step_paged(ids, kv)
    assert shapes == [(3, d), (3, d)] and plain.shape == (3, 264)
    for got in (plain, hooked):
        _close(got, every[:, -1].double(), "last position")


@pytest.mark.parametrize("where", ["class", "subclass", "instance"])
def test_wrapped_forward_paged_is_called(cuda, where, monkeypatch):
    torch.manual_seed(4)
    m = models.WhisperClassSpeechEncoderDecoderModel(0, 2, 8, 512, 80, 264, 64).to("cuda")
    ids = torch.randint(0, 264, (3, 1), device="cuda")
    pools = [_paged(m.decoder_layers[0], 3, 1) for _ in range(2)]
    kv = PagedKV([p.k_pools[0] for p in pools], [p.v_pools[0] for p in pools], pools[0].block_tables,
                 pools[0].ctx_lens, pools[0].max_ctx)
    seen, original = [], DecoderLayer.forward_paged

    def wrapper(self, x, layer, kv, cross, pending=None):
        seen.append((layer, torch.is_tensor(x), pending is None or torch.is_tensor(pending)))
        return original(self, x, layer, kv, cross, pending)

    with torch.no_grad():
        want = m.decode_step_paged(ids, kv)
        if where == "class":
            monkeypatch.setattr(DecoderLayer, "forward_paged", wrapper)
        for layer in m.decoder_layers:
            if where == "subclass":
                layer.__class__ = type("Wrapped", (DecoderLayer,), {"forward_paged": wrapper})
            elif where == "instance":
                layer.forward_paged = types.MethodType(wrapper, layer)
        got = m.decode_step_paged(ids, kv)
    assert seen == [(0, True, True), (1, True, True)]
    _close(got, want.double(), where)


class Plain(nn.Module):
    """An MLP of torch's own ops."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        for mod in self.inner:
            x = mod(x)
        return x


@pytest.mark.parametrize("cross", [False, True])
def test_gradients_reach_the_norm_ahead_of_a_torch_mlp(cuda, cross):
    """Attention ends a graph here; what follows it in torch's ops passes gradients on to the norm's parameters."""
    layer = _layer()
    layer.mlp = Plain(layer.mlp)
    x, enc = torch.randn(2, 20, D, device="cuda"), torch.randn(2, 9, D, device="cuda")
    g = torch.randn(2, 20, D, device="cuda")
    norm = layer.norm3 if cross else layer.norm2
    out = layer(x, encoder_hidden_states=enc if cross else None)[0]
    out.backward(g)
    m = copy.deepcopy(layer).double()
    m.zero_grad()
    taken = []
    (m.norm3 if cross else m.norm2).register_forward_pre_hook(lambda mod, args: taken.append(args[0]))
    want = _reference(m, x, enc if cross else None)[0]
    _close(out.detach(), want, "output")
    s = taken[0]
    ref = m.norm3 if cross else m.norm2
    (s + m.mlp(ref(s))).backward(g.double())
    for name in ("weight", "bias"):
        _close(getattr(norm, name).grad, getattr(ref, name).grad, name, 1e-5)


def test_tangents_pass_the_residual_adds(cuda):
    layer = _layer()
    layer.mlp = Plain(layer.mlp)
    x, t = torch.randn(2, 20, D, device="cuda"), torch.randn(2, 20, D, device="cuda")
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        out = layer(torch.autograd.forward_ad.make_dual(x, t))[0]
        got = torch.autograd.forward_ad.unpack_dual(out)
        assert got.tangent is not None and got.tangent.shape == x.shape
        primal = got.primal.clone()
    _close(primal, _reference(layer, x)[0], "primal")


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [51200, 51864])
def test_lm_head_of_a_vocabulary_the_decode_kernel_takes(cuda, dt, n):
    """proj over the rows around the crossover to the library, by whichever path serves them."""
    head = nn.Linear(384, n, bias=False).to("cuda", dt)
    for m in (1, 17, 40, 41, 64, 128):
        x = torch.randn(m, 384, device="cuda").to(dt)
        with torch.no_grad():
            got = models.proj(head, x).double()
            want = x.double() @ head.weight.double().t()
            bound = 384 * 2.0 ** -24 * (x.double().abs() @ head.weight.double().abs().t())
        assert bool(((got - want).abs() <= EPS[dt] * want.abs() + bound + 1e-30).all()), m


# rows past the decode batch: q/k/v by head, GELU in the epilogue, adds and norms in one launch (16-bit); fp32 attention of
# several queries on the matrix cores (2 x 300 queries of 4 heads over 300 keys are past its bound)
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("b,s", [(1, 150), (3, 97), (2, 300)])
@pytest.mark.parametrize("is_decoder,form", [(False, "plain"), (False, "masked"), (False, "cross"), (True, "plain"),
                                             (True, "cross"), (True, "cross masked")])
def test_forward_of_many_rows(cuda, dt, b, s, is_decoder, form):
    """DecoderLayer.forward over prompts and frames: output, returned K/V and cross K/V against float64."""
    d, heads, te = 256, 4, 110
    layer = _layer(dt, d, heads, is_decoder)
    x = torch.randn(b, s, d, device="cuda").to(dt)
    enc = torch.randn(b, te, d, device="cuda").to(dt) if "cross" in form else None
    keep = cross_keep = None
    if form == "masked":
        keep = torch.arange(s, device="cuda")[None] < torch.randint(1, s + 1, (b, 1), device="cuda")
        keep[0, ::3] = False  # not a prefix
        keep[:, 1] = True
    if form == "cross masked":
        cross_keep = torch.arange(te, device="cuda")[None] < torch.randint(1, te + 1, (b, 1), device="cuda")
    with torch.no_grad():
        y, (k, v), cross = layer(x, encoder_hidden_states=enc,
                                 attention_mask=None if keep is None else keep.long(),
                                 encoder_attention_mask=None if cross_keep is None else cross_keep.long())
    want, wk, wv = _reference(layer, x, enc, keep, cross_keep)
    rel = 2e-6 if dt == torch.float32 else 2 * EPS[dt]  # a rounding of each of the layer's tensors, as root mean square
    assert k.shape == (b, heads, s, 64)
    for got, ref, what in ((y, want, "output"), (k, wk, "k"), (v, wv, "v")):
        _close(got, ref, f"{form} {what}", rel)
    assert (cross is None) == (enc is None)
