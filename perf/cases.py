"""Performance cases: the work a user of this package has it do, through its public entry points.

A case is a dict of plain values. `prepare` makes what a serving program holds before the call (weights, K/V pools,
block tables, captured graphs), `run` makes one pass, `exact` gives the same outputs in plain float64 torch.

Kinds:
  layer    one decode step of one decoder layer (DecoderLayer.forward_paged, one token per row), replayed from a HIP
           graph as the graph decode replays it: fused append + paged self-attention, cross-attention, MLP
  step     a whole decode step (decode_step_paged: embedding, decoder layers, LM head), replayed from a HIP graph
  tts      a whole decode step of the multi-codebook TTS model, replayed from a HIP graph
  prompt   the eager prefill of a prompt through one decoder layer (several tokens per row, causal)
  self     the paged self-attention calls of a few layers with their fused append, replayed from a HIP graph
  cross    one cross-attention call over the encoder K/V of the decode slots
  encoder  one encoder layer over a request's frames (DecoderLayer.forward, non-causal)
  store    encoder K/V rows appended into a paged pool and gathered back as a zero-padded batch
"""
import math
import os
import sys

import torch
import torch.nn.functional as F

_PKG = os.path.join(os.getcwd(), "inference-speech-model_amd")  # the package's folder in the tree under test
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from speech_serving import native  # noqa: E402
from speech_serving.models import (CrossKV, DecoderLayer, PagedKV, StreamingMultiCodebookTTSModel,  # noqa: E402
                                   WhisperClassSpeechEncoderDecoderModel)

HEAD_DIM = 64  # every Whisper-class and TTS shape here
BLOCK = 16     # KV block size of the block manager
_DTYPE = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}
_BYTES = {"fp32": 4, "fp16": 2, "bf16": 2}
_LAYERS = ("self_attn_q", "self_attn_k", "self_attn_v", "self_attn_out", "cross_attn_q", "cross_attn_out")


def listed():
    return [
        # The smallest decode call: a tiny-shaped decoder layer (d_model 384, 4 heads), 4 requests, fp32.
        {"name": "layer_tiny_b4_fp32", "kind": "layer", "dtype": "fp32", "d": 384, "heads": 4, "batch": 4,
         "ctx": 68, "enc_min": 1500, "enc": 1500},
        # Base-shaped layer under continuous batching: 32 slots, encoder lengths 500..1500, fp16.
        {"name": "layer_base_b32_fp16", "kind": "layer", "dtype": "fp16", "d": 512, "heads": 8, "batch": 32,
         "ctx": 228, "enc_min": 500, "enc": 1500},
        # Large-v3-shaped layer at the decode batch of 64, mixed context lengths up to a full decode.
        {"name": "layer_large_v3_b64_bf16", "kind": "layer", "dtype": "bf16", "d": 1280, "heads": 20, "batch": 64,
         "ctx": 452, "enc_min": 1500, "enc": 1500},
        # The same layer at the serving configuration's 128 slots.
        {"name": "layer_large_v3_b128_bf16", "kind": "layer", "dtype": "bf16", "d": 1280, "heads": 20, "batch": 128,
         "ctx": 452, "enc_min": 1500, "enc": 1500},
        # A whole decode step of the small-shaped decoder (12 layers), 64 graph slots: returns logits.
        {"name": "step_small_b64_bf16", "kind": "step", "dtype": "bf16", "d": 768, "heads": 12, "batch": 64,
         "layers": 12, "vocab": 51865, "ctx": 452, "enc_min": 1500, "enc": 1500},
        # A whole decode step of the default multi-codebook TTS model, 64 requests: returns logits.
        {"name": "tts_step_b64_bf16", "kind": "tts", "dtype": "bf16", "d": 256, "heads": 4, "batch": 64,
         "layers": 4, "codebooks": 4, "vocab": 1024, "ctx": 288},
        # Admission: the 4-token start prompt of 128 large-v3-shaped requests, prefilled as one batch.
        {"name": "prompt_large_v3_b128_q4_bf16", "kind": "prompt", "dtype": "bf16", "d": 1280, "heads": 20,
         "batch": 128, "q": 4, "enc_min": 1500, "enc": 1500},
        # Admission with a long text prompt (up to half the decoder's 448 positions), a few requests.
        {"name": "prompt_large_v3_b8_q201_bf16", "kind": "prompt", "dtype": "bf16", "d": 1280, "heads": 20,
         "batch": 8, "q": 201, "enc_min": 1500, "enc": 1500},
        # Paged decode attention alone: 32 heads, batch 64, context lengths 1..448, fp16 (four layers' launches).
        {"name": "self_attention_b64_fp16", "kind": "self", "dtype": "fp16", "heads": 32, "batch": 64,
         "layers": 4, "ctx": 448},
        # Cross-attention alone at the large-v3 shape: the most bytes of a decode step.
        {"name": "cross_attention_b64_bf16", "kind": "cross", "dtype": "bf16", "heads": 20, "batch": 64,
         "enc_min": 1500, "enc": 1500},
        # One encoder layer of the large-v3 shape over a 30 s request (1500 positions).
        {"name": "encoder_layer_large_v3_bf16", "kind": "encoder", "dtype": "bf16", "d": 1280, "heads": 20,
         "batch": 1, "enc": 1500},
        # Encoder K/V of 16 requests stored into paged blocks and gathered back for contiguous readers.
        {"name": "kv_store_b16_bf16", "kind": "store", "dtype": "bf16", "heads": 20, "batch": 16, "enc_min": 500,
         "enc": 1500},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "step", "tts", "prompt", "prompt", "self", "cross", "encoder",
                       "store"])
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp16", "fp32"])
    heads = rng.choice([4, 6, 8, 12, 16, 20])  # tiny .. large
    enc = _log_int(rng, 100, 1500)
    case = {"kind": kind, "dtype": dtype, "heads": heads, "batch": _log_int(rng, 1, 128)}
    if kind in ("layer", "step", "prompt", "encoder"):
        case["d"] = 64 * heads if heads != 4 else rng.choice([256, 384])
    if kind in ("layer", "step", "prompt", "cross", "store"):
        case["enc_min"] = rng.choice([enc, max(1, enc // 3)])
        case["enc"] = enc
    if kind in ("layer", "step"):
        case["ctx"] = _log_int(rng, 4, 452)
    if kind == "layer" and dtype == "fp32":
        case["batch"] = _log_int(rng, 1, 64)
    if kind == "step":
        case["layers"] = rng.randint(1, 6)
        case["batch"] = _log_int(rng, 1, 64)
        case["vocab"] = rng.choice([51865, 51866])
    if kind == "tts":
        case["batch"] = _log_int(rng, 1, 64)
        case["heads"] = rng.choice([4, 8])
        case["d"] = 64 * case["heads"]
        case["layers"] = rng.randint(2, 6)
        case["codebooks"] = rng.choice([1, 4, 8])
        case["vocab"] = rng.choice([256, 1024])
        case["ctx"] = _log_int(rng, 4, 512)
    if kind == "prompt":
        case["q"] = _log_int(rng, 2, 224)
        case["batch"] = _log_int(rng, 1, min(128, max(1, 1608 // case["q"])))
        if dtype == "fp32":
            case["batch"] = min(case["batch"], max(1, 200 // case["q"]))
    if kind == "self":
        case["layers"] = rng.randint(1, 4)
        case["batch"] = _log_int(rng, 1, 96)
        case["ctx"] = _log_int(rng, 8, 448)
    if kind == "cross":
        case["batch"] = _log_int(rng, 1, 96)
        if dtype == "fp32":
            case["batch"] = min(case["batch"], 48)
    if kind == "encoder":
        case["batch"] = 1
        case["enc"] = enc if dtype != "fp32" else min(enc, 600)
    if kind == "store":
        case["batch"] = _log_int(rng, 1, 16)
    return case


# ---------------------------------------------------------------------------
# Inputs: plain tensors on the GPU, made from the seed alone.
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, dt, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dt)


def _randn_low(g, dt, *shape):
    """N(0, 1) drawn in the dtype itself (large K/V buffers: no float32 copy)."""
    return torch.randn(*shape, generator=g, device="cuda", dtype=dt)


def _lengths(g, n, lo, hi):
    """n lengths U[lo, hi], longest first (the order graph decode lays its rows out in)."""
    v = torch.randint(lo, hi + 1, (n,), generator=g, device="cuda", dtype=torch.int32)
    return torch.sort(v, descending=True).values.contiguous()


def _tables(g, batch, width, blocks):
    perm = torch.randperm(blocks, generator=g, device="cuda")[: batch * width]
    return perm.view(batch, width).to(torch.int32).contiguous()


def _norm_pair(g, dt, d):
    return _randn(g, dt, d, std=0.1) + 1.0, _randn(g, dt, d, std=0.1)


def _layer_weights(g, dt, d, hd):
    w = {}
    for name in _LAYERS:
        n, k = (d, hd) if name.endswith("out") else (hd, d)
        w[name] = _randn(g, dt, n, k, std=0.02)
    for name in ("norm1", "norm2", "norm3"):
        w[name] = _norm_pair(g, dt, d)
    w["fc1"] = (_randn(g, dt, 4 * d, d, std=0.02), _randn(g, dt, 4 * d, std=0.02))
    w["fc2"] = (_randn(g, dt, d, 4 * d, std=0.02), _randn(g, dt, d, std=0.02))
    return w


def _cross_buffers(case, g, dt, n_layers):
    """Slot-major encoder K/V [S, L, 2, H, T, D] and the rows' lengths."""
    kv = _randn_low(g, dt, case["batch"], n_layers, 2, case["heads"], case["enc"], HEAD_DIM)
    lens = torch.randint(case["enc_min"], case["enc"] + 1, (case["batch"],), generator=g, device="cuda",
                         dtype=torch.int32)
    return kv, lens


def _paged_inputs(case, g, dt, n_layers, ctx_lo, ctx_hi):
    width = -(-ctx_hi // BLOCK)
    blocks = case["batch"] * width + 3
    pools = [_randn_low(g, dt, 2, blocks, BLOCK, case["heads"], HEAD_DIM) for _ in range(n_layers)]
    return {"pools": pools, "tables": _tables(g, case["batch"], width, blocks),
            "ctx": _lengths(g, case["batch"], ctx_lo, ctx_hi), "max_ctx": width * BLOCK}


def _inputs(case, seed):
    g, dt, kind, b = _gen(seed), _DTYPE[case["dtype"]], case["kind"], case["batch"]
    hd = case["heads"] * HEAD_DIM
    s = {}
    if kind in ("layer", "step", "prompt"):
        n = case.get("layers", 1)
        s["w"] = [_layer_weights(g, dt, case["d"], hd) for _ in range(n)]
        if kind == "prompt":  # the prompt's tokens are the row's only keys
            s.update(_paged_inputs(case, g, dt, n, case["q"], case["q"]))
        else:
            s.update(_paged_inputs(case, g, dt, n, 1, case["ctx"]))
        s["cross"], s["enc_lens"] = _cross_buffers(case, g, dt, n)
        if kind == "step":
            s["embed"] = _randn(g, dt, case["vocab"], case["d"], std=0.02)
            s["head"] = _randn(g, dt, case["vocab"], case["d"], std=0.02)
            s["norm"] = _norm_pair(g, dt, case["d"])
            s["ids"] = torch.randint(0, case["vocab"], (b, 1), generator=g, device="cuda")
        else:
            q = case.get("q", 1)
            s["x"] = _randn(g, dt, b, q, case["d"])
            s["pending"] = _randn(g, dt, b, q, case["d"], std=0.5)
    elif kind == "tts":
        s["w"] = [_layer_weights(g, dt, case["d"], hd) for _ in range(case["layers"])]
        s.update(_paged_inputs(case, g, dt, case["layers"], 1, case["ctx"]))
        s["embed"] = [_randn(g, dt, case["vocab"], case["d"], std=0.02) for _ in range(case["codebooks"])]
        s["head"] = [_randn(g, dt, case["vocab"], case["d"], std=0.02) for _ in range(case["codebooks"])]
        s["norm"] = _norm_pair(g, dt, case["d"])
        s["ids"] = torch.randint(0, case["vocab"], (b, 1, case["codebooks"]), generator=g, device="cuda")
    elif kind == "self":
        s.update(_paged_inputs(case, g, dt, case["layers"], 1, case["ctx"]))
        s["qkv"] = [[_randn(g, dt, b, case["heads"], HEAD_DIM) for _ in range(3)] for _ in range(case["layers"])]
    elif kind == "cross":
        s["cross"], s["enc_lens"] = _cross_buffers(case, g, dt, 1)
        s["q"] = _randn(g, dt, b, 1, case["heads"], HEAD_DIM)
    elif kind == "encoder":
        s["w"] = [_layer_weights(g, dt, case["d"], hd)]
        s["x"] = _randn(g, dt, b, case["enc"], case["d"])
    elif kind == "store":
        width = -(-case["enc"] // BLOCK)
        blocks = b * width + 3
        s["pools"] = [torch.zeros(2, blocks, BLOCK, case["heads"], HEAD_DIM, device="cuda", dtype=dt)]
        s["tables"] = _tables(g, b, width, blocks)
        s["lens"] = torch.randint(case["enc_min"], case["enc"] + 1, (b,), generator=g, device="cuda",
                                  dtype=torch.int32)
        lens = s["lens"].long()
        row = torch.repeat_interleave(torch.arange(b, device="cuda"), lens)
        pos = torch.arange(row.numel(), device="cuda") - (lens.cumsum(0) - lens)[row]
        s["slots"] = s["tables"].long()[row, pos // BLOCK] * BLOCK + pos % BLOCK
        s["row"], s["pos"] = row, pos
        s["kv"] = [_randn(g, dt, row.numel(), case["heads"], HEAD_DIM) for _ in range(2)]
    return s


# ---------------------------------------------------------------------------
# The program's state and one pass.
# ---------------------------------------------------------------------------
def _load_layer(layer, w):
    for name in _LAYERS:
        getattr(layer, name).weight.data = w[name]
    for name in ("norm1", "norm2", "norm3"):
        getattr(layer, name).weight.data, getattr(layer, name).bias.data = w[name]
    layer.mlp[0].weight.data, layer.mlp[0].bias.data = w["fc1"]
    layer.mlp[2].weight.data, layer.mlp[2].bias.data = w["fc2"]


def _paged_kv(s):
    return PagedKV([p[0] for p in s["pools"]], [p[1] for p in s["pools"]], s["tables"], s["ctx"], s["max_ctx"],
                   rows_longest_first=True)


def _cross_kv(s):
    n = s["cross"].shape[1]
    return CrossKV([s["cross"][:, l, 0] for l in range(n)], [s["cross"][:, l, 1] for l in range(n)], s["enc_lens"],
                   s["cross"].shape[4])


def _captured(case, s, step):
    """step() captured into a HIP graph after a warm-up on a side stream, as the graph decode captures its buckets."""
    dt = _DTYPE[case["dtype"]]
    native.reserve_attention(case["batch"], case["heads"], HEAD_DIM, s["max_ctx"], dt, "cuda")
    if "cross" in s:
        native.reserve_attention(case["batch"], case["heads"], HEAD_DIM, case["enc"], dt, "cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.no_grad(), torch.cuda.stream(side):
        step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph, stream=side):
        out = step()
    return {"graph": graph, "out": out, "keep": (s, step, native.reserve_workspace(0, "cuda"))}


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    with torch.device("cuda"):
        if kind in ("layer", "prompt", "encoder"):
            layer = DecoderLayer(case["d"], case["heads"], HEAD_DIM, is_decoder=kind != "encoder")
        elif kind == "step":
            model = WhisperClassSpeechEncoderDecoderModel(0, case["layers"], case["heads"], case["d"], 80,
                                                          case["vocab"], HEAD_DIM)
        elif kind == "tts":
            model = StreamingMultiCodebookTTSModel(case["layers"], case["heads"], case["d"], case["codebooks"],
                                                   case["vocab"])
    if kind in ("layer", "prompt", "encoder"):
        _load_layer(layer, s["w"][0])
        if kind == "encoder":
            return {"call": lambda: layer(s["x"])[:2]}
        kv, cross = _paged_kv(s), _cross_kv(s)

        def one():
            x, y = layer.forward_paged(s["x"], 0, kv, cross, s["pending"])
            return x, y, s["pools"][0]

        return {"call": one} if kind == "prompt" else _captured(case, s, one)
    if kind in ("step", "tts"):
        layers = model.decoder_layers if kind == "step" else model.layers
        for layer, w in zip(layers, s["w"]):
            _load_layer(layer, w)
        norm = model.decoder_norm if kind == "step" else model.norm
        norm.weight.data, norm.bias.data = s["norm"]
        if kind == "step":
            model.decoder_embed.weight.data, model.lm_head.weight.data = s["embed"], s["head"]
        else:
            for i in range(case["codebooks"]):
                model.embeddings.embeddings[i].weight.data = s["embed"][i]
                model.heads.heads[i].weight.data = s["head"][i]
        kv = _paged_kv(s)
        if kind == "step":
            cross = _cross_kv(s)
            return _captured(case, s, lambda: model.decode_step_paged(s["ids"], kv, cross))
        return _captured(case, s, lambda: model.decode_step_paged(s["ids"], kv))
    scale = 1.0 / math.sqrt(HEAD_DIM)
    if kind == "self":
        def attend():
            out = [native.paged_attention(q, p[0], p[1], s["tables"], s["ctx"], s["max_ctx"], scale, k_new=k,
                                          v_new=v, rows_longest_first=True)
                   for (q, k, v), p in zip(s["qkv"], s["pools"])]
            return out, s["pools"]

        return _captured(case, s, attend)
    if kind == "cross":
        k, v = s["cross"][:, 0, 0], s["cross"][:, 0, 1]
        return {"call": lambda: native.dense_attention(s["q"], k, v, s["enc_lens"], case["enc"], scale)}
    k_pool, v_pool = s["pools"][0]

    def store():
        native.append(s["kv"][0], s["kv"][1], k_pool, v_pool, s["slots"])
        k, v = native.gather(k_pool, v_pool, s["tables"], s["lens"], case["enc"])
        return k, v, k_pool, v_pool

    return {"call": store}


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    with torch.no_grad():
        return state["call"]()


# ---------------------------------------------------------------------------
# What a pass cannot do without: each input read once, each output written once.
# ---------------------------------------------------------------------------
def work(case):
    e, b, h, kind = _BYTES[case["dtype"]], case["batch"], case["heads"], case["kind"]
    hd = h * HEAD_DIM
    n, q, d = case.get("layers", 1), case.get("q", 1), case.get("d", 0)
    enc = (case.get("enc_min", 0) + case.get("enc", 0)) / 2
    if kind == "store":
        rows, out = b * enc, b * case["enc"]
        return {"bytes": 2 * hd * e * (2 * rows + rows + out) + 8 * rows, "flops": 0}
    if kind == "cross":
        return {"bytes": 2 * b * enc * hd * e + 2 * b * hd * e, "flops": 4 * b * enc * hd}
    if kind == "self":
        ctx = (case["ctx"] + 1) / 2
        return {"bytes": n * (2 * b * ctx * hd * e + 6 * b * hd * e), "flops": n * 4 * b * ctx * hd}
    if kind == "encoder":
        t = case["enc"]
        w = 4 * hd * d + 8 * d * d
        return {"bytes": e * (w + 2 * t * d + 2 * t * hd), "flops": 2 * t * w + 4 * t * t * hd}
    rows = b * q
    ctx = (q + 1) / 2 if kind == "prompt" else (case["ctx"] + 1) / 2
    weights = (4 if kind == "tts" else 6) * hd * d + 8 * d * d
    kv = b * (0 if kind == "prompt" else ctx) + 2 * rows + (0 if kind == "tts" else b * enc)
    nbytes = n * e * (weights + 2 * hd * kv)
    flops = n * (2 * rows * weights + 4 * rows * (ctx + (0 if kind == "tts" else enc)) * hd)
    if kind in ("step", "tts"):
        out = case["vocab"] * case.get("codebooks", 1)
        nbytes += e * (out * d + rows * out)
        flops += 2 * rows * out * d
    else:
        nbytes += 4 * rows * d * e
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "store":
        return "exact"
    # Measured against float64: one rounding of the output per op (self, cross), a layer's six products and
    # softmaxes (layer, prompt, encoder), and whole models, where a rounding travels through the layers that follow.
    if case["dtype"] == "fp32":
        return {"rel": 1e-5, "max": 2e-4}
    if case["kind"] in ("self", "cross"):
        return {"rel": 8e-4, "max": 8e-3} if case["dtype"] == "fp16" else {"rel": 6e-3, "max": 6e-2}
    if case["kind"] in ("step", "tts"):
        return {"rel": 4e-3, "max": 4e-2} if case["dtype"] == "fp16" else {"rel": 2.5e-2, "max": 2e-1}
    return {"rel": 1.5e-3, "max": 2e-2} if case["dtype"] == "fp16" else {"rel": 1e-2, "max": 1e-1}


# ---------------------------------------------------------------------------
# The same outputs in float64.
# ---------------------------------------------------------------------------
def _ln(x, pair):
    return F.layer_norm(x, (x.shape[-1],), pair[0].double(), pair[1].double(), 1e-5)


def _attend(q, k, v, visible):
    """q [H, Q, D] over k, v [H, T, D]; query i sees the first visible[i] keys."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(HEAD_DIM)
    t = torch.arange(k.shape[1], device=q.device)
    s = s.masked_fill(t[None, None, :] >= visible[None, :, None], -math.inf)
    return torch.matmul(torch.softmax(s, dim=-1), v)


def _exact_self(s, l, q, k, v):
    """Causal paged self-attention of q, k, v [B, Q, H, D] (float64) after appending k, v; pools updated in place."""
    kp, vp = s["pools"][l][0], s["pools"][l][1]
    b, n = q.shape[:2]
    out = torch.empty_like(q)
    for r in range(b):
        ctx = int(s["ctx"][r])
        new = torch.arange(max(0, ctx - n), ctx, device=q.device)
        table = s["tables"][r].long()
        blk, off = table[new // BLOCK], new % BLOCK
        kp[blk, off], vp[blk, off] = k[r, n - len(new):], v[r, n - len(new):]
        use = table[: -(-ctx // BLOCK)]
        kk = kp[use].reshape(-1, *kp.shape[2:])[:ctx].transpose(0, 1)
        vv = vp[use].reshape(-1, *vp.shape[2:])[:ctx].transpose(0, 1)
        seen = ctx - n + 1 + torch.arange(n, device=q.device)
        out[r] = _attend(q[r].transpose(0, 1), kk, vv, seen).transpose(0, 1)
    return out


def _exact_cross(q, ck, cv, lens):
    out = torch.empty_like(q)
    for r in range(q.shape[0]):
        t = int(lens[r])
        seen = torch.full((q.shape[1],), t, device=q.device)
        out[r] = _attend(q[r].transpose(0, 1), ck[r, :, :t].double(), cv[r, :, :t].double(), seen).transpose(0, 1)
    return out


def _exact_layer(s, l, x, cross):
    """x + everything of decoder layer l but its MLP output, and the MLP output, in float64."""
    w, heads = s["w"][l], s["pools"][l].shape[3]
    b, q, _ = x.shape
    lin = lambda t, m: torch.matmul(t, m.double().t())  # noqa: E731
    split = lambda t: t.view(b, q, heads, HEAD_DIM)  # noqa: E731
    h = _ln(x, w["norm1"])
    a = _exact_self(s, l, *(split(lin(h, w[f"self_attn_{c}"])) for c in "qkv"))
    x = x + lin(a.reshape(b, q, -1), w["self_attn_out"])
    if cross:
        c = _exact_cross(split(lin(_ln(x, w["norm2"]), w["cross_attn_q"])), s["cross"][:, l, 0], s["cross"][:, l, 1],
                         s["enc_lens"])
        x = x + lin(c.reshape(b, q, -1), w["cross_attn_out"])
    h = _ln(x, w["norm3" if cross else "norm2"])
    y = F.gelu(lin(h, w["fc1"][0]) + w["fc1"][1].double())
    return x, lin(y, w["fc2"][0]) + w["fc2"][1].double()


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "encoder" and case["batch"] > 1:
        return None
    s, kind = _inputs(case, seed), case["kind"]
    if "pools" in s:
        s["pools"] = [p.double() for p in s["pools"]]
    if kind in ("layer", "prompt"):
        x, y = _exact_layer(s, 0, s["x"].double() + s["pending"].double(), True)
        return x, y, s["pools"][0]
    if kind in ("step", "tts"):
        if kind == "step":
            x = s["embed"].double()[s["ids"]]
        else:
            x = sum(t.double()[s["ids"][..., i]] for i, t in enumerate(s["embed"]))
        for l in range(case["layers"]):
            x, y = _exact_layer(s, l, x, kind == "step")
            x = x + y
        h = _ln(x[:, -1], s["norm"])
        if kind == "step":
            return torch.matmul(h, s["head"].double().t())
        return torch.stack([torch.matmul(h, w.double().t()) for w in s["head"]], dim=1)
    if kind == "self":
        out = [_exact_self(s, l, *(t.double().unsqueeze(1) for t in qkv))[:, 0] for l, qkv in enumerate(s["qkv"])]
        return out, s["pools"]
    if kind == "cross":
        return _exact_cross(s["q"].double(), s["cross"][:, 0, 0], s["cross"][:, 0, 1], s["enc_lens"])
    if kind == "encoder":
        w, x = s["w"][0], s["x"].double()
        lin = lambda t, m: torch.matmul(t, m.double().t())  # noqa: E731
        t = case["enc"]
        h = _ln(x, w["norm1"])[0]
        q, k, v = (lin(h, w[f"self_attn_{c}"]).view(t, case["heads"], HEAD_DIM).transpose(0, 1) for c in "qkv")
        seen = torch.full((t,), t, device=x.device)
        a = _attend(q, k, v, seen).transpose(0, 1).reshape(t, -1)
        x = x + lin(a, w["self_attn_out"])
        y = F.gelu(lin(_ln(x, w["norm2"]), w["fc1"][0]) + w["fc1"][1].double())
        return x + lin(y, w["fc2"][0]) + w["fc2"][1].double(), (k.unsqueeze(0), v.unsqueeze(0))
    k_pool, v_pool = s["pools"][0]
    outs = []
    for src, pool in ((s["kv"][0], k_pool), (s["kv"][1], v_pool)):
        pool.view(-1, *pool.shape[2:])[s["slots"]] = src.double()
        o = torch.zeros(case["batch"], case["heads"], case["enc"], HEAD_DIM, device="cuda", dtype=torch.float64)
        o[s["row"], :, s["pos"]] = src.double()
        outs.append(o)
    return outs[0], outs[1], k_pool, v_pool
